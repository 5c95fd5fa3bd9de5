"""Inertial SBA (sba_imu_solve) in the corners of its kernels, against the FP64 oracle with the bounds of the parity
scenes: both compute in FP64. The reduced system's factor keeps its nonzero 16 x 16 tiles in shared memory up to 64 of
them (10 free key frames that share points: 55 tiles; 11: 66; 32 on two-frame tracks: 63; 33: 65), the point kernels
take 8 lanes per point (up to 13 pairs and 26 observations of a point here), and the pose blocks 512 observations at a
time."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

import imu_cases as IC  # noqa: E402
from cuvslam_amd import imu  # noqa: E402
from oracle import imu_oracle as IO  # noqa: E402
from test_gpu_imu import check_parity  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("iterations", [2, 10])
def test_information_that_is_not_symmetric(iterations):
    # the reduced system is then not symmetric either; its lower triangle is factored
    p, calib, _ = IC.make_scenario(6, shape=(6, 2, 80, 4))
    p.max_iterations = iterations
    p.observation_infos = np.array(p.observation_infos)
    p.observation_infos[:, 0, 1] = 0.2 * p.observation_infos[:, 0, 0]
    p.observation_infos[:, 1, 0] = 0.1 * p.observation_infos[:, 0, 0]
    ref = IO.solve(p, calib)
    q = p.copy()
    assert imu.IMUBundlerGpuFixedVel(IC.calibration()).solve(q)
    check_parity(q, ref)


# (key frames, fixed, points, track length)
@pytest.mark.parametrize("shape", [(2, 1, 40, 2), (3, 1, 513, 3), (9, 2, 120, 7), (10, 2, 120, 8), (11, 2, 120, 9),
                                   (12, 2, 60, 12), (13, 2, 60, 13), (34, 2, 340, 2), (35, 2, 350, 2)])
def test_route_edges_match_oracle(shape):
    p, calib, _ = IC.make_scenario(5, shape=shape)
    ref = IO.solve(p, calib)
    q = p.copy()
    assert imu.IMUBundlerGpuFixedVel(IC.calibration()).solve(q)
    check_parity(q, ref)
