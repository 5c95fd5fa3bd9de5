"""Inertial SBA (sba_imu_solve) in the corners of its kernels, against the FP64 oracle with the bounds of the parity
scenes: both compute in FP64."""
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
