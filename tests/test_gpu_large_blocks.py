"""The blocked factor of windows with more than 40 free key frames at its block edges: reduced systems whose order
leaves a last 64-row block of 2, 8, 54, 58, 60, 62 and 64 rows."""
import numpy as np
import pytest

import cuvslam_amd as ca
from oracle import sba_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("free", [41, 42, 43, 44, 53, 63, 64, 75])
def test_steps_match_oracle(free):
    p, _, _ = ca.scene.loop(seed=free, num_keyframes=free + 1, num_points=60 * free, num_stereo_pairs=2,
                            loop_length_m=0.25 * free, outlier_rate=0.0, max_iterations=3)
    assert p.rig_from_world.shape[0] - p.num_fixed_key_frames == free
    ref = O.solve(p, "f64", loss=ca.LOSS_HUBER, fixed_iterations=1)
    q, again = p.copy(), p.copy()
    solver = ca.SchurComplementBundlerGpu(loss=ca.LOSS_HUBER, fixed_iterations=True)
    assert solver.solve(q) and solver.solve(again)
    assert q.accepted == ref["accepted"]
    # three steps of an FP32 system factored in FP64: the cost follows the FP64 one to the FP32 rounding of its inputs
    assert abs(q.last_cost_f64 - ref["last_cost"]) <= 1e-6 * ref["last_cost"]
    assert again.last_cost_f64 == q.last_cost_f64 and np.array_equal(again.points, q.points)
