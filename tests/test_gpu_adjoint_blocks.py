"""The block-sparse products of the implicit differentiation where their tiles and slots can go wrong: fewer tiles than
workgroups, one point, one free key frame, fixed points, a rig of several cameras (several observations per pair), and
a batch whose other windows do not take part."""
import numpy as np
import pytest

import cuvslam_amd as ca
from lm_cases import reference_style_problem
from oracle import sba_oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(b)


def window(kind):
    if kind == "rig":
        p = reference_style_problem(3, num_points=80)
        noise = np.random.default_rng(5).normal(0, 1e-3, p.observation_xys.shape)
        p.observation_xys = (p.observation_xys + noise).astype(np.float32)
        p.max_iterations = 50
        return p
    points, key_frames, fixed = {"one free key frame": (40, 4, 3), "few points": (9, 6, 3), "tile edge": (256, 5, 2),
                                 "many tiles": (3000, 12, 3), "fixed points": (120, 6, 2)}[kind]
    p = ca.scene.generate(seed=11, num_points=points, num_keyframes=key_frames, num_fixed_keyframes=fixed, z_max=9.0,
                          xy_extent=2.0, max_iterations=50)[0]
    if kind == "fixed points":
        p.num_fixed_points = 50
    return p


@pytest.mark.parametrize("kind", ["one free key frame", "few points", "tile edge", "many tiles", "fixed points", "rig"])
@pytest.mark.parametrize("in_batch", [False, True])
def test_adjoint_matches_oracle(kind, in_batch):
    p = window(kind)
    solver = ca.SchurComplementBundlerGpu(loss=ca.LOSS_STUDENT_T, fixed_iterations=True)
    other = ca.scene.generate(seed=12, num_points=100, num_keyframes=5, num_fixed_keyframes=2, max_iterations=50)[0]
    batch = solver.batch([p, other] if in_batch else [p])
    batch.run()
    poses, pts, _ = batch.refine(newton_steps=3, gauss_newton_steps=4, max_cg=300, tol=1e-13)
    ncf, npf = p.rig_from_world.shape[0] - p.num_fixed_key_frames, p.points.shape[0] - p.num_fixed_points
    g = np.random.default_rng(1).standard_normal(6 * ncf + 3 * npf)
    seen = np.bincount(p.point_ids, minlength=p.points.shape[0])[:npf] > 0  # the others have no block in the Hessian
    g[6 * ncf:] *= 1e-3 * np.repeat(seen, 3)
    dxy, dinfo, it, a = batch.adjoint(g, max_cg=300, tol=1e-13)
    assert 0 < it < 300
    ra, rdxy, rdinfo, rit = O.implicit_grad(p, g, pts, poses, loss=ca.LOSS_STUDENT_T, tol=1e-13)
    # both stop at a residual of 1e-13 of the right-hand side; the bound leaves a condition number of 1e6 for the rest
    assert rel(a, ra) < 1e-7 and rel(dxy, rdxy) < 1e-7 and rel(dinfo, rdinfo) < 1e-7
