"""The 16 x 16 diagonal factor of the reduced camera system at the places where its four-row panels can go wrong: a
non-positive pivot at every row of a tile, rows of very different scale, and pivots that nearly cancel."""
import os
import subprocess

import numpy as np
import pytest

import cuvslam_amd as ca

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def solver():
    return ca.SchurComplementBundlerGpu(loss=ca.LOSS_HUBER)


@pytest.mark.parametrize("row", range(24))
def test_a_non_positive_pivot_fails_at_every_row(solver, row):
    n = 24  # a full tile and a half one
    A = np.diag(np.arange(2.0, n + 2.0))
    if row:
        A[row, row - 1] = A[row - 1, row] = 1.0
    b = np.ones(n)
    x, rc = solver.debug_factor(A, b)
    assert rc == 0
    np.testing.assert_allclose(A @ x, b, atol=1e-13)
    # the row's pivot becomes -1 (row 0), or its square exceeds the product of the two diagonal entries
    B = A.copy()
    B[row, row] = -1.0 if row == 0 else 0.125 / A[row - 1, row - 1]
    assert np.linalg.eigvalsh(B)[0] < 0
    _, rc = solver.debug_factor(B, b)
    assert rc == ca.sba._lib.SBA_E_INFEASIBLE


@pytest.mark.parametrize("n", [6, 12, 18, 30, 48, 96])
@pytest.mark.parametrize("decades", [0, 4])
def test_rows_of_different_scale(solver, n, decades):
    rng = np.random.default_rng(100 * n + decades)
    M = rng.standard_normal((n, n))
    d = 2.0 ** np.round(np.linspace(-1, 1, n)[rng.permutation(n)] * decades * 3.32)  # exact in FP32
    A = np.float64(np.float32(M @ M.T / n + np.eye(n))) * d[:, None] * d[None, :]
    b = np.float64(np.float32(rng.standard_normal(n)))
    x, rc = solver.debug_factor(A, b)
    assert rc == 0
    # Cholesky's backward error is row- and column-scaled (Higham, Accuracy and Stability, 10.1): in the scaled unknowns
    # the error is at most 8 n (n + 1) eps times the condition number of the unit-diagonal matrix
    s = 1 / np.sqrt(np.diag(A))
    H = A * s[:, None] * s[None, :]
    y, ref = x / s, np.linalg.solve(H, b * s)
    assert np.linalg.norm(y - ref) <= 8 * n * (n + 1) * np.finfo(float).eps * np.linalg.cond(H) * np.linalg.norm(ref)


@pytest.mark.parametrize("n, row", [(12, 0), (12, 2), (24, 22), (48, 44), (48, 46), (96, 94)])
@pytest.mark.parametrize("a", [2.0, 3.0, 7.0, 11.0, 13.0])
def test_a_singular_pair_fails_or_stays_finite(solver, n, row, a):
    # the second pivot of the pair is zero but for rounding; (48, 46) and (96, 94) end in the last pivot of the last tile,
    # which no later pivot checks
    A = np.eye(n)
    A[row:row + 2, row:row + 2] = a
    x, rc = solver.debug_factor(A, np.ones(n))
    assert rc == ca.sba._lib.SBA_E_INFEASIBLE or np.isfinite(x).all()



def test_tile_factor_is_backward_stable():
    # the factor and inverse themselves: a solve shows their errors only through the condition of the system
    r = subprocess.run([os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "factor_tile_check")], text=True,
                       capture_output=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
