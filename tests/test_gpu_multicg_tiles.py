"""The vector kernels of the multi-RHS CG at the edges of their tiles: every
number of components, sizes around one workgroup's dofs (256 / K) and beyond
one pass of the whole grid, maxiter at and around the steps taken."""
import numpy as np
import pytest

import oracle
from helpers import N, dvec, say

pytestmark = pytest.mark.gpu


def _banded(n):
    """Diagonally dominant tridiagonal matrix (condition number below 5)."""
    rows = [[j for j in (i - 1, i, i + 1) if 0 <= j < n] for i in range(n)]
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int64)
    cols = np.concatenate(rows).astype(np.int32)
    diag = 3.0 + np.arange(n) % 3
    vals = np.where(cols == np.repeat(np.arange(n), np.diff(rp)), np.repeat(diag, np.diff(rp)), -1.0)
    return rp, cols, vals, diag


@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("n", [1, 31, 33, 85, 257, 40001])
def test_cg_multi_tiles(device, K, n):
    say(f"[multicg tiles] K={K} n={n}")
    rp, c, v, diag = _banded(n)
    rng = np.random.default_rng(n + K)
    F = rng.uniform(-1, 1, (n, K))
    A = N.CreateCSR(n, n, rp, c, v)
    pre = N.CreateJacobi(diag, np.ones(n, dtype=np.uint8))
    for maxiter in (0, 1, 16, 17, 200):
        dF, dU = dvec(F.ravel()), N.DeviceVector(n * K, 8)
        steps, hist = N.CGSolveMulti(A, pre, dF, dU, K, True, 1e-12, False, maxiter)
        assert steps <= maxiter + 1 and len(hist) == steps
        U = dU.download().reshape(n, K)
        if maxiter < 200:
            if maxiter == 0:
                assert np.all(U == 0.0)
            continue
        R = F - np.stack([oracle.spmv(rp, c, v, np.ascontiguousarray(U[:, j])) for j in range(K)], 1)
        # the test bounds ||(r_j, C r_j)_j|| by 1e-24 of its start and C is
        # within a factor 5 of a multiple of the identity
        assert np.linalg.norm(R) <= 1e-12 * 5 * K * np.linalg.norm(F)
        # beta falls by (sqrt 5 - 1)^2 / (sqrt 5 + 1)^2 < 0.15 a step at least
        assert steps <= 40
