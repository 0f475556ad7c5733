"""The runs SpMV at the edges of its tasks: run lengths 1 to 8 rows, column
lists from empty to longer than one pass of 64 lanes, task counts around one
wavefront's and one workgroup's, the last run's padding lanes; plain,
accumulating and several vectors (each bit-identical to a single apply)."""
import numpy as np
import pytest

import oracle
from helpers import N, dvec, relerr_inf, say

pytestmark = pytest.mark.gpu


def runs_matrix(rng, nruns, rows, lens, width):
    rowptr, cols = [0], []
    for _ in range(nruns):
        L = int(rng.choice(lens))
        c = np.sort(rng.choice(width, size=min(L, width), replace=False))
        for _ in range(int(rng.choice(rows))):
            cols.append(c)
            rowptr.append(rowptr[-1] + len(c))
    cols = np.concatenate(cols).astype(np.int32)
    return np.array(rowptr, dtype=np.int64), cols, rng.uniform(-1, 1, len(cols))


@pytest.mark.parametrize("rows", [[1], [2], [3], [4], [5], [6], [7], [8], [1, 2, 3, 4, 5, 6, 7, 8]])
@pytest.mark.parametrize("lens", [[0, 1, 7, 8, 9], [31, 32, 33, 64, 65], [128, 255, 512, 513, 700]])
@pytest.mark.parametrize("nruns", [1, 9, 333])
def test_runs_edges(device, monkeypatch, rows, lens, nruns):
    monkeypatch.setenv("NGSAMD_SPMV", "runs")
    say(f"[runs] rows={rows} lens={lens} nruns={nruns}")
    rng = np.random.default_rng(17)
    width = 800
    rp, c, v = runs_matrix(rng, nruns, rows, lens, width)
    n = len(rp) - 1
    A = N.CreateCSR(n, width, rp, c, v)
    x = rng.uniform(-1, 1, width)
    ref = oracle.spmv(rp, c, v, x)
    scale = max(np.abs(ref).max(), 1.0)
    dx, dy = dvec(x), N.DeviceVector(n, 8)
    A.mult(dx, dy)
    y = dy.download()
    # 700 products of at most 1, two orders of summation
    assert np.abs(y - ref).max() <= 1e-13 * scale
    y0 = rng.uniform(-1, 1, n)
    dy.upload(y0)
    A.mult_add(-0.75, dx, dy)
    assert np.abs(dy.download() - (y0 - 0.75 * ref)).max() <= 1e-13 * scale
    for K in (1, 2, 3, 4, 7, 8):
        X = rng.uniform(-1, 1, (width, K))
        X[:, K - 1] = x
        dX, dY = dvec(X.ravel()), N.DeviceVector(n * K, 8)
        N.CSRMultMulti(A, dX, dY, K)
        assert np.array_equal(dY.download().reshape(n, K)[:, K - 1], y)


def test_runs_infinite_entries_stay_in_their_columns(device, monkeypatch):
    """Padding lanes repeat a run's last column: an infinite x entry there
    gives +-inf in its rows, as the plain sum does, and nothing elsewhere."""
    monkeypatch.setenv("NGSAMD_SPMV", "runs")
    rng = np.random.default_rng(3)
    rp, c, v = runs_matrix(rng, 50, [2, 3], [20, 35], 100)
    n = len(rp) - 1
    v = np.abs(v) + 0.1
    x = rng.uniform(0.5, 1, 100)
    hit = int(c[rp[1] - 1])  # last column of the first run
    x[hit] = np.inf
    A = N.CreateCSR(n, 100, rp, c, v)
    dx, dy = dvec(x), N.DeviceVector(n, 8)
    A.mult(dx, dy)
    y = dy.download()
    has = np.array([hit in c[rp[i]:rp[i + 1]] for i in range(n)])
    assert np.all(np.isposinf(y[has])) and np.all(np.isfinite(y[~has]))
    x[hit] = 0.0
    xr = x.copy()
    assert relerr_inf(y[~has], oracle.spmv(rp, c, v, xr)[~has]) < 1e-13
