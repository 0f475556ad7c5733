"""The batched runs SpMV at the edges of its blocks: run lengths 1 to 8 rows,
column lists from empty to longer than a block, problems of one row and of
many blocks; every block count per wavefront gives the same bits."""
import numpy as np
import pytest

import oracle
from helpers import N, dvec, say

pytestmark = pytest.mark.gpu


def block_diagonal(rng, sizes, rows, lens):
    rowptr, cols, off = [0], [], [0]
    for n in sizes:
        r = 0
        while r < n:
            c = off[-1] + np.sort(rng.choice(n, size=min(int(rng.choice(lens)), n), replace=False))
            for _ in range(min(int(rng.choice(rows)), n - r)):
                cols.append(c)
                rowptr.append(rowptr[-1] + len(c))
                r += 1
        off.append(off[-1] + n)
    cols = np.concatenate(cols).astype(np.int32)
    return np.array(rowptr, dtype=np.int64), cols, rng.uniform(-1, 1, len(cols)), np.array(off, dtype=np.int64)


@pytest.mark.parametrize("rows", [[2], [3], [4], [5], [6], [7], [8], [1, 2, 3, 4, 5, 6, 7, 8]])
@pytest.mark.parametrize("lens", [[0, 1, 7, 8, 9], [31, 33, 65, 128], [300, 341, 500, 300, 341, 500, 1500]])
def test_batch_runs_edges(device, monkeypatch, rows, lens):
    say(f"[batch runs] rows={rows} lens={lens}")
    rng = np.random.default_rng(23)
    rp, c, v, off = block_diagonal(rng, [1, 17, 2000, 5, 333], rows, lens)
    n = len(rp) - 1
    x, y0 = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
    ref = oracle.spmv(rp, c, v, x)
    # up to 1500 products of at most 1 in two orders of summation
    tol = 2 * 1500 * 2.0**-53 * max(np.abs(v).max(), 1.0) * 1500**0.5
    first = blocks = None
    for bn in ("1024", "2048", "4096"):
        monkeypatch.setenv("NGSAMD_SPMV_NNZ", bn)
        A = N.CreateBatchCSR(rp, c, v, off, True)
        dx, dy = dvec(x), N.DeviceVector(n, 8)
        A.mult(dx, dy)
        y = dy.download()
        assert np.abs(y - ref).max() <= tol
        first, blocks = (y, N.BatchInfo(A)[2]) if first is None else (first, blocks)
        assert N.BatchInfo(A)[2] == blocks  # the runs layout: the same blocks whatever a wavefront takes
        assert np.array_equal(y, first)
        dy.upload(y0)
        A.mult_add(-0.75, dx, dy)
        assert np.abs(dy.download() - (y0 - 0.75 * ref)).max() <= tol
