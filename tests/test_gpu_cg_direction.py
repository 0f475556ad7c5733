"""CG on a small CSR operator, whose kernel forms the search direction (two
kernels an iteration): iteration counts, residual history and solutions against
the oracle's PCG where the first check, the iteration limit or the breakdown
test ends the loop, with and without an initial guess, with graphs of 2 and 16
iterations and without."""
import numpy as np
import pytest

import oracle
from oracle import fe_oracle as O
from helpers import N, dvec, problem, say

pytestmark = pytest.mark.gpu


def pcg(P, inv, f, u0, tol, maxiter):
    A = lambda t: oracle.spmv(P["rowptr"], P["cols"], P["vals"], t)  # noqa: E731
    g = f - A(u0)
    u, its, res = O.pcg(A, inv, g, tol=tol, maxiter=maxiter)
    return u0 + u, its, res


@pytest.mark.parametrize("dim,n,p", [(2, 2, 2), (2, 9, 3), (2, 20, 5), (3, 4, 3)])
@pytest.mark.parametrize("maxiter", [1, 2, 3, 17, 2000])
@pytest.mark.parametrize("chunk", [0, 2, 16])
def test_against_oracle(device, monkeypatch, dim, n, p, maxiter, chunk):
    say(f"[cg direction] {dim}D {n} p={p} maxiter={maxiter} chunk={chunk}")
    monkeypatch.setenv("NGSAMD_SPMV", "runs")  # at p=2 the runs save too few column numbers
    P = problem(dim, n, p, seed_kappa=4)
    A = N.CreateCSR(P["ndof"], P["ndof"], P["rowptr"], P["cols"], P["vals"])
    assert N.CSRInfo(A)[2]  # its product forms the direction
    free = P["fes"].freedofs.astype(np.uint8)
    diag, inv = O.jacobi_invdiag(P["rowptr"], P["cols"], P["vals"], free)
    C = N.CreateJacobi(diag, free)
    rng = np.random.default_rng(8)
    f = np.where(free != 0, rng.uniform(-1, 1, P["ndof"]), 0.0)
    for u0 in (None, rng.uniform(-1, 1, P["ndof"])):
        start = np.zeros(P["ndof"]) if u0 is None else u0
        ref, its_ref, res_ref = pcg(P, inv, f, start, 1e-10, maxiter)
        du = dvec(start)
        its, res = N.CGSolve(A, C, dvec(f), du, u0 is None, 1e-10, -1.0, maxiter, chunk)
        assert abs(its - its_ref) <= (1 if its_ref < maxiter else 0)
        assert np.allclose(res[:3], res_ref[:3], rtol=1e-9, atol=0)
        if its == its_ref:
            assert np.abs(du.download() - ref).max() <= 1e-9 * max(np.abs(ref).max(), 1e-300)


@pytest.mark.parametrize("dim,n,p,forms", [(2, 128, 3, True), (3, 14, 4, True), (2, 200, 3, False)])
@pytest.mark.parametrize("chunk", [0, 16])
def test_at_the_limit(device, dim, n, p, forms, chunk):
    """The largest grids whose product forms the direction (1024 workgroups, up to
    28 tasks each), and the first that leaves it to a kernel of its own."""
    say(f"[cg direction] {dim}D {n} p={p} chunk={chunk}")
    P = problem(dim, n, p, seed_kappa=4)
    A = N.CreateCSR(P["ndof"], P["ndof"], P["rowptr"], P["cols"], P["vals"])
    layout, workgroups, formed, _ = N.CSRInfo(A)
    assert layout == 2 and formed == forms and (workgroups == 1024) == forms
    free = P["fes"].freedofs.astype(np.uint8)
    diag, inv = O.jacobi_invdiag(P["rowptr"], P["cols"], P["vals"], free)
    rng = np.random.default_rng(9)
    f = np.where(free != 0, rng.uniform(-1, 1, P["ndof"]), 0.0)
    u0 = np.where(free != 0, rng.uniform(-1, 1, P["ndof"]), 0.0)
    ref, its_ref, res_ref = pcg(P, inv, f, u0, 1e-10, 18)
    du = dvec(u0)
    its, res = N.CGSolve(A, N.CreateJacobi(diag, free), dvec(f), du, False, 1e-10, -1.0, 18, chunk)
    assert its == its_ref == 18
    assert np.allclose(res, res_ref, rtol=1e-9, atol=0)
    assert np.abs(du.download() - ref).max() <= 1e-9 * np.abs(ref).max()


def test_zero_right_hand_side(device, monkeypatch):
    monkeypatch.setenv("NGSAMD_SPMV", "runs")
    P = problem(2, 6, 2, seed_kappa=1)
    A = N.CreateCSR(P["ndof"], P["ndof"], P["rowptr"], P["cols"], P["vals"])
    assert N.CSRInfo(A)[2]
    free = P["fes"].freedofs.astype(np.uint8)
    diag, _ = O.jacobi_invdiag(P["rowptr"], P["cols"], P["vals"], free)
    C = N.CreateJacobi(diag, free)
    du = dvec(np.full(P["ndof"], 3.0))
    its, res = N.CGSolve(A, C, dvec(np.zeros(P["ndof"])), du, True, 1e-10, -1.0, 100, 16)
    assert its == 1 and res[0] == 0.0 and not du.download().any()


@pytest.mark.parametrize("layout", ["runs", "stream"])
@pytest.mark.parametrize("n,chunk", [(1, 0), (5000, 16), (250000, 0), (250000, 16)])
def test_breakdown_leaves_the_solution(device, monkeypatch, layout, n, chunk):
    """<s, A s> = 0 at the first step: every workgroup of the update sees it, or
    the flag that the first one sets, and none of them touches u."""
    say(f"[cg breakdown] {layout} n={n} chunk={chunk}")
    monkeypatch.setenv("NGSAMD_SPMV", layout)
    # pairs of rows with two columns each, all values 0
    i = np.arange(n, dtype=np.int32)
    cols = np.stack([i // 2 * 2, np.minimum(i // 2 * 2 + 1, n - 1)], 1)
    cols = cols[:, :1] if n == 1 else cols
    rp = np.arange(n + 1, dtype=np.int64) * cols.shape[1]
    A = N.CreateCSR(n, n, rp, np.ascontiguousarray(cols.ravel()), np.zeros(cols.size))
    C = N.CreateJacobi(np.full(n, 2.0), None)
    u0 = np.random.default_rng(1).uniform(-1, 1, n)
    for _ in range(3):
        du = dvec(u0)
        its, res = N.CGSolve(A, C, dvec(np.ones(n)), du, False, 1e-10, -1.0, 50, chunk)
        assert its == 1 and res[0] == pytest.approx(np.sqrt(n / 2), rel=1e-12)
        assert np.array_equal(du.download(), u0)
