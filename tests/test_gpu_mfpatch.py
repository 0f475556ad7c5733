"""The matrix-free apply over element patches against the general gather
(NGSAMD_MF_PATCH=0) and the oracle: every order, structured meshes whose
element count leaves a partial tile, a partial patch or a single patch, 4- and
8-tile patches, unstructured meshes, every precision, FP32 and FP64 vectors,
accumulation, overlapping vectors, a changed coefficient, CG's inner product."""
import numpy as np
import pytest

from oracle import fe_oracle as O
from helpers import N, dvec, say

pytestmark = pytest.mark.gpu

import ngsolve_amd as ngs  # noqa: E402

TOL = {"f64": 1e-14, "f32": 2e-6, "f16x3": 2e-6, "f16": 4e-3, "bf16": 3e-2}


def build(monkeypatch, fes, kappa, precision, patch):
    monkeypatch.setenv("NGSAMD_MF_PATCH", "1" if patch else "0")
    u, v = fes.TnT()
    mat = ngs.BilinearForm(ngs.ElementCoefficient(kappa) * ngs.grad(u) * ngs.grad(v) * ngs.dx,
                           mf=ngs.MFOpts(precision=precision)).Assemble().mat
    assert N.MatrixFreePatchInfo(mat.op)[0] == (patch and (fes.mesh.ngmesh.dim, fes.order) != (2, 1))
    return mat


def compare(monkeypatch, mesh, p, precision):
    fes = ngs.H1(mesh, order=p, dirichlet=".*")
    rng = np.random.default_rng(7)
    kappa = np.exp(rng.standard_normal(mesh.ne))
    A, B = build(monkeypatch, fes, kappa, precision, True), build(monkeypatch, fes, kappa, precision, False)
    x = rng.uniform(-1, 1, fes.ndof)
    out = []
    for M in (A, B):
        dx, dy = dvec(x), dvec(np.full(fes.ndof, 7.0))
        M.op.mult(dx, dy)
        y = dy.download()
        M.op.mult(dx, dy)
        assert np.array_equal(y, dy.download())  # same bits every time
        fx, fy = dvec(x.astype(np.float32), 4), N.DeviceVector(fes.ndof, 4)
        M.op.mult_f32(fx, fy)
        y0 = rng.uniform(-1, 1, fes.ndof) if not out else out[0][3]
        da = dvec(y0)
        M.op.mult_add(-0.5, dx, da)
        out.append((y, fy.download().astype(np.float64), da.download(), y0))
    scale = np.abs(out[1][0]).max()
    t = TOL[precision]
    assert np.abs(out[0][0] - out[1][0]).max() <= t * scale
    assert np.abs(out[0][1] - out[1][1]).max() <= max(t, 1e-6) * scale
    assert np.abs(out[0][2] - out[1][2]).max() <= t * (scale + 1)
    return fes, kappa, A, x, out[0][0]


@pytest.mark.parametrize("precision", ["f64", "f32", "f16x3", "f16", "bf16"])
@pytest.mark.parametrize("dim,p", [(2, 1), (2, 2), (2, 3), (2, 4), (2, 5), (3, 1), (3, 2), (3, 3), (3, 4)])
def test_orders_and_precisions(device, monkeypatch, dim, p, precision):
    say(f"[mfpatch] {dim}D p={p} {precision}")
    mesh = ngs.MakeStructured2DMesh(nx=9, ny=7) if dim == 2 else ngs.MakeStructured3DMesh(nx=3, ny=4, nz=5)
    compare(monkeypatch, mesh, p, precision)


@pytest.mark.parametrize("cells", [(1, 1, 1), (2, 1, 1), (2, 2, 2), (5, 5, 5), (11, 3, 1)])
def test_partial_tiles_and_patches(device, monkeypatch, cells):
    # 6, 12, 48, 750 and 198 elements
    mesh = ngs.MakeStructured3DMesh(nx=cells[0], ny=cells[1], nz=cells[2])
    for p in (1, 4):
        compare(monkeypatch, mesh, p, "f64")


def test_eight_tile_patches(device, monkeypatch):
    # above 4 * 128 elements per CU: patches of 8 tiles
    mesh = ngs.MakeStructured3DMesh(nx=29, ny=27, nz=29)
    assert mesh.ne > 4 * 128 * 256
    for precision in ("f64", "f16x3"):
        A = compare(monkeypatch, mesh, 2, precision)[2]
        assert N.MatrixFreePatchInfo(A.op)[1:3] == (128, -(-mesh.ne // 128))


@pytest.mark.parametrize("name,p", [("square", 3), ("square", 5), ("cube", 3), ("cube", 4)])
def test_unstructured(device, monkeypatch, name, p):
    import os
    path = os.path.join(os.path.dirname(__file__), "golden", name + ".vol.gz")
    fes, kappa, A, x, y = compare(monkeypatch, ngs.Mesh(path), p, "f64")
    # the host assembly as an independent sum
    u, v = fes.TnT()
    a = ngs.BilinearForm(ngs.ElementCoefficient(kappa) * ngs.grad(u) * ngs.grad(v) * ngs.dx).Assemble().mat
    ref = O.csr_matvec(a.rowptr, a.cols, a.vals, x) if hasattr(O, "csr_matvec") else None
    if ref is None:
        import scipy.sparse as sp
        ref = sp.csr_matrix((a.vals, a.cols, a.rowptr)) @ x
    assert np.abs(y - ref).max() <= 1e-13 * np.abs(ref).max()


def test_overlapping_vectors_and_new_coefficient(device, monkeypatch):
    mesh = ngs.MakeStructured3DMesh(nx=4, ny=4, nz=4)
    fes, kappa, A, x, y = compare(monkeypatch, mesh, 3, "f64")
    d = dvec(x)
    A.op.mult(d, d)
    assert np.array_equal(d.download(), y)
    # the same with FP32 vectors, accumulating, and with vectors that overlap in part
    f = dvec(x, 4)
    fy = N.DeviceVector(fes.ndof, 4)
    A.op.mult_f32(f, fy)
    A.op.mult_f32(f, f)
    assert np.array_equal(f.download(), fy.download())
    a, d = dvec(x), dvec(x)
    A.op.mult_add(-0.5, d, d)
    other = dvec(x)
    A.op.mult_add(-0.5, other, a)
    assert np.array_equal(d.download(), a.download())
    n = fes.ndof
    for itemsize in (8, 4):
        for shift in (1, 37, n - 1):
            both = N.DeviceVector(n + shift, itemsize)
            for first in (0, shift):  # x before y, y before x
                host = np.zeros(n + shift)
                host[first:first + n] = x
                both.upload(host.astype(np.float64 if itemsize == 8 else np.float32))
                px = N.DeviceVector.wrap(both.ptr + itemsize * first, n, itemsize)
                py = N.DeviceVector.wrap(both.ptr + itemsize * (shift - first), n, itemsize)
                (A.op.mult if itemsize == 8 else A.op.mult_f32)(px, py)
                got = both.download()[shift - first:shift - first + n]
                assert np.array_equal(got, y if itemsize == 8 else fy.download())
    k2 = kappa[::-1].copy()
    B = build(monkeypatch, fes, k2, "f64", False)
    A.op.set_kappa(dvec(k2))
    dx, dy, dz = dvec(x), N.DeviceVector(fes.ndof, 8), N.DeviceVector(fes.ndof, 8)
    A.op.mult(dx, dy)
    B.op.mult(dx, dz)
    assert np.abs(dy.download() - dz.download()).max() <= 1e-14 * np.abs(dz.download()).max()


@pytest.mark.parametrize("cells", [(1, 1, 1), (6, 5, 7)])
def test_cg_inner_product(device, monkeypatch, cells):
    """CG takes <s, A s> from the patch kernel's partial sums (with one patch:
    no shared dofs)."""
    mesh = ngs.MakeStructured3DMesh(nx=cells[0], ny=cells[1], nz=cells[2])
    fes = ngs.H1(mesh, order=3, dirichlet=".*")
    rng = np.random.default_rng(5)
    kappa = np.exp(rng.standard_normal(mesh.ne))
    f = dvec(rng.uniform(0.5, 1, fes.ndof))
    sol, its = [], []
    for patch in (True, False):
        A = build(monkeypatch, fes, kappa, "f64", patch)
        if patch:
            on, size, npatch, shared = N.MatrixFreePatchInfo(A.op)
            assert size == 64 and npatch == -(-mesh.ne // 64) and (shared > 0) == (npatch > 1)
        C = A.CreateSmoother(fes.FreeDofs)
        u = N.DeviceVector(fes.ndof, 8)
        it, _ = N.CGSolve(A.op, C.op, f, u, True, 1e-12, -1.0, 2000, 16)
        sol.append(u.download())
        its.append(it)
    assert abs(its[0] - its[1]) <= 1
    # both stop at 1e-12 in the preconditioned residual
    assert np.linalg.norm(sol[0] - sol[1]) <= 1e-10 * max(np.linalg.norm(sol[1]), 1e-300)


@pytest.mark.parametrize("precision", ["f16", "bf16"])
@pytest.mark.parametrize("dim,p", [(2, 1), (2, 2), (2, 3), (2, 4), (2, 5), (3, 1), (3, 2), (3, 3), (3, 4)])
def test_16bit_rounding_of_every_class(device, monkeypatch, dim, p, precision):
    """One 16-bit term: each element class keeps the rounding of its own factor,
    with patches or not.  The same 16-bit operands leave the order of the sums over
    the elements; another class's rounded factor (3D p=4) moved results by 4e-5
    (FP16) and 4e-4 (BF16), FP64 entries rounded twice by up to 1e-5 (BF16)."""
    say(f"[mfpatch 16-bit] {dim}D p={p} {precision}")
    mesh = ngs.MakeStructured2DMesh(nx=31, ny=17) if dim == 2 else ngs.MakeStructured3DMesh(nx=5, ny=6, nz=7)
    check_16bit(monkeypatch, mesh, p, precision)


@pytest.mark.parametrize("precision", ["f16", "bf16"])
@pytest.mark.parametrize("cells", [(1, 1, 1), (2, 1, 1), (4, 2, 1), (2, 2, 2), (29, 27, 29)])
def test_16bit_tiles_of_two_references(device, monkeypatch, cells, precision):
    """3D p=4: tiles of either reference class, in a single patch that is not
    full (6, 12), one that is exactly (48 elements), more, and patches of 8 tiles."""
    mesh = ngs.MakeStructured3DMesh(nx=cells[0], ny=cells[1], nz=cells[2])
    A = check_16bit(monkeypatch, mesh, 4, precision)
    size = 128 if mesh.ne > 4 * 128 * 256 else 64
    assert N.MatrixFreePatchInfo(A.op)[1:3] == (size, -(-mesh.ne // (size - 16)))
    compare(monkeypatch, mesh, 4, precision)


def check_16bit(monkeypatch, mesh, p, precision):
    fes = ngs.H1(mesh, order=p, dirichlet=".*")
    rng = np.random.default_rng(11)
    kappa, x = np.exp(rng.standard_normal(mesh.ne)), rng.uniform(-1, 1, fes.ndof)
    out = []
    for patch in (True, False):
        M = build(monkeypatch, fes, kappa, precision, patch)
        dx, dy = dvec(x), N.DeviceVector(fes.ndof, 8)
        M.op.mult(dx, dy)
        out.append(dy.download())
        A = M if patch else A
    # the same products in FP32 sums of at most 60 terms: 60 * 2^-24 = 3.6e-6 of an
    # element's result at worst, its terms' errors independent 60^(1/2) * 2^-24 = 5e-7
    assert np.linalg.norm(out[0] - out[1]) <= 1e-6 * np.linalg.norm(out[1])
    return A


def shuffled(mesh, seed=3):
    """The mesh with its vertices renumbered and each element's given in another
    (even) order: elements of every vertex order."""
    m, rng = mesh.ngmesh, np.random.default_rng(seed)
    num = rng.permutation(m.nv)
    els, bnd = num[np.asarray(m.elements)], num[np.asarray(m.boundary)]
    even = {2: [(0, 1, 2), (1, 2, 0), (2, 0, 1)],
            3: [(0, 1, 2, 3), (1, 2, 0, 3), (2, 0, 1, 3), (1, 0, 3, 2), (0, 3, 1, 2), (3, 1, 0, 2), (2, 3, 0, 1),
                (0, 2, 3, 1), (3, 0, 2, 1), (3, 2, 1, 0), (1, 3, 2, 0), (2, 1, 3, 0)]}[m.dim]
    els = np.stack([e[list(even[k])] for e, k in zip(els, rng.integers(0, len(even), len(els)))])
    pts = np.zeros((m.nv, 3))
    pts[num, :m.dim] = np.asarray(m.coords)
    line = lambda head, a: [head + " ".join(str(v + 1) for v in r) for r in a]  # noqa: E731
    text = ["mesh3d", "dimension", str(m.dim)]
    if m.dim == 2:
        text += ["surfaceelements", str(len(els))] + line("1 1 0 0 3 ", els)
        text += ["edgesegmentsgi2", str(len(bnd))] + line("1 0 ", bnd)
    else:
        text += ["surfaceelements", str(len(bnd))] + line("1 1 1 0 3 ", bnd)
        text += ["volumeelements", str(len(els))] + line("1 4 ", els)
    text += ["points", str(m.nv)] + [" ".join(repr(float(v)) for v in r) for r in pts] + ["endmesh"]
    return ngs.Mesh(N.ReadVolMesh("\n".join(text)))


@pytest.mark.parametrize("precision", ["f64", "f32", "f16x3", "f16", "bf16"])
@pytest.mark.parametrize("dim,p", [(2, 2), (2, 3), (2, 4), (2, 5), (3, 1), (3, 2), (3, 3), (3, 4)])
def test_every_vertex_order(device, monkeypatch, dim, p, precision):
    """One reference class for all 6 or 24 vertex orders; one-term 16-bit operators
    whose factors round to more than two sets of numbers keep the general gather."""
    say(f"[mfpatch orders] {dim}D p={p} {precision}")
    mesh = shuffled(ngs.MakeStructured2DMesh(nx=23, ny=17) if dim == 2 else ngs.MakeStructured3DMesh(nx=6, ny=5, nz=7))
    fes = ngs.H1(mesh, order=p, dirichlet=".*")
    assert len(N.BuildClasses(fes.space, fes.integration_rule(2 * p))) == (6 if dim == 2 else 24)
    rng = np.random.default_rng(2)
    kappa, x = np.exp(rng.standard_normal(mesh.ne)), rng.uniform(-1, 1, fes.ndof)
    out = []
    for patch in "10":
        monkeypatch.setenv("NGSAMD_MF_PATCH", patch)
        u, v = fes.TnT()
        M = ngs.BilinearForm(ngs.ElementCoefficient(kappa) * ngs.grad(u) * ngs.grad(v) * ngs.dx,
                             mf=ngs.MFOpts(precision=precision)).Assemble().mat
        on = N.MatrixFreePatchInfo(M.op)[0]
        say(f"  patches: {on}")
        assert on == (patch == "1") or (patch == "1" and precision in ("f16", "bf16"))
        dx, dy = dvec(x), N.DeviceVector(fes.ndof, 8)
        M.op.mult(dx, dy)
        out.append(dy.download())
    # as in compare; the 16-bit operands are the same numbers (test_16bit_rounding_of_every_class)
    t = {"f64": 1e-14, "f32": 2e-6, "f16x3": 2e-6, "f16": 1e-6, "bf16": 1e-6}[precision]
    assert np.linalg.norm(out[0] - out[1]) <= t * np.linalg.norm(out[1])
