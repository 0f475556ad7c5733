"""The work that a program built on ngsolve_amd has the GPU do, as a list of
cases with their inputs, one pass of each, and what the result should be.

The discretisations are the structured 2D / 3D simplex meshes of the
benchmark, the tests and the examples (64^2 p=3, 128^2 p=3, 32^3 p=4, the
batch of 2D problems with nx in 8..96 and p in 1..5) and ragged sizes between
them; the coefficient is one lognormal value per element throughout.

Kinds of case
  csr       y = A x with the assembled FP64 matrix (BaseMatrix.Mult)
  mf        y = A x with the matrix-free operator, in each of its precisions,
            on FP64 vectors or on FP32 vectors (as inner operators take them)
  cg        Jacobi-, two-level- or block-Jacobi-preconditioned device CG to
            1e-10 on the CSR or the matrix-free operator
  cg_multi  several right-hand sides in lockstep
  ir        FP64 refinement to 1e-10 around a lower-precision matrix-free CG
  batch     many small 2D problems solved together, FP64 or refined from FP32
  adjoint   forward solve, functional and gradient through torch.autograd
  assemble  sparsity pattern and matrix values built on the device
"""
import math

import numpy as np
import torch

import ngsolve_amd as ngs
from ngsolve_amd import batch as ngbatch
from ngsolve_amd._native import N
from ngsolve_amd.autograd import ApplySymmetric, PoissonProblem, SolvePoisson
from ngsolve_amd.la import BlockJacobiPrecond, LowOrderBlock, MultiGrid, TwoLevelPrecond

TOL = 1e-10  # relative tolerance of every solve


def listed():
    return [
        # one product in an interactive 2D problem: the launch is what counts
        {"name": "csr_2d_p3_small", "kind": "csr", "dim": 2, "nx": 61, "ny": 67, "nz": 0, "p": 3},
        # the benchmark's product: 2.1M dofs, 159M nonzeros
        {"name": "csr_3d_p4_large", "kind": "csr", "dim": 3, "nx": 32, "ny": 32, "nz": 32, "p": 4},
        # the same operator applied without a matrix
        {"name": "mf_f64_3d_p4_large", "kind": "mf", "dim": 3, "nx": 32, "ny": 32, "nz": 32, "p": 4,
         "precision": "f64", "vec": 64},
        # the product that a refinement's inner iteration makes, odd sizes
        {"name": "mf_f16x3_3d_p3", "kind": "mf", "dim": 3, "nx": 23, "ny": 19, "nz": 27, "p": 3,
         "precision": "f16x3", "vec": 32},
        # high order in 2D with the reference's fp32 option, odd sizes
        {"name": "mf_f32_2d_p5", "kind": "mf", "dim": 2, "nx": 181, "ny": 203, "nz": 0, "p": 5,
         "precision": "f32", "vec": 64},
        # the reference's CPU-sized problem, solved: hundreds of small dependent steps
        {"name": "cg_csr_2d_p3", "kind": "cg", "dim": 2, "nx": 64, "ny": 64, "nz": 0, "p": 3, "op": "csr",
         "pre": "jacobi"},
        # a 3D solve with the P1 multigrid as coarse part
        {"name": "cg_csr_3d_p4_twolevel", "kind": "cg", "dim": 3, "nx": 20, "ny": 16, "nz": 24, "p": 4, "op": "csr",
         "pre": "twolevel"},
        # four load cases of one matrix
        {"name": "cg_multi4_3d_p4", "kind": "cg_multi", "dim": 3, "nx": 15, "ny": 17, "nz": 14, "p": 4, "nrhs": 4},
        # the benchmark's mixed-precision solve
        {"name": "ir_f16x3_3d_p4_large", "kind": "ir", "dim": 3, "nx": 32, "ny": 32, "nz": 32, "p": 4,
         "precision": "f16x3"},
        # a parameter study: many independent small problems
        {"name": "batch48_mixed", "kind": "batch", "nprob": 48, "nx_min": 8, "nx_max": 96, "p_min": 1, "p_max": 5,
         "mixed": True},
        # a gradient for an inverse problem: forward and adjoint solve
        {"name": "adjoint_2d_p3", "kind": "adjoint", "dim": 2, "nx": 128, "ny": 128, "nz": 0, "p": 3},
        # a new matrix after the coefficient or the mesh has changed
        {"name": "assemble_3d_p3", "kind": "assemble", "dim": 3, "nx": 13, "ny": 11, "nz": 12, "p": 3},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mesh(rng, dim, els_lo, els_hi, even=False):
    """Ragged cells per direction for a number of elements drawn over its
    logarithm (even: multiples of 4, for a multigrid hierarchy of three levels)."""
    cells = _log_int(rng, els_lo, els_hi) / (2 if dim == 2 else 6)
    n = [max(2, cells ** (1.0 / dim) * math.exp(rng.uniform(-0.3, 0.3))) for _ in range(dim)]
    n = [4 * max(1, int(round(v / 4))) if even else int(round(v)) for v in n]
    return {"dim": dim, "nx": n[0], "ny": n[1], "nz": n[2] if dim == 3 else 0}


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def draw(rng):
    most = max(_cost(c) for c in listed())
    case = _draw(rng)
    while _cost(case) > most:
        case = _draw(rng)
    return case


def _draw(rng):
    kind = rng.choice(["csr", "csr", "mf", "mf", "mf", "cg", "cg", "cg_multi", "ir", "batch", "adjoint", "assemble"])
    dim = rng.choice([2, 3])
    p = rng.randint(1, 5) if dim == 2 else rng.randint(1, 4)
    if kind == "csr":
        return {"kind": kind, **_mesh(rng, dim, 1500, 120000), "p": p}
    if kind == "mf":
        precision = rng.choice(["f64", "f64", "f32", "f16x3", "bf16", "f16"])
        return {"kind": kind, **_mesh(rng, dim, 1500, 150000), "p": p, "precision": precision,
                "vec": 64 if precision == "f64" else rng.choice([32, 64])}
    if kind == "cg":
        pre = rng.choice(["jacobi", "jacobi", "twolevel", "block"])
        op = "csr" if pre != "jacobi" else rng.choice(["csr", "mf"])
        p = max(p, 2) if pre != "jacobi" else p
        return {"kind": kind, **_mesh(rng, dim, 1500, 25000, even=pre == "twolevel"), "p": p, "op": op, "pre": pre}
    if kind == "cg_multi":
        return {"kind": kind, **_mesh(rng, dim, 1500, 20000), "p": p, "nrhs": rng.randint(2, 8)}
    if kind == "ir":
        return {"kind": kind, **_mesh(rng, dim, 3000, 60000), "p": max(p, 2),
                "precision": rng.choice(["f32", "f16x3", "bf16"])}
    if kind == "batch":
        lo = rng.randint(8, 40)
        return {"kind": kind, "nprob": _log_int(rng, 6, 40), "nx_min": lo, "nx_max": lo + rng.randint(4, 50),
                "p_min": 1, "p_max": rng.randint(2, 5), "mixed": rng.random() < 0.5}
    if kind == "adjoint":
        return {"kind": kind, **_mesh(rng, 2, 2000, 30000), "p": rng.randint(1, 4)}
    return {"kind": kind, **_mesh(rng, dim, 1000, 12000), "p": p}


# ---------------------------------------------------------------- preparation

def _device(a, dtype=torch.float64):
    """A torch tensor of the values and the library's vector over the same memory."""
    t = torch.tensor(np.ascontiguousarray(a), dtype=dtype, device="cuda").reshape(-1)
    torch.cuda.synchronize()  # the library works on a stream of its own
    return t, N.DeviceVector.wrap(t.data_ptr(), t.numel(), t.element_size())


def _space(case):
    if case["dim"] == 2:
        mesh = ngs.MakeStructured2DMesh(nx=case["nx"], ny=case["ny"])
    else:
        mesh = ngs.MakeStructured3DMesh(nx=case["nx"], ny=case["ny"], nz=case["nz"])
    return mesh, ngs.H1(mesh, order=case["p"], dirichlet=".*")


def _kappa(mesh, rng):
    return np.exp(rng.standard_normal(mesh.ne))


def _form(fes, kappa, **kw):
    u, v = fes.TnT()
    return ngs.BilinearForm(ngs.ElementCoefficient(kappa) * ngs.grad(u) * ngs.grad(v) * ngs.dx, **kw)


def _vector(a):
    t, v = _device(a)
    return t, ngs.BaseVector(len(a), _dev=v)


def _load(fes):
    """The load vector of f = 1 (one point rule of order p integrates it exactly)."""
    v = fes.TestFunction()
    return ngs.LinearForm(1 * v * ngs.dx(intorder=fes.order)).Assemble().vec.NumPy().copy()


def _loads(fes, rng, nrhs):
    """Load vectors of f = 1 scaled dof by dof, one column each."""
    return _load(fes)[:, None] * rng.uniform(0.5, 1.5, (fes.ndof, nrhs))


def _problems(case, seed):
    """The batch: sizes and orders belong to the case, coefficients and loads to the seed."""
    sizes, rng = np.random.default_rng(5), np.random.default_rng(seed)
    out = []
    for _ in range(case["nprob"]):
        nx = int(sizes.integers(case["nx_min"], case["nx_max"] + 1))
        p = int(sizes.integers(case["p_min"], case["p_max"] + 1))
        out.append(ngbatch.Problem(nx, p, np.exp(rng.standard_normal(2 * nx * nx)),
                                   rng.uniform(-1.0, 1.0, _counts(2, nx, nx, 0, p)[1])))
    return out


def _bits(fes):
    return np.asarray(fes.space.freedofs).astype(bool)


def _adjoint_inputs(case, seed):
    rng = np.random.default_rng(seed)
    mesh, fes = _space(case)
    kappa = np.exp(0.5 * rng.standard_normal(mesh.ne))
    u_obs = 0.05 * rng.standard_normal(fes.ndof) * _bits(fes)
    return mesh, fes, kappa, u_obs


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    s = {"kind": kind}
    if kind == "batch":
        s["solver"] = ngbatch.BatchSolver(_problems(case, seed), with_f32=case["mixed"])
        s["mixed"] = case["mixed"]
        return s
    if kind == "adjoint":
        mesh, fes, kappa, u_obs = _adjoint_inputs(case, seed)
        u, v = fes.TnT()
        s["problem"] = PoissonProblem(fes, _load(fes), tol=TOL)
        s["mass"] = ngs.BilinearForm(u * v * ngs.dx).Assemble().mat
        s["kappa"] = torch.tensor(kappa, device="cuda", requires_grad=True)
        s["u_obs"] = torch.tensor(u_obs, device="cuda")
        return s
    mesh, fes = _space(case)
    kappa = _kappa(mesh, rng)
    if kind == "assemble":
        s["fes"], s["kappa"] = fes, kappa
        return s
    if kind in ("csr", "mf"):
        x = rng.uniform(-1.0, 1.0, fes.ndof)
        if kind == "csr":
            s["A"] = _form(fes, kappa, device_assembly=True).Assemble().mat
        else:
            s["A"] = _form(fes, kappa, mf=ngs.MFOpts(precision=case["precision"])).Assemble().mat
        if kind == "mf" and case["vec"] == 32:
            s["in"], s["x"] = _device(x, torch.float32)
            s["out"], s["y"] = _device(np.zeros(fes.ndof), torch.float32)
            s["kind"] = "mf32"
        else:
            s["in"], s["x"] = _vector(x)
            s["out"], s["y"] = _vector(np.zeros(fes.ndof))
        return s
    # solves
    free = fes.FreeDofs
    if kind == "cg_multi":
        a = _form(fes, kappa).Assemble().mat
        k = case["nrhs"]
        s["A"], s["pre"], s["nrhs"] = a, a.CreateSmoother(free), k
        s["in"], s["f"] = _device(_loads(fes, rng, k))
        s["out"], s["u"] = _device(np.zeros(fes.ndof * k))
        return s
    s["in"], s["f"] = _vector(_loads(fes, rng, 1)[:, 0])
    s["out"], s["u"] = _vector(np.zeros(fes.ndof))
    if kind == "ir":
        hi = _form(fes, kappa, mf=ngs.MFOpts()).Assemble().mat
        lo = _form(fes, kappa, mf=ngs.MFOpts(precision=case["precision"])).Assemble().mat
        s["inv"] = ngs.IRCGSolver(hi, lo, hi.CreateSmoother(free), tol=TOL)
        s["kind"] = "solve"
        return s
    if case["op"] == "mf":
        a = _form(fes, kappa, mf=ngs.MFOpts()).Assemble().mat
    else:
        a = _form(fes, kappa).Assemble().mat
    pre = a.CreateSmoother(free)
    if case["pre"] == "twolevel":
        dims = (case["nx"], case["ny"]) if case["dim"] == 2 else (case["nx"], case["ny"], case["nz"])
        vertices = _bits(fes)[:mesh.nv]
        pre = TwoLevelPrecond(pre, MultiGrid(LowOrderBlock(a, mesh.nv), dims, vertices))
    elif case["pre"] == "block":
        pre = BlockJacobiPrecond(a, fes.CreateSmoothingBlocks())
    s["inv"] = ngs.DevCGSolver(a, pre, tol=TOL, maxiter=20000)
    s["kind"] = "solve"
    return s


# ----------------------------------------------------------------------- pass

def run(s):
    kind = s["kind"]
    if kind in ("csr", "mf"):
        s["y"].data = s["A"] * s["x"]
        return s["out"]
    if kind == "mf32":
        s["A"].op.mult_f32(s["x"], s["y"])
        return s["out"]
    if kind == "solve":
        s["u"].data = s["inv"] * s["f"]
        return s["out"]
    if kind == "cg_multi":
        N.CGSolveMulti(s["A"].op, s["pre"].op, s["f"], s["u"], s["nrhs"], tol=TOL, maxiter=20000)
        return s["out"]
    if kind == "batch":
        if s["mixed"]:
            s["solver"].solve_mixed(tol=TOL)
        else:
            s["solver"].solve_fp64(tol=TOL)
        return s["solver"].solution()
    if kind == "adjoint":
        kappa = s["kappa"]
        kappa.grad = None
        u = SolvePoisson.apply(kappa, s["problem"])
        r = u - s["u_obs"]
        j = 0.5 * torch.dot(r, ApplySymmetric.apply(r, s["mass"].op))
        j.backward()
        return {"u": u.detach(), "J": j.detach(), "grad": kappa.grad}
    # assemble
    a = _form(s["fes"], s["kappa"], device_assembly=True).Assemble().mat
    return {"rowptr": a.rowptr, "cols": a.cols, "vals": a.vals}


# ----------------------------------------------------------------------- work

def _counts(dim, nx, ny, nz, p):
    """(elements, dofs, nonzeros, dofs per element) of the H1 space of order p."""
    if dim == 2:
        simplices = [(nx + 1) * (ny + 1), 3 * nx * ny + nx + ny, 2 * nx * ny]
    else:
        q, f, e = nx * ny * nz, nx * ny + ny * nz + nx * nz, nx + ny + nz
        simplices = [(nx + 1) * (ny + 1) * (nz + 1), 7 * q + 3 * f + e, 12 * q + 2 * f, 6 * q]
    closed = [math.comb(p + k, k) for k in range(dim + 1)]  # dofs of a closed k-simplex
    own, pairs = [], []  # dofs / ordered pairs of dofs that no smaller simplex holds
    for k in range(dim + 1):
        own.append(closed[k] - sum(math.comb(k + 1, j + 1) * own[j] for j in range(k)))
        pairs.append(closed[k] ** 2 - sum(math.comb(k + 1, j + 1) * pairs[j] for j in range(k)))
    return (simplices[dim], sum(a * b for a, b in zip(simplices, own)),
            sum(a * b for a, b in zip(simplices, pairs)), closed[dim])


def _iterations(dim, n, p, pre="jacobi"):
    """About the CG steps to TOL with lognormal coefficients on n cells per
    direction (measured: 2D 64^2 p=3 420, 128^2 p=3 670 to 840, 3D 32^3 p=4
    320 to 360, 20x16x24 p=4 with the two-level preconditioner 216)."""
    if pre == "twolevel":
        return 210
    return (2.1 * n * p if dim == 2 else 6.0 * n + 30 * p) + 20


def _apply_work(case, matfree, itemsize=8):
    dim, p = case["dim"], case["p"]
    ne, n, nnz, nd = _counts(dim, case["nx"], case["ny"], case["nz"], p)
    if matfree:
        r = math.comb(p - 1 + dim, dim)  # gradients: polynomials of degree p-1
        return (ne * (nd * 4 + (dim * (dim + 1) // 2 + 1) * 8) + 2 * n * itemsize,
                ne * (4 * dim * r * nd + 2 * dim * dim * r))
    return nnz * 12 + (n + 1) * 4 + 2 * n * 8, 2 * nnz


def work(case):
    kind = case["kind"]
    if kind in ("csr", "mf"):
        b, f = _apply_work(case, kind == "mf", case.get("vec", 64) // 8)
        return {"bytes": b, "flops": f}
    if kind == "batch":
        nx, p = 0.5 * (case["nx_min"] + case["nx_max"]), 0.5 * (case["p_min"] + case["p_max"])
        _, n, nnz, _ = _counts(2, int(nx), int(nx), 0, int(round(p)))
        its = case["nprob"] * _iterations(2, nx, p)
        return {"bytes": its * (nnz * (8 if case["mixed"] else 12) + 7 * n * 8), "flops": its * (2 * nnz + 12 * n)}
    ne, n, nnz, nd = _counts(case["dim"], case["nx"], case["ny"], case["nz"], case["p"])
    if kind == "assemble":
        return {"bytes": ne * (nd * 4 + 56) + nnz * 12 + n * 8, "flops": ne * nd * nd * 12}
    cells = (case["nx"] * case["ny"] * max(case["nz"], 1)) ** (1.0 / case["dim"])
    its = _iterations(case["dim"], cells, case["p"], case.get("pre", "jacobi"))
    if kind == "cg_multi":
        k = case["nrhs"]
        return {"bytes": its * (nnz * 12 + k * 7 * n * 8), "flops": its * k * (2 * nnz + 12 * n)}
    matfree = kind in ("ir", "adjoint") or case.get("op") == "mf"
    b, f = _apply_work(case, matfree, 4 if kind == "ir" else 8)
    vec = 4 if kind == "ir" else 8
    solves = 2 if kind == "adjoint" else 1
    # per step: the operator, and u, d, w and s updated from one another
    return {"bytes": solves * its * (b + 5 * n * vec), "flops": solves * its * (f + 12 * n)}


# ------------------------------------------------------------------ tolerance

def tolerance(case):
    """About four times what two orders of summation, or two orders of the
    steps of a solve, were seen to differ by (FP64 products 1e-16 to 4e-16
    from 64-bit torch, FP32 and split FP16 1e-7 to 2e-7, FP16 4e-4, BF16
    2e-3; "max" by the largest of some 1e5 values)."""
    kind = case["kind"]
    if kind == "csr":
        return {"rel": 2e-15, "max": 1e-13}
    if kind == "mf":
        return {"f64": {"rel": 2e-15, "max": 1e-13}, "f32": {"rel": 1e-6, "max": 2e-5},
                "f16x3": {"rel": 1e-6, "max": 2e-5}, "f16": {"rel": 2e-3, "max": 0.05},
                "bf16": {"rel": 1e-2, "max": 0.25}}[case["precision"]]
    if kind == "assemble":
        return {"rel": 1e-15, "max": 1e-13}
    # solves stop at TOL in the residual, perhaps one step earlier or later:
    # 1e-9 from the exact solution with the two-level preconditioner, 1e-12
    # to 3e-10 with the others
    return {"rel": 1e-8, "max": 1e-6}


# ---------------------------------------------------------------------- exact

class _Elements:
    """The H1 form in plain torch, FP64: element matrices from the tabulated
    shape functions, products by gather and scatter over the elements."""

    def __init__(self, fes, kappa, mass=False):
        p, mesh = fes.order, fes.mesh.ngmesh
        ir = fes.integration_rule(2 * p if mass else max(2 * p - 2, 0))
        w = torch.tensor(np.asarray(ir.weights), device="cuda")
        detj, ginv = (torch.tensor(np.asarray(a), device="cuda") for a in N.ComputeGeometry(mesh))
        self.n = fes.ndof
        self.free = torch.tensor(_bits(fes), device="cuda")
        dofs, mats = [], []
        el_dofs = torch.tensor(np.asarray(fes.space.el_dofs), device="cuda").long()
        self.order = []
        for c in N.BuildClasses(fes.space, ir):
            e = torch.tensor(np.asarray(c["elements"]), device="cuda").long()
            dofs.append(el_dofs[e])
            self.order.append(e)
            if mass:
                f = torch.tensor(np.asarray(c["shape"]), device="cuda")  # [q][i]
                ref = (f * w[:, None]).T @ f
                mats.append(detj[e].abs()[:, None, None] * ref)
            else:
                b = torch.tensor(np.asarray(c["bmat"]), device="cuda")  # [q][i][d]
                m = torch.zeros(len(e), b.shape[1], b.shape[1], dtype=torch.float64, device="cuda")
                g = kappa[e, None, None] * detj[e].abs()[:, None, None] * ginv[e]
                for d in range(b.shape[2]):
                    for k in range(b.shape[2]):
                        m += g[:, d, k][:, None, None] * ((b[:, :, d] * w[:, None]).T @ b[:, :, k])
                mats.append(m)
        self.dofs, self.mats, self.order = torch.cat(dofs), torch.cat(mats), torch.cat(self.order)

    def apply(self, x):
        y = torch.zeros(self.n, *x.shape[1:], dtype=torch.float64, device="cuda")
        xe = x[self.dofs]
        if x.dim() == 1:
            ye = (self.mats * xe[:, None, :]).sum(2)
        else:
            ye = torch.stack([(self.mats * xe[:, None, :, j]).sum(2) for j in range(x.shape[1])], 2)
        return y.index_add_(0, self.dofs.reshape(-1), ye.reshape(-1, *x.shape[1:]))

    def diagonal(self):
        d = torch.zeros(self.n, dtype=torch.float64, device="cuda")
        return d.index_add_(0, self.dofs.reshape(-1), torch.diagonal(self.mats, dim1=1, dim2=2).reshape(-1))

    def solve(self, f):
        """Jacobi-PCG on the free dofs to the limit of FP64."""
        inv = torch.where(self.free, 1.0 / self.diagonal(), 0.0)
        u, r = torch.zeros_like(f), f.clone()
        z = inv * r
        s, rz = z.clone(), torch.dot(r, z)
        first = float(rz)
        for k in range(20000):
            if first == 0.0 or (k % 16 == 0 and float(rz) <= 1e-26 * first):
                break
            w = self.apply(s)
            alpha = rz / torch.dot(s, w)
            u += alpha * s
            r -= alpha * w
            z = inv * r
            rz, old = torch.dot(r, z), rz
            s = z + (rz / old) * s
        return u

    def csr(self):
        """Row pointers, columns and values of the assembled matrix."""
        nd = self.dofs.shape[1]
        keys = (self.dofs[:, :, None] * self.n + self.dofs[:, None, :]).reshape(-1)
        pat, at = torch.unique(keys, return_inverse=True)
        vals = torch.zeros(len(pat), dtype=torch.float64, device="cuda").index_add_(0, at, self.mats.reshape(-1))
        rows = pat // self.n
        rowptr = torch.zeros(self.n + 1, dtype=torch.int64, device="cuda")
        rowptr[1:] = torch.cumsum(torch.bincount(rows, minlength=self.n), 0)
        assert nd == self.mats.shape[1]
        return rowptr, (pat % self.n).to(torch.int32), vals


def _tensor(a):
    return torch.tensor(np.ascontiguousarray(a), device="cuda")


def exact(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "batch":
        out = []
        problems = _problems(case, seed)
        if sum(pr.ndof for pr in problems) > 1_000_000:
            return None  # one after the other takes too long
        for pr in problems:
            mesh = ngs.MakeStructured2DMesh(nx=pr.nx, ny=pr.nx)
            fes = ngs.H1(mesh, order=pr.p, dirichlet=".*")
            a = _Elements(fes, _tensor(pr.kappa))
            out.append(a.solve(_tensor(pr.rhs)))
        return torch.cat(out)
    if kind == "adjoint":
        mesh, fes, kappa, u_obs = _adjoint_inputs(case, seed)
        a, m = _Elements(fes, _tensor(kappa)), _Elements(fes, None, mass=True)
        u = a.solve(_tensor(_load(fes)))
        r = u - _tensor(u_obs)
        mr = m.apply(r)
        lam = a.solve(mr)
        ue, le = (u * a.free)[a.dofs], (lam * a.free)[a.dofs]
        g = -torch.einsum("ei,eij,ej->e", le, a.mats, ue) / _tensor(kappa)[a.order]
        grad = torch.empty_like(g)
        grad[a.order] = g
        return {"u": u, "J": 0.5 * torch.dot(r, mr), "grad": grad}
    mesh, fes = _space(case)
    a = _Elements(fes, _tensor(_kappa(mesh, rng)))
    if kind == "assemble":
        rowptr, cols, vals = a.csr()
        return {"rowptr": rowptr, "cols": cols, "vals": vals}
    if kind in ("csr", "mf"):
        x = rng.uniform(-1.0, 1.0, fes.ndof)
        if case.get("vec") == 32:
            x = x.astype(np.float32).astype(np.float64)
        return a.apply(_tensor(x))
    k = case.get("nrhs", 1)
    f = _loads(fes, rng, k)
    cols = [a.solve(_tensor(f[:, j])) for j in range(k)]
    return cols[0] if k == 1 else torch.stack(cols, 1).reshape(-1)
