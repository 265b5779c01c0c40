"""The work this library is used for, as measurable cases.

Every case is one call (or the short sequence of calls that belongs together)
of the library's public interface, on a problem of the kind its users have:

  cg        conjugate gradients with the Jacobi preconditioner (FP64)
  rr        FP32 CG with FP64 residual replacement to an FP64 residual
  bicgstab  BiCGSTAB on upwind convection-diffusion
  gmres     restarted GMRES with right Jacobi on the same operator
  heat      one implicit time step's stage: I - gamma F rewritten, then CG
  batch     many small independent systems in one call
  mesh      CG with Jacobi on an unstructured mesh's matrix
  product   y = A x of a general matrix with rows of uneven length
  amg       CG preconditioned by an aggregation V-cycle with Gauss-Seidel
  adjoint   loss and gradients of a backward-Euler trajectory

Inputs are made on the GPU by torch from the seed; matrices enter the library
from host CSR arrays, vectors are torch tensors the library works on in place.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from flecsolve_amd import fsx

DEV = "cuda"
F64 = torch.float64
ELL = 8.0  # correlation length of the coefficient fields, in cells

_ctx = None


def _context() -> fsx.Context:
    """The one context a program keeps."""
    global _ctx
    if _ctx is None:
        _ctx = fsx.Context(0)
    return _ctx


# ---- the cases ---------------------------------------------------------------

def listed():
    return [
        # the mesh of flecsolve's heat example (100 x 100 vertices): a solve of
        # thousands of unknowns, bound by launches and reductions
        dict(name="cg_poisson_98x98", kind="cg", nx=98, ny=98, nz=1, sigma=0.0),
        # an ordinary 3-D diffusion solve
        dict(name="cg_diffusion_80x72x64", kind="cg", nx=80, ny=72, nz=64, sigma=1.0),
        # a large FP64 solve, no edge a multiple of the wavefront
        dict(name="cg_diffusion_161x160x159", kind="cg", nx=161, ny=160, nz=159, sigma=1.0),
        # the benchmark's problem: 256^3 lognormal diffusion, mixed precision
        dict(name="rr_diffusion_256", kind="rr", nx=256, ny=256, nz=256, sigma=1.0),
        # nonsymmetric solves of transport problems
        dict(name="bicgstab_convdiff_128x120x112", kind="bicgstab", nx=128, ny=120, nz=112),
        dict(name="gmres_convdiff_104x100x96", kind="gmres", nx=104, ny=100, nz=96),
        # a stage of the implicit heat example on a fine mesh: about a
        # hundred iterations from a near guess, after a change of the matrix
        dict(name="heat_stage_1022x1022", kind="heat", nx=1022, ny=1022, nz=1),
        # many small systems of uneven size
        dict(name="batch_rr_160", kind="batch", systems=160, emin=8, emax=40, method="rr"),
        # a finite-element-like mesh: symmetric, no regular structure
        dict(name="mesh_cg_400k", kind="mesh", rows=400_000, degree=14),
        # one product of a general matrix, rows of 3 to 60 entries
        dict(name="product_ragged_1m", kind="product", rows=1_000_003, degree=20, f32=False),
        # the reference's default multigrid (pairwise aggregation, Gauss-Seidel)
        dict(name="amg_cg_48x44x40", kind="amg", nx=48, ny=44, nz=40, sigma=1.0),
        # gradient of a heat trajectory with respect to every matrix entry
        dict(name="adjoint_rr_48x8", kind="adjoint", nx=48, ny=48, nz=48, steps=8, method="rr"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cg", "cg", "rr", "bicgstab", "gmres", "heat", "batch", "mesh",
                       "product", "amg", "adjoint"])

    def box(lo, hi):
        return dict(nx=_log_int(rng, lo, hi), ny=_log_int(rng, lo, hi), nz=_log_int(rng, lo, hi))

    if kind == "cg":
        if rng.random() < 0.4:
            return dict(kind=kind, nx=_log_int(rng, 40, 900), ny=_log_int(rng, 40, 900), nz=1,
                        sigma=0.0)
        return dict(kind=kind, sigma=rng.choice([1.0, 1.0, 2.0]), **box(20, 160))
    if kind == "rr":
        return dict(kind=kind, sigma=rng.choice([1.0, 1.0, 2.0]), **box(24, 180))
    if kind in ("bicgstab", "gmres"):
        return dict(kind=kind, **box(20, 128 if kind == "bicgstab" else 100))
    if kind == "heat":
        return dict(kind=kind, nx=_log_int(rng, 98, 2046), ny=_log_int(rng, 98, 2046), nz=1)
    if kind == "batch":
        return dict(kind=kind, systems=_log_int(rng, 8, 200), emin=rng.randint(5, 12),
                    emax=rng.randint(16, 44), method=rng.choice(["rr", "cg"]))
    if kind == "mesh":
        return dict(kind=kind, rows=_log_int(rng, 5_000, 400_000), degree=rng.randint(5, 24))
    if kind == "product":
        return dict(kind=kind, rows=_log_int(rng, 10_000, 1_000_000), degree=rng.randint(4, 40),
                    f32=rng.random() < 0.3)
    if kind == "amg":
        return dict(kind=kind, sigma=1.0, **box(16, 48))
    return dict(kind=kind, steps=rng.randint(3, 8), method=rng.choice(["rr", "cg"]),
                **box(16, 48))


# ---- problems (torch, from the seed alone) -----------------------------------

def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1_000_003 + stream) & 0x7FFFFFFFFFFF)
    return g


def _uniform(n, seed, stream, lo=-1.0, hi=1.0):
    return torch.rand(n, generator=_gen(seed, stream), device=DEV, dtype=F64) * (hi - lo) + lo


def _smooth_noise(shape, seed, stream):
    """Unit-variance Gaussian random field with correlation length ELL."""
    s = ELL / math.sqrt(2.0)
    R = int(math.ceil(3.0 * s))
    w = np.exp(-np.arange(-R, R + 1) ** 2 / (2.0 * s * s))
    w /= math.sqrt(float((w * w).sum()))
    axes = [a for a, m in enumerate(shape) if m > 1]
    big = [m + 2 * R if a in axes else m for a, m in enumerate(shape)]
    f = torch.randn(big, generator=_gen(seed, stream), device=DEV, dtype=F64)
    for a in axes:
        out = torch.zeros([shape[a] if b == a else m for b, m in enumerate(f.shape)],
                          device=DEV, dtype=F64)
        for t in range(2 * R + 1):
            out.add_(f.narrow(a, t, shape[a]), alpha=float(w[t]))
        f = out
    return f


class Grid:
    """A stencil matrix on an nx x ny x nz grid, x fastest: for each column
    offset (ascending) the coefficient per row and where it is present."""

    def __init__(self, case, offs, coef, mask):
        self.nx, self.ny, self.nz = case["nx"], case["ny"], case["nz"]
        self.n = self.nx * self.ny * self.nz
        self.offs = offs
        self.coef = [c.reshape(-1) for c in coef]
        self.mask = [m.reshape(-1) for m in mask]

    def csr(self):
        """Host arrays: row pointers, columns (int32), values."""
        m = torch.stack(self.mask, 1)
        v = torch.stack(self.coef, 1)[m].cpu().numpy()
        r = torch.arange(self.n, device=DEV, dtype=torch.int32)[:, None]
        c = (r + torch.tensor(self.offs, device=DEV, dtype=torch.int32))[m].cpu().numpy()
        rp = torch.zeros(self.n + 1, device=DEV, dtype=torch.int64)
        torch.cumsum(m.sum(1), 0, out=rp[1:])
        return rp.to(torch.int32).cpu().numpy(), c, v

    def operator(self):
        """x -> A x in plain torch."""
        coef = [torch.where(m, c, torch.zeros_like(c)) for c, m in zip(self.coef, self.mask)]
        pad = max(self.offs)

        def apply(x):
            xp = torch.nn.functional.pad(x, (pad, pad))
            y = torch.zeros_like(x)
            for o, c in zip(self.offs, coef):
                y.addcmul_(c, xp[pad + o:pad + o + self.n])
            return y
        return apply

    def diag(self):
        return self.coef[self.offs.index(0)]


def _edges(case):
    """Offsets of the cell's neighbours and where each lies on the grid."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    shape = (nz, ny, nx)
    idx = [torch.arange(m, device=DEV).reshape([m if a == b else 1 for b in range(3)])
           for a, m in enumerate(shape)]
    full = torch.ones(shape, device=DEV, dtype=torch.bool)
    lo = [full & (idx[a] > 0) for a in range(3)]
    hi = [full & (idx[a] < shape[a] - 1) for a in range(3)]
    axes = (0, 1, 2) if nz > 1 else (1, 2)
    step = (nx * ny, nx, 1)
    offs = [-step[a] for a in axes] + [0] + [step[a] for a in reversed(axes)]
    mask = [lo[a] for a in axes] + [full] + [hi[a] for a in reversed(axes)]
    return shape, axes, offs, mask


def _diffusion(case, seed, scale=1.0, shift=0.0):
    """shift I + scale (-div k grad), k lognormal with the case's sigma on the
    grid's nodes and the ring around them, arithmetic-mean faces, Dirichlet."""
    shape, axes, offs, mask = _edges(case)
    ring = [m + 2 if a in axes else m for a, m in enumerate(shape)]
    if case.get("sigma"):
        k = torch.exp(case["sigma"] * _smooth_noise(ring, seed, 1))
    else:
        k = torch.ones(ring, device=DEV, dtype=F64)

    def node(a, s):
        v = k
        for b in axes:
            v = v.narrow(b, 1 + (s if a == b else 0), shape[b])
        return v

    mid = node(None, 0)
    lo = [scale * (0.5 * (mid + node(a, -1))) for a in axes]
    hi = [scale * (0.5 * (mid + node(a, 1))) for a in axes]
    dia = shift + sum(lo) + sum(hi)
    coef = [-f for f in lo] + [dia] + [-f for f in reversed(hi)]
    return Grid(case, offs, coef, mask)


def _convdiff(case, seed):
    """Upwind convection-diffusion, cell velocities around (10, 5, 2.5)."""
    shape, axes, offs, mask = _edges(case)
    vel = [c * (0.5 + torch.rand(shape, generator=_gen(seed, 2 + a), device=DEV, dtype=F64))
           for a, c in enumerate((2.5, 5.0, 10.0))]
    one = torch.ones(shape, device=DEV, dtype=F64)
    coef = ([-one - vel[a] for a in axes] + [2.0 * len(axes) * one + sum(vel[a] for a in axes)]
            + [-one for a in axes])
    return Grid(case, offs, coef, mask)


class Coo:
    """A general matrix: sorted (row, column) pairs and their values."""

    def __init__(self, n, rows, cols, vals):
        self.n, self.rows, self.cols, self.vals = n, rows, cols, vals

    def csr(self):
        rp = torch.zeros(self.n + 1, device=DEV, dtype=torch.int64)
        torch.cumsum(torch.bincount(self.rows, minlength=self.n), 0, out=rp[1:])
        return (rp.to(torch.int32).cpu().numpy(), self.cols.to(torch.int32).cpu().numpy(),
                self.vals.cpu().numpy())

    def operator(self):
        def apply(x):
            return torch.zeros_like(x).index_add_(0, self.rows, self.vals * x[self.cols])
        return apply

    def diag(self):
        d = torch.zeros(self.n, device=DEV, dtype=F64)
        on = self.rows == self.cols
        d[self.rows[on]] = self.vals[on]
        return d


def _pairs(n, degree, seed, spread):
    """Distinct (row, column) keys off the diagonal, most of them near it: rows
    of uneven length, `degree` on average."""
    g = _gen(seed, 5)
    want = torch.rand(n, generator=g, device=DEV, dtype=F64)
    cnt = torch.clamp((degree * (0.25 + 1.5 * want * want * 1.5)).to(torch.int64), 1, 60)
    rows = torch.repeat_interleave(torch.arange(n, device=DEV), cnt)
    near = torch.randn(rows.numel(), generator=g, device=DEV, dtype=F64) * spread
    far = torch.rand(rows.numel(), generator=g, device=DEV, dtype=F64) < 0.02
    anywhere = torch.randint(0, n, (rows.numel(),), generator=g, device=DEV)
    cols = torch.where(far, anywhere, rows + torch.round(near).to(torch.int64))
    ok = (cols >= 0) & (cols < n) & (cols != rows)
    return torch.unique(rows[ok] * n + cols[ok])


def _mesh(case, seed):
    """Graph Laplacian of a random mesh plus a positive diagonal: symmetric."""
    n = case["rows"]
    half = _pairs(n, max(2.0, case["degree"] / 2.0), seed, 40.0 + 0.02 * math.sqrt(n))
    i, j = half // n, half % n
    lo, hi = torch.minimum(i, j), torch.maximum(i, j)
    e = torch.unique(lo * n + hi)
    i, j = e // n, e % n
    # multiples of 2^-20: the row sums on the diagonal are exact in any order
    w = -torch.round(_uniform(e.numel(), seed, 6, 0.1, 1.0) * 2.0 ** 20) / 2.0 ** 20
    d = torch.full((n,), 0.02, device=DEV, dtype=F64)
    d.index_add_(0, i, -w)
    d.index_add_(0, j, -w)
    dia = torch.arange(n, device=DEV)
    rows, cols = torch.cat([i, j, dia]), torch.cat([j, i, dia])
    vals = torch.cat([w, w, d])
    order = torch.argsort(rows * n + cols)
    return Coo(n, rows[order], cols[order], vals[order])


def _ragged(case, seed):
    n = case["rows"]
    e = _pairs(n, case["degree"], seed, 300.0)
    vals = _uniform(e.numel(), seed, 6)
    if case["f32"]:
        vals = vals.float()
    return Coo(n, e // n, e % n, vals)


def _batch(case, seed):
    """Block-diagonal diffusion systems: (matrix, first row of each system).
    Edges come from the case, not the seed: another seed has other values."""
    rs = np.random.RandomState(case["systems"] * 131 + case["emin"] * 17 + case["emax"])
    edges = rs.randint(case["emin"], case["emax"] + 1, case["systems"])
    k = torch.exp(_smooth_noise((66, 66, 66), seed, 7))
    first, rows, cols, vals = [0], [], [], []
    for s, e in enumerate(edges):
        e = int(e)
        at = [int(v) for v in rs.randint(0, 66 - e - 2 + 1, 3)]
        sub = k[at[0]:at[0] + e + 2, at[1]:at[1] + e + 2, at[2]:at[2] + e + 2]
        shape, axes, offs, mask = _edges(dict(nx=e, ny=e, nz=e))
        node = lambda a, o: sub[tuple(slice(1 + (o if a == b else 0), 1 + (o if a == b else 0) + e)  # noqa: E731
                                      for b in range(3))]
        mid = node(None, 0)
        lo = [0.5 * (mid + node(a, -1)) for a in axes]
        hi = [0.5 * (mid + node(a, 1)) for a in axes]
        coef = [-f for f in lo] + [sum(lo) + sum(hi)] + [-f for f in reversed(hi)]
        m = torch.stack([q.reshape(-1) for q in mask], 1)
        r = torch.arange(e ** 3, device=DEV)[:, None] + first[-1]
        vals.append(torch.stack([q.reshape(-1) for q in coef], 1)[m])
        cols.append((r + torch.tensor(offs, device=DEV))[m])
        rows.append(r.expand(-1, len(offs))[m])
        first.append(first[-1] + e ** 3)
    return (Coo(first[-1], torch.cat(rows), torch.cat(cols), torch.cat(vals)),
            np.array(first, np.int64))


HEAT_GAMMA = 30.0  # gamma alpha / h^2 of a late step of the heat example


def _heat(case, seed):
    """F = alpha Laplacian / h^2 (5-point) and the state u it acts on."""
    shape, axes, offs, mask = _edges(case)
    one = torch.ones(shape, device=DEV, dtype=F64)
    F = Grid(case, offs, [one] * len(axes) + [-2.0 * len(axes) * one] + [one] * len(axes), mask)
    u = 25.0 * torch.exp(0.5 * _smooth_noise(shape, seed, 8)).reshape(-1)
    rhs = u * (1.0 + 0.01 * _smooth_noise(shape, seed, 9).reshape(-1))
    return F, u.contiguous(), rhs


def _problem(case, seed):
    kind = case["kind"]
    if kind in ("cg", "rr", "amg"):
        return _diffusion(case, seed)
    if kind in ("bicgstab", "gmres"):
        return _convdiff(case, seed)
    if kind == "mesh":
        return _mesh(case, seed)
    if kind == "product":
        return _ragged(case, seed)
    return _diffusion(dict(case, sigma=1.0), seed, scale=1e-3 * (case["nx"] + 1) ** 2, shift=1.0)


def _trajectory(case, seed, n):
    """Start and target of the backward-Euler trajectory."""
    shape = (case["nz"], case["ny"], case["nx"])
    u0 = torch.exp(_smooth_noise(shape, seed, 10)).reshape(-1).contiguous()
    return u0, u0 * _uniform(n, seed, 11, 0.2, 0.6)


# ---- prepare and run ---------------------------------------------------------

def _wrap(t: torch.Tensor) -> fsx.Vector:
    """The library's vector over a torch tensor's memory."""
    ctx = _context()
    h = C.c_void_p()
    dt = fsx.F64 if t.dtype == F64 else fsx.F32
    fsx.check(fsx.lib().fsx_vec_wrap(ctx.h, t.data_ptr(), t.numel(), dt, C.byref(h)))
    v = fsx.Vector(ctx, t.numel(), dt, _handle=h)
    v.tensor = t
    return v


def _vec(n, dtype=F64):
    return _wrap(torch.zeros(n, device=DEV, dtype=dtype))


def prepare(case, seed):
    ctx = _context()
    kind = case["kind"]
    st = dict(case)
    if kind == "heat":
        F, u, rhs = _heat(case, seed)
        st["F"] = ctx.csr(*F.csr())
        st["A"] = st["F"].convert(fsx.F64)
        st["u"], st["b"], st["x"] = _wrap(u), _wrap(rhs), _vec(F.n)
        st["settings"] = fsx.Settings(maxiter=10000, rtol=1e-6)
    elif kind == "batch":
        M, first = _batch(case, seed)
        A = st["A"] = ctx.csr(*M.csr())
        st["batch"] = fsx.Batch(A, first)
        st["b"], st["x"] = _wrap(_uniform(M.n, seed, 3)), _vec(M.n)
        st["dinv"] = A.diag_inv()
        if case["method"] == "rr":
            st["A32"] = A.convert(fsx.F32)
            st["A32"].set_values_sym_scaled(A)
            st["settings"] = fsx.Settings(maxiter=5000, rtol=3e-2)
        else:
            st["settings"] = fsx.Settings(maxiter=5000, rtol=1e-10, use_zero_guess=True)
    else:
        M = _problem(case, seed)
        A = st["A"] = ctx.csr(*M.csr())
        if kind == "product":
            x = _uniform(M.n, seed, 3)
            st["x"] = _wrap(x.float() if case["f32"] else x)
            st["y"] = _vec(M.n, st["x"].tensor.dtype)
        elif kind == "adjoint":
            u0, target = _trajectory(case, seed, M.n)
            st["u0"], st["target"] = _wrap(u0), _wrap(target)
            st["G"], st["uT"], st["g0"] = _vec(A.nnz), _vec(M.n), _vec(M.n)
            st["settings"] = fsx.Settings(maxiter=5000, rtol=1e-12)
            st["dinv"] = A.diag_inv()
            if case["method"] == "rr":
                st["A32"] = A.convert(fsx.F32)
                st["A32"].set_values_sym_scaled(A)
                st["inner"] = fsx.Settings(maxiter=5000, rtol=3e-2)
        else:
            st["b"], st["x"] = _wrap(_uniform(M.n, seed, 3)), _vec(M.n)
            st["settings"] = fsx.Settings(maxiter=20000, rtol=1e-10, use_zero_guess=True)
            if kind == "rr":
                st["A32"] = A.convert(fsx.F32)
                st["A32"].set_values_sym_scaled(A)
                st["settings"] = fsx.Settings(maxiter=20000, rtol=3e-2)
            elif kind == "gmres":
                st["settings"] = fsx.Settings(maxiter=5000, rtol=1e-10, use_zero_guess=True,
                                              max_krylov_dim=30, restart=True, pre_side=1)
            elif kind == "amg":
                st["amg"] = fsx.AMG(A, fsx.AmgSettings(maxiter=1, atol=0.0))
            if kind in ("cg", "mesh", "gmres"):
                st["dinv"] = A.diag_inv()
    torch.cuda.synchronize()
    return st


def run(st):
    kind = st["kind"]
    ctx = _context()
    lib = fsx.lib()
    if kind in ("cg", "mesh"):
        fsx.cg_solve(st["A"], st["b"], st["x"], st["settings"], dinv=st["dinv"])
    elif kind == "rr":
        fsx.check(lib.fsx_zero(ctx.h, st["x"].h))
        fsx.ir_cg_rr_solve(st["A"], st["A32"], st["b"], st["x"], 1e-10, st["settings"])
    elif kind == "bicgstab":
        fsx.bicgstab_solve(st["A"], st["b"], st["x"], st["settings"])
    elif kind == "gmres":
        fsx.gmres_solve(st["A"], st["b"], st["x"], st["settings"], dinv=st["dinv"])
    elif kind == "heat":
        st["A"].shift_scale(st["F"], 1.0, -HEAT_GAMMA)
        fsx.check(lib.fsx_copy(ctx.h, st["u"].h, st["x"].h))
        fsx.cg_solve(st["A"], st["b"], st["x"], st["settings"])
    elif kind == "batch":
        if st["method"] == "rr":
            fsx.check(lib.fsx_zero(ctx.h, st["x"].h))
            st["batch"].rr_cg(st["A32"], st["b"], st["x"], 1e-10, st["settings"])
        else:
            st["batch"].cg(st["b"], st["x"], st["settings"], dinv=st["dinv"])
    elif kind == "product":
        st["A"].spmv(st["x"], st["y"])
        return st["y"].tensor
    elif kind == "amg":
        st["amg"].cg(st["b"], st["x"], st["settings"])
    else:
        loss, stats = C.c_double(), fsx.BEStats()
        ckpt = max(1, st["steps"] // 2)
        if st["method"] == "rr":
            rc = lib.fsx_be_adjoint_rr(ctx.h, st["A"].h, st["A32"].h, st["u0"].h,
                                       st["target"].h, st["steps"], ckpt,
                                       C.byref(st["settings"]), C.byref(st["inner"]),
                                       C.byref(loss), st["G"].h, st["uT"].h, st["g0"].h,
                                       C.byref(stats))
        else:
            rc = lib.fsx_be_adjoint(ctx.h, st["A"].h, None, st["dinv"].h, st["u0"].h,
                                    st["target"].h, st["steps"], ckpt, C.byref(st["settings"]),
                                    C.byref(loss), st["G"].h, st["uT"].h, st["g0"].h,
                                    C.byref(stats))
        fsx.check(rc)
        return dict(loss=loss.value, G=st["G"].tensor, uT=st["uT"].tensor, g0=st["g0"].tensor)
    return st["x"].tensor


# ---- what a pass cannot do without, and how far it may be off ------------------

def _rows(case):
    if "nx" in case:
        return case["nx"] * case["ny"] * case["nz"]
    if "rows" in case:
        return case["rows"]
    return case["systems"] * ((case["emin"] + case["emax"]) / 2.0) ** 3 * 1.2


def work(case):
    """Bytes and operations of one pass.  A solve's iterations are part of the
    method: each reads the matrix's values (half of a symmetric matrix's
    off-diagonal ones) and reads or writes each of the iteration's vectors as
    often as its data dependences force.  The iteration counts are the
    method's on problems like these, fitted to the grid's longest edge."""
    kind, n = case["kind"], float(_rows(case))
    edge = max(case.get(k, 1) for k in ("nx", "ny", "nz"))
    width = 4 if case.get("nz", 1) > 1 or kind == "batch" else 3   # stored half stencil
    sym64 = 8.0 * width
    ops = 2.0 * (2 * width - 1)
    if kind == "cg":
        its = (3.5 if case["nz"] == 1 else 5.8 * (1.0 + 0.6 * max(0.0, case["sigma"] - 1.0))) * edge
        return dict(bytes=its * n * (sym64 + 72), flops=its * n * (ops + 12))
    if kind == "rr":
        its = 5.8 * (1.0 + 0.6 * max(0.0, case["sigma"] - 1.0)) * edge
        return dict(bytes=its * n * (sym64 / 2 + 36), flops=its * n * (ops + 10))
    if kind == "bicgstab":
        its = 1.8 * edge
        return dict(bytes=its * n * (2 * 56 + 112), flops=its * n * (2 * 14 + 24))
    if kind == "gmres":
        its = 3.6 * edge
        return dict(bytes=its * n * (56 + 24 + 16 * 16), flops=its * n * (14 + 64))
    if kind == "heat":
        its = 110.0
        return dict(bytes=n * (2 * sym64 + its * (sym64 + 64)), flops=its * n * (ops + 10))
    if kind == "batch":
        its = 3.5 * (case["emin"] + case["emax"])
        return dict(bytes=its * n * (sym64 / 2 + 36), flops=its * n * (ops + 10))
    if kind == "mesh":
        its, nnz = 119.0, n * (case["degree"] + 1.0)
        return dict(bytes=its * (nnz * 12 + n * 76), flops=its * (2 * nnz + 12 * n))
    if kind == "product":
        nnz, b = n * case["degree"], 4.0 if case["f32"] else 8.0
        return dict(bytes=nnz * (b + 4) + n * (2 * b + 4), flops=2 * nnz)
    if kind == "amg":
        its = 0.55 * edge
        # four symmetric sweeps of two, residuals and transfers over levels
        # that add up to about half the fine one
        return dict(bytes=its * n * (1.5 * 10 * (12 * 7 + 24)), flops=its * n * 1.5 * 10 * 14)
    its = 2.5 * case["steps"] * 1.5 * edge
    return dict(bytes=its * n * (sym64 / 2 + 36), flops=its * n * (ops + 10))


def tolerance(case):
    kind = case["kind"]
    if kind == "product":
        return {"rel": 1e-6 if case["f32"] else 1e-14}
    if kind == "heat":
        return {"rel": 4e-6}          # two stopped at a residual of 1e-6
    if kind == "adjoint":
        return {"rel": 2e-11}         # solves to 1e-12
    return {"rel": 2e-8}              # two stopped at a residual of 1e-10


def _bicgstab_torch(op, b, dinv, rtol, maxiter):
    x = torch.zeros_like(b)
    r = b.clone()
    r0, p, v = r.clone(), torch.zeros_like(b), torch.zeros_like(b)
    rho = alpha = om = torch.ones((), device=DEV, dtype=F64)
    stop = rtol * float(b.norm())
    for it in range(maxiter):
        rho1 = torch.dot(r0, r)
        beta = (rho1 / rho) * (alpha / om)
        rho = rho1
        p = r + beta * (p - om * v)
        ph = dinv * p
        v = op(ph)
        alpha = rho / torch.dot(r0, v)
        s = r - alpha * v
        sh = dinv * s
        t = op(sh)
        om = torch.dot(t, s) / torch.dot(t, t)
        x = x + alpha * ph + om * sh
        r = s - om * t
        if it % 10 == 9 and float(r.norm()) <= stop:
            break
    return x


def _cg_torch(op, b, dinv, rtol, maxiter):
    x = torch.zeros_like(b)
    r = b.clone()
    z = dinv * r
    p = z.clone()
    rho = torch.dot(r, z)
    stop = rtol * float(b.norm())
    for it in range(maxiter):
        w = op(p)
        alpha = rho / torch.dot(p, w)
        x.addcmul_(alpha, p)
        r.addcmul_(-alpha, w)
        if it % 20 == 19 and float(r.norm()) <= stop:
            break
        z = dinv * r
        rho1 = torch.dot(r, z)
        p = z + (rho1 / rho) * p
        rho = rho1
    return x


def _tight(op, b, dinv, solve, guess=None):
    """A x = b to rounding: three solves, each on the last one's residual."""
    x = torch.zeros_like(b) if guess is None else guess.clone()
    for _ in range(3):
        r = b - op(x)
        if float(r.norm()) <= 1e-15 * float(b.norm()):
            break
        x = x + solve(op, r, dinv, 1e-7, 30000)
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind == "product":
        M = _ragged(case, seed)
        x = _uniform(M.n, seed, 3)
        if case["f32"]:
            x = x.float().double()
            M.vals = M.vals.double()
        return M.operator()(x)
    if kind == "heat":
        F, u, rhs = _heat(case, seed)
        lap = F.operator()
        d = torch.full((F.n,), 1.0 / (1.0 + 4.0 * HEAT_GAMMA), device=DEV, dtype=F64)
        return _tight(lambda x: x - HEAT_GAMMA * lap(x), rhs, d, _cg_torch, guess=u)
    if kind == "batch":
        M, _ = _batch(case, seed)
        return _tight(M.operator(), _uniform(M.n, seed, 3), 1.0 / M.diag(), _cg_torch)
    M = _problem(case, seed)
    op, dinv = M.operator(), 1.0 / M.diag()
    if kind != "adjoint":
        solve = _bicgstab_torch if kind in ("bicgstab", "gmres") else _cg_torch
        return _tight(op, _uniform(M.n, seed, 3), dinv, solve)
    u0, target = _trajectory(case, seed, M.n)
    us = [u0]
    for _ in range(case["steps"]):
        us.append(_tight(op, us[-1], dinv, _cg_torch, guess=us[-1]))
    diff = us[-1] - target
    lam = 2.0 * diff
    at = torch.stack(M.mask, 1)
    rows = torch.arange(M.n, device=DEV)[:, None].expand(-1, len(M.offs))[at]
    cols = rows + torch.tensor(M.offs, device=DEV).expand(M.n, -1)[at]
    G = torch.zeros(rows.numel(), device=DEV, dtype=F64)
    for s in range(case["steps"], 0, -1):
        lam = _tight(op, lam, dinv, _cg_torch, guess=lam)
        G -= lam[rows] * us[s][cols]
    return dict(loss=float(torch.dot(diff, diff)), G=G, uT=us[-1], g0=lam)
