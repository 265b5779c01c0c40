"""Fused, graph-captured CG (fsx_cg_solve) and FP32-inner / FP64-outer
refinement against the oracle (gpu).

Bar (from the hot-path contract): iteration counts within +-2 of the
oracle's, solutions within 1e-10 relative of the oracle's.  The reductions
sum in a different (tree) order than the reference's serial loop, so the two
trajectories drift apart at the level of rounding; the solution comparison
uses a tolerance a factor below the solve tolerance where the problem's
conditioning allows, and otherwise compares against the exact solution.
"""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

from flecsolve_amd import fsx
from flecsolve_amd import problems as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def poisson(n):
    rp, ci, v = P.poisson2d(n)
    return rp, ci, v, O.Csr(rp, ci, v)


def diffusion(n, sigma=1.0, seed=2001):
    k = P.lognormal_field(n, sigma, 8.0, seed)
    rp, ci, v = P.diffusion3d(n, k)
    return rp, ci, v, O.Csr(rp, ci, v)


def test_cg_poisson64_cfg1(ctx):
    """2D Poisson 64x64, unpreconditioned CG to rtol 1e-8, x0 = 0."""
    rp, ci, v, Ao = poisson(64)
    b = P.uniform(64 * 64, P.seeds()["poisson2d_rhs"])
    s = dict(maxiter=1000, rtol=1e-8, use_zero_guess=True)
    xo, io, ho = O.cg(Ao, b, np.zeros_like(b), O.Settings(**s), hist_cap=1000)
    A = ctx.csr(rp, ci, v)
    bd, xd = ctx.vec(b), ctx.zeros(b.size)
    info = fsx.cg_solve(A, bd, xd, fsx.Settings(**s))
    assert info.reason == io.reason == "converged_rtol"
    assert abs(info.iters - io.iters) <= 2
    assert rel(xd.get(), xo) <= 1e-10
    h = fsx.cg_history(ctx)
    m = min(len(h), io.iters)
    np.testing.assert_allclose(h[:m], ho[:m], rtol=1e-6)
    assert info.rhs_norm == io.rhs_norm


@pytest.mark.parametrize("n", [16, 48])
def test_cg_jacobi_diffusion(ctx, n):
    rp, ci, v, Ao = diffusion(n)
    b = P.uniform(n ** 3, 2002)
    s = dict(maxiter=3000, rtol=1e-10, use_zero_guess=True)
    xo, io, _ = O.cg(Ao, b, np.zeros_like(b), O.Settings(**s), P=O.prec(1, Ao.dinv()))
    A = ctx.csr(rp, ci, v)
    d = A.diag_inv()
    xd = ctx.zeros(b.size)
    info = fsx.cg_solve(A, ctx.vec(b), xd, fsx.Settings(**s), dinv=d)
    assert info.reason == "converged_rtol"
    assert abs(info.iters - io.iters) <= 2
    assert rel(xd.get(), xo) <= 1e-10
    S = sp.csr_matrix((v, ci, rp))
    assert np.linalg.norm(b - S @ xd.get()) / np.linalg.norm(b) < 2e-10


def test_cg_nonzero_guess_and_repeat(ctx):
    rp, ci, v, Ao = diffusion(20)
    n = 20 ** 3
    b = P.uniform(n, 1)
    x0 = O.set_random(n, 7)
    s = dict(maxiter=500, rtol=1e-9)
    xo, io, _ = O.cg(Ao, b, x0, O.Settings(**s))
    A = ctx.csr(rp, ci, v)
    for _ in range(2):  # second call replays the cached graph
        xd = ctx.vec(x0)
        info = fsx.cg_solve(A, ctx.vec(b), xd, fsx.Settings(**s))
        assert abs(info.iters - io.iters) <= 2
        assert rel(xd.get(), xo) <= 1e-9
        assert info.sol_norm_initial == io.sol_norm_initial


def test_cg_quirks(ctx):
    rp, ci, v, Ao = poisson(8)
    A = ctx.csr(rp, ci, v)
    b = P.uniform(64, 1)
    # maxiter hit: iters == 0, diverged_iters (cg.hh:135-136)
    info = fsx.cg_solve(A, ctx.vec(b), ctx.zeros(64),
                        fsx.Settings(maxiter=3, rtol=1e-12, use_zero_guess=True))
    assert info.iters == 0 and info.reason == "diverged_iters"
    xo, io, _ = O.cg(Ao, b, np.zeros(64), O.Settings(maxiter=3, rtol=1e-12,
                                                    use_zero_guess=True))
    assert info.res_norm_final == pytest.approx(io.res_norm_final, rel=1e-6)
    # zero rhs: converged before the loop, b_norm := 1
    info = fsx.cg_solve(A, ctx.zeros(64), ctx.zeros(64),
                        fsx.Settings(maxiter=3, rtol=1e-12, use_zero_guess=True))
    assert info.iters == 0 and info.reason == "converged_rtol" and info.rhs_norm == 1.0
    # maxiter == 0
    info = fsx.cg_solve(A, ctx.vec(b), ctx.zeros(64),
                        fsx.Settings(maxiter=0, rtol=1e-12, use_zero_guess=True))
    assert info.reason == "diverged_iters"


def test_cg_chunk_boundaries(ctx):
    # convergence exactly at, before and after a captured chunk boundary
    d = np.repeat(np.arange(1.0, 18.0), 3)  # 17 distinct eigenvalues
    n = d.size
    rp = np.arange(n + 1, dtype=np.int32)
    A = ctx.csr(rp, np.arange(n, dtype=np.int32), d)
    Ao = O.Csr(rp, np.arange(n, dtype=np.int32), d)
    b = O.set_random(n, 3)
    for maxiter in (15, 16, 17, 40):
        s = dict(maxiter=maxiter, rtol=1e-12, use_zero_guess=True)
        xo, io, _ = O.cg(Ao, b, np.zeros(n), O.Settings(**s))
        xd = ctx.zeros(n)
        info = fsx.cg_solve(A, ctx.vec(b), xd, fsx.Settings(**s))
        assert (info.iters, info.reason) == (io.iters, io.reason), maxiter
        np.testing.assert_allclose(xd.get(), xo, rtol=1e-10, atol=1e-14)


def test_fp32_cg(ctx):
    rp, ci, v, Ao = diffusion(24)
    n = 24 ** 3
    b = P.uniform(n, 5).astype(np.float32)
    A32 = ctx.csr(rp, ci, v).convert(fsx.F32)
    d = ctx.csr(rp, ci, v).diag_inv(fsx.F32)
    xd = ctx.zeros(n, fsx.F32)
    info = fsx.cg_solve(A32, ctx.vec(b), xd, fsx.Settings(maxiter=500, rtol=1e-4,
                                                         use_zero_guess=True), dinv=d)
    assert info.reason == "converged_rtol"
    S = sp.csr_matrix((v, ci, rp))
    x = xd.get().astype(np.float64)
    assert np.linalg.norm(b - S @ x) / np.linalg.norm(b) < 2e-4


@pytest.mark.parametrize("jacobi", [1, 2])
@pytest.mark.parametrize("sigma", [1.0, 2.5])
def test_ir_reaches_1e10_and_matches_fp64(ctx, sigma, jacobi):
    n = 32
    rp, ci, v, Ao = diffusion(n, sigma, seed=3001)
    N = n ** 3
    b = P.uniform(N, 3002)
    A64 = ctx.csr(rp, ci, v)
    A32 = A64.convert(fsx.F32)
    if jacobi == 2:
        A32.set_values_sym_scaled(A64)
    xd = ctx.zeros(N)
    info = fsx.ir_cg_solve(A64, A32, ctx.vec(b), xd, 1e-10,
                           fsx.Settings(maxiter=2000, rtol=1e-4), jacobi=jacobi)
    assert info.status == 1 and info.rel_res_final <= 1e-10
    S = sp.csr_matrix((v, ci, rp))
    x = xd.get()
    assert np.linalg.norm(b - S @ x) / np.linalg.norm(b) <= 1.01e-10
    xo, io, _ = O.cg(Ao, b, np.zeros(N), O.Settings(maxiter=5000, rtol=1e-12,
                                                   use_zero_guess=True),
                     P=O.prec(1, Ao.dinv()))
    # both are 1e-10-residual solutions: error bounded by cond * 1e-10
    assert rel(x, xo) < 1e-6


@pytest.mark.parametrize("plan", [4, 3, 2])
def test_grid_stride_sizes_iteration_matched(ctx, plan):
    """More rows than one capped SpMV grid covers (> 8192 x 256), so each
    thread owns several rows: SpMV+dot and 25 CG iterations against the
    oracle, iteration-matched (both stop at maxiter), on the symmetric
    stencil, slice-offset and sliced layouts."""
    n = 132
    rp, ci, v, Ao = diffusion(n)
    N = n ** 3
    assert N > 8192 * 256
    b = P.uniform(N, 2002)
    A = ctx.csr(rp, ci, v)
    assert A.plan() == (4, 0)
    A.set_plan(plan)
    bd = ctx.vec(b)
    w = ctx.zeros(N)
    pw = fsx.spmv_dot(A, bd, w)
    wref = Ao.spmv(b)
    np.testing.assert_array_equal(w.get(), wref)
    assert abs(pw - O.dot(wref, b)) <= 1e-12 * np.abs(wref * b).sum()
    s = dict(maxiter=25, rtol=1e-12, use_zero_guess=True)
    xo, io, ho = O.cg(Ao, b, np.zeros(N), O.Settings(**s), P=O.prec(1, Ao.dinv()),
                      hist_cap=25)
    xd = ctx.zeros(N)
    info = fsx.cg_solve(A, bd, xd, fsx.Settings(**s), dinv=A.diag_inv())
    assert info.reason == io.reason == "diverged_iters"
    np.testing.assert_allclose(fsx.cg_history(ctx), ho, rtol=1e-10)
    assert rel(xd.get(), xo) <= 1e-12


def test_wide_block_shape_iteration_matched(ctx):
    """From 2^23 rows the FP64 reducing product runs in 512-thread blocks
    (another block partial tree than below that size): 204^3 = 8,489,664
    rows, the SpMV+dot bit-compared and 25 CG + Jacobi iterations against
    the oracle, iteration-matched (both stop at maxiter)."""
    n = 204
    rp, ci, v, Ao = diffusion(n)
    N = n ** 3
    assert N >= 1 << 23
    b = P.uniform(N, 2002)
    A = ctx.csr(rp, ci, v)
    assert A.plan() == (4, 0)
    bd = ctx.vec(b)
    w = ctx.zeros(N)
    pw = fsx.spmv_dot(A, bd, w)
    wref = Ao.spmv(b)
    np.testing.assert_array_equal(w.get(), wref)
    assert abs(pw - O.dot(wref, b)) <= 1e-12 * np.abs(wref * b).sum()
    s = dict(maxiter=25, rtol=1e-12, use_zero_guess=True)
    xo, io, ho = O.cg(Ao, b, np.zeros(N), O.Settings(**s), P=O.prec(1, Ao.dinv()),
                      hist_cap=25)
    xd = ctx.zeros(N)
    info = fsx.cg_solve(A, bd, xd, fsx.Settings(**s), dinv=A.diag_inv())
    assert info.reason == io.reason == "diverged_iters"
    np.testing.assert_allclose(fsx.cg_history(ctx), ho, rtol=1e-10)
    assert rel(xd.get(), xo) <= 1e-12


def test_layouts_give_identical_trajectories(ctx):
    """Every serial-row layout gives the same SpMV bits; the fused dot
    products are reduced over each layout's own block grid, so iterates
    agree to rounding and the iteration counts match."""
    n = 40
    rp, ci, v, Ao = diffusion(n)
    b = P.uniform(n ** 3, 77)
    A = ctx.csr(rp, ci, v)
    d = A.diag_inv()
    bd = ctx.vec(b)
    out = []
    for plan in (4, 3, 2, 0):
        A.set_plan(plan)
        x = ctx.zeros(n ** 3)
        info = fsx.cg_solve(A, bd, x, fsx.Settings(maxiter=2000, rtol=1e-10,
                                                   use_zero_guess=True), dinv=d)
        out.append((info.iters, x.get()))
    for it, x in out[1:]:
        assert abs(it - out[0][0]) <= 1
        assert rel(x, out[0][1]) <= 1e-12


def test_graphs_after_matrix_rebuild(ctx):
    """Captured solver graphs hold the device arrays of the matrix they were
    captured for.  Matrices of one shape are built, solved and freed in turn
    on one context (their buffers may come back at the old addresses), and
    every solve must match its own residual -- no graph replays against the
    arrays of a freed matrix."""
    import gc
    n = 24
    N = n ** 3
    for rep, sigma in enumerate((1.0, 2.0, 1.5)):
        rp, ci, v, Ao = diffusion(n, sigma, seed=4000 + rep)
        b = P.uniform(N, 4100 + rep)
        A = ctx.csr(rp, ci, v)
        A32 = A.convert(fsx.F32)
        S = sp.csr_matrix((v, ci, rp))
        x = ctx.zeros(N)
        info = fsx.ir_cg_solve(A, A32, ctx.vec(b), x, 1e-10,
                               fsx.Settings(maxiter=2000, rtol=1e-4))
        assert info.status == 1
        assert np.linalg.norm(b - S @ x.get()) / np.linalg.norm(b) <= 1.01e-10
        x2 = ctx.zeros(N)
        i2 = fsx.cg_solve(A, ctx.vec(b), x2, fsx.Settings(maxiter=3000, rtol=1e-9,
                                                          use_zero_guess=True),
                          dinv=A.diag_inv())
        assert i2.reason == "converged_rtol"
        assert np.linalg.norm(b - S @ x2.get()) / np.linalg.norm(b) <= 1e-9
        del A, A32, x, x2
        gc.collect()


@pytest.mark.parametrize("plan", [4, 3, 2, 0])
def test_sym_scaled_f32_values(ctx, plan):
    """S A S in FP32, S = 1/sqrt(diag): values bit for bit against numpy
    (a_ij (s_i s_j) rounded once, so symmetric A gives bitwise symmetric
    values and keeps the symmetric stencil layout), on each SpMV layout;
    errors for a missing or non-positive diagonal."""
    n = 20
    rp, ci, v, _ = diffusion(n, 2.0, seed=5001)
    A64 = ctx.csr(rp, ci, v)
    A64.set_plan(plan)
    A32 = A64.convert(fsx.F32)
    A32.set_plan(plan)
    A32.set_values_sym_scaled(A64)
    assert A32.plan() == (plan, 0)
    rows = np.repeat(np.arange(n ** 3), np.diff(rp))
    d = v[ci == rows]
    sv = 1.0 / np.sqrt(d)
    want = (v * (sv[rows] * sv[ci])).astype(np.float32)
    np.testing.assert_array_equal(A32.download()[2], want)
    W = sp.csr_matrix((want, ci, rp))
    assert (W != W.T).nnz == 0
    x = P.uniform(n ** 3, 5002).astype(np.float32)
    y = ctx.zeros(n ** 3, fsx.F32)
    A32.spmv(ctx.vec(x, fsx.F32), y)
    ref = sp.csr_matrix((want.astype(np.float64), ci, rp)) @ x.astype(np.float64)
    assert np.abs(y.get() - ref).max() <= 1e-5 * np.abs(ref).max()
    bad = ctx.csr(np.array([0, 1, 2], np.int32), np.array([1, 0], np.int32),
                  np.array([1.0, 1.0]))
    with pytest.raises(fsx.FsxError):
        bad.convert(fsx.F32).set_values_sym_scaled(bad)
    neg = ctx.csr(np.array([0, 1, 2], np.int32), np.array([0, 1], np.int32),
                  np.array([1.0, -1.0]))
    with pytest.raises(fsx.FsxError):
        neg.convert(fsx.F32).set_values_sym_scaled(neg)


def test_new_entry_points_reject_bad_arguments(ctx):
    """Errors, not faults: a refinement (jacobi = 2) or refined adjoint whose
    FP32 matrix is not a copy of A's pattern, an unknown mode, a stage matrix
    that is F itself or does not share F's pattern."""
    rp, ci, v = P.poisson2d(12)
    A = ctx.csr(rp, ci, v)
    other = ctx.csr(rp, ci, v)          # same values, its own index arrays
    A32_other = other.convert(fsx.F32)
    b, x = ctx.vec(P.uniform(144, 1)), ctx.zeros(144)
    inner = fsx.Settings(maxiter=100, rtol=1e-4)
    with pytest.raises(fsx.FsxError):
        fsx.ir_cg_solve(A, A32_other, b, x, 1e-10, inner, jacobi=2)
    with pytest.raises(fsx.FsxError):
        fsx.ir_cg_solve(A, A.convert(fsx.F32), b, x, 1e-10, inner, jacobi=3)
    with pytest.raises(fsx.FsxError):
        fsx.be_forward_ir(A, A32_other, b, 2, fsx.Settings(maxiter=100, rtol=1e-10), inner)
    with pytest.raises(fsx.FsxError):
        A.shift_scale(A, 1.0, -0.5)
    with pytest.raises(fsx.FsxError):
        other.convert(fsx.F64).shift_scale(A, 1.0, -0.5)
    # the good path still works afterwards
    A32 = A.convert(fsx.F32)
    A32.set_values_sym_scaled(A)
    info = fsx.ir_cg_solve(A, A32, b, x, 1e-10, inner, jacobi=2)
    assert info.status == 1


def test_cg_user_diagnostic(ctx):
    """The fused CG with the reference's user diagnostic (cg.hh:112-116):
    called after every iteration with the updated x and |r|, before the
    tolerance test.  A diagnostic that never stops gives fsx_cg_solve's
    iterates bit for bit, its |r| values are the residual history; one that
    stops at iteration 9 ends the solve there with converged_user and the
    oracle's x (its diagnostic stopping at the same call); the reference
    test's A-norm diagnostic (solvers/test/cg.cc:16-54: monotone decrease
    and the Trefethen-Bau bound for b = 0, x0 = set_random) holds; an
    exception in the diagnostic aborts the solve."""
    n = 40
    rp, ci, v = P.poisson2d(n)
    Ao = O.Csr(rp, ci, v)
    A = ctx.csr(rp, ci, v)
    d = A.diag_inv()
    b = P.uniform(n * n, 31)
    s = dict(maxiter=2000, rtol=1e-10, use_zero_guess=True)
    x1 = ctx.zeros(n * n)
    i1 = fsx.cg_solve(A, ctx.vec(b), x1, fsx.Settings(**s), dinv=d)
    h1 = fsx.cg_history(ctx)
    seen = []
    x2 = ctx.zeros(n * n)
    i2 = fsx.cg_solve_diag(A, ctx.vec(b), x2, fsx.Settings(**s),
                           lambda x, res: seen.append(res) and False, dinv=d)
    assert i2.as_dict() == i1.as_dict()
    assert np.array_equal(x2.get(), x1.get())
    np.testing.assert_array_equal(np.array(seen), h1)

    # stop at the 9th call: converged_user, iters = 9
    calls = []
    x3 = ctx.zeros(n * n)
    i3 = fsx.cg_solve_diag(A, ctx.vec(b), x3, fsx.Settings(**s),
                           lambda x, res: calls.append(res) or len(calls) == 9, dinv=d)
    oc = []
    xo, io, _ = O.cg(Ao, b, np.zeros(n * n), O.Settings(**s), P=O.prec(1, Ao.dinv()),
                     diag=lambda x, res: oc.append(res) or len(oc) == 9)
    assert i3.reason == io.reason == "converged_user"
    assert i3.iters == io.iters == 9
    assert rel(x3.get(), xo) <= 1e-13
    np.testing.assert_allclose(calls, oc, rtol=1e-12)

    # the reference test: b = 0, x0 = random, the A-norm of the error (= x)
    # falls monotonically and below 2 ((sqrt k - 1)/(sqrt k + 1))^i |e0|_A
    lam = np.array([4 - 2 * np.cos(np.pi * i / (n + 1)) - 2 * np.cos(np.pi * j / (n + 1))
                    for i in range(1, n + 1) for j in range(1, n + 1)])
    kappa = lam.max() / lam.min()
    S = sp.csr_matrix((v, ci, rp))
    x0 = np.random.default_rng(7).random(n * n)
    anorm = lambda y: np.sqrt(y @ (S @ y))
    e0 = anorm(x0)
    errs = []
    xd = ctx.vec(x0)
    i4 = fsx.cg_solve_diag(A, ctx.zeros(n * n), xd,
                           fsx.Settings(maxiter=2000, rtol=1e-9, use_zero_guess=False),
                           lambda x, res: errs.append(anorm(x.get())) and False)
    assert i4.reason == "converged_rtol" and i4.iters == len(errs)
    frac = (np.sqrt(kappa) - 1) / (np.sqrt(kappa) + 1)
    bound = 2 * frac ** np.arange(1, len(errs) + 1) * e0
    assert np.all(np.diff(np.concatenate([[e0], errs])) < 0)
    assert np.all(np.array(errs) < bound)

    class Stop(RuntimeError):
        pass

    def bad(x, res):
        raise Stop("from the diagnostic")

    with pytest.raises(Stop):
        fsx.cg_solve_diag(A, ctx.vec(b), ctx.zeros(n * n), fsx.Settings(**s), bad, dinv=d)
    # the context still solves afterwards
    x5 = ctx.zeros(n * n)
    i5 = fsx.cg_solve(A, ctx.vec(b), x5, fsx.Settings(**s), dinv=d)
    assert i5.as_dict() == i1.as_dict()


@pytest.mark.parametrize("dims", [(3, 5, 4), (32, 32), (33, 31), (181, 180), (512, 512), (513, 512),
                                  (64, 64, 64), (65, 64, 64)])
def test_resident_solves_iteration_matched(ctx, dims):
    """Small stencil systems run all iterations in one launch, a thread per
    four rows: row counts below, at and past a workgroup's 1024, and at and
    past the largest system (262144 rows), told by the launches made; 25
    iterations with Jacobi and without, from a nonzero guess, against the
    oracle's trajectory."""
    S = None
    for m in dims:
        L = sp.diags([2.0 * np.ones(m), -np.ones(m - 1), -np.ones(m - 1)], [0, 1, -1])
        S = L if S is None else sp.kron(sp.eye(m), S) + sp.kron(L, sp.eye(S.shape[0]))
    S = sp.csr_matrix(S)
    n = S.shape[0]
    # a varying diagonal, so that Jacobi differs from the identity
    S = sp.csr_matrix(S + sp.diags(P.uniform(n, 71, 0.0, 2.0)))
    S.sort_indices()
    rp, ci, v = S.indptr.astype(np.int32), S.indices.astype(np.int32), S.data
    Ao = O.Csr(rp, ci, v)
    A = ctx.csr(rp, ci, v)
    assert A.plan() == (4, 0) or n < 1000
    b, x0 = P.uniform(n, 72), P.uniform(n, 73)
    s = dict(maxiter=25, rtol=1e-15)
    for jac in (True, False):
        xo, io, ho = O.cg(Ao, b, x0, O.Settings(**s), P=O.prec(1, Ao.dinv()) if jac else None,
                          hist_cap=25)
        xd = ctx.vec(x0)
        d, bd, before = A.diag_inv() if jac else None, ctx.vec(b), ctx.counters()[1]
        info = fsx.cg_solve(A, bd, xd, fsx.Settings(**s), dinv=d)
        launches = ctx.counters()[1] - before
        assert (launches < 25) == (n <= 262144 and A.plan() == (4, 0)), launches
        assert info.reason == io.reason
        np.testing.assert_allclose(fsx.cg_history(ctx), ho, rtol=1e-9)
        assert rel(xd.get(), xo) <= 1e-12


@pytest.mark.parametrize("n", [48, 400])  # one and two rows per lane in the launched product
def test_solves_from_two_threads(ctx, n):
    """Two threads, each on a context of its own, solve small systems at once:
    one resident solve runs at a time and the other thread's takes the
    launched loop, with the same bits."""
    import threading
    rp, ci, v = P.poisson2d(n)
    b = P.uniform(n * n, 81)
    s = dict(maxiter=2000, rtol=1e-10, use_zero_guess=True)

    def solve(c, out, reps):
        A = c.csr(rp, ci, v)
        d, bd, x = A.diag_inv(), c.vec(b), c.zeros(n * n)
        for _ in range(reps):
            i = fsx.cg_solve(A, bd, x, fsx.Settings(**s), dinv=d)
            out.append((i.iters, x.get()))

    want, got = [], [[], []]
    solve(ctx, want, 1)
    ctxs = [fsx.Context(0), fsx.Context(0)]
    th = [threading.Thread(target=solve, args=(ctxs[k], got[k], 15)) for k in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for out in got:
        assert len(out) == 15
        for it, x in out:
            assert it == want[0][0]
            np.testing.assert_array_equal(x, want[0][1])


def context_with(monkeypatch, **env):
    """A context created under environment switches (read at creation)."""
    for k, v in env.items():
        monkeypatch.setenv(k, str(v))
    c = fsx.Context(0)
    for k in env:
        monkeypatch.delenv(k)
    return c


@pytest.mark.parametrize("how", ["jacobi", "identity", "noalloc", "diag", "rr"])
@pytest.mark.parametrize("give_up", [1, 2, 4])
def test_resident_give_up_continues(ctx, monkeypatch, how, give_up):
    """A resident launch that gives up, at a solve's first launch or after
    launches that already advanced it: the launched loop goes on from where
    the last good launch ended, so iterates, iteration counts, history and the
    diagnostic's calls are those of a solve that never was resident, bit for
    bit (one row per lane on both sides)."""
    n = 24
    rp, ci, v, _ = diffusion(n)
    N = n ** 3
    b, x0 = P.uniform(N, 91), P.uniform(N, 92)

    def solve(c):
        A = c.csr(rp, ci, v)
        bd, x, seen = c.vec(b), c.vec(x0), []
        s = fsx.Settings(maxiter=500, rtol=1e-9)
        if how == "rr":
            A32 = A.convert(fsx.F32)
            A32.set_values_sym_scaled(A)
            i = fsx.ir_cg_rr_solve(A, A32, bd, x, 1e-10, fsx.Settings(maxiter=500, rtol=1e-3))
            return x.get(), (i.status, i.outer_iters, i.inner_iters_total), seen, []
        d = A.diag_inv() if how != "identity" else None
        if how == "diag":
            u = [c.vec(P.uniform(N, 95 + k)) for k in range(4)]
            rr, rz = C.c_double(), C.c_double()

            def diag(xv, res):
                # sums of the diagnostic's own, on the same context
                seen.append((res, xv.get().tobytes(), fsx.nrm2(xv)))
                fsx.check(fsx.lib().fsx_cg_update(c.h, 0.0, u[0].h, u[1].h, None, u[2].h, u[3].h,
                                                  None, C.byref(rr), C.byref(rz)))
                return False
            i = fsx.cg_solve_diag(A, bd, x, s, diag, dinv=d)
        else:
            i = (fsx.cg_solve_noalloc if how == "noalloc" else fsx.cg_solve)(A, bd, x, s, dinv=d)
        h = [] if how == "noalloc" else fsx.cg_history(c)
        return x.get(), i.as_dict(), seen, list(h)

    want = solve(context_with(monkeypatch, FSX_CG_RESIDENT=0))
    got = solve(context_with(monkeypatch, FSX_CG_RESIDENT_ITERS=7,
                             FSX_CG_RESIDENT_GIVE_UP=give_up))
    np.testing.assert_array_equal(got[0], want[0])
    assert got[1:] == want[1:]
    # past the last iteration: the launch before the end gives up, or none
    if how == "jacobi" and give_up == 1:
        last = (want[1]["iters"] + 6) // 7
        for k in (last, last + 1):
            got = solve(context_with(monkeypatch, FSX_CG_RESIDENT_ITERS=7,
                                     FSX_CG_RESIDENT_GIVE_UP=k))
            np.testing.assert_array_equal(got[0], want[0])
            assert got[1:] == want[1:]


def test_resident_give_up_is_remembered(ctx, monkeypatch):
    """After a give-up a context's solves take the launched loop (five launches
    an iteration) at once, segments of a refinement included."""
    n = 20
    rp, ci, v, _ = diffusion(n)
    b = P.uniform(n ** 3, 93)

    def launches(c, refine=False):
        A = c.csr(rp, ci, v)
        d, bd, x = A.diag_inv(), c.vec(b), c.zeros(n ** 3)
        A32 = A.convert(fsx.F32)
        A32.set_values_sym_scaled(A)
        before = c.counters()[1]
        if refine:
            i = fsx.ir_cg_rr_solve(A, A32, bd, x, 1e-10, fsx.Settings(maxiter=500, rtol=1e-2))
            its = i.inner_iters_total
        else:
            its = fsx.cg_solve(A, bd, x, fsx.Settings(maxiter=500, rtol=1e-9), dinv=d).iters
        return c.counters()[1] - before, its

    # resident: a reset and a launch beside the setup's few
    k, its = launches(context_with(monkeypatch, FSX_CG_RESIDENT_GIVE_UP=0))
    assert its > 40 and k < 20
    c = context_with(monkeypatch, FSX_CG_RESIDENT_GIVE_UP=1)
    never = context_with(monkeypatch, FSX_CG_RESIDENT=0)
    extra = 2
    for refine in (False, False, True):
        k, its = launches(c, refine)
        k0, its0 = launches(never, refine)
        assert its == its0 and k0 >= (3 if refine else 5) * its0
        assert k == k0 + extra  # the reset and launch that gave up
        extra = 0


@pytest.mark.parametrize("dims", [(130, 1007), (362, 363), (64, 64, 50), (7, 93, 397), (512, 512)])
def test_resident_bits_do_not_depend_on_the_path(ctx, monkeypatch, dims):
    """Whether a solve of small size is resident depends on other threads, so
    its bits must not: the launched loop and the resident one at sizes below,
    at and past the two rows per lane of the launched FP64 product, up to the
    largest resident system, in one launch and in several."""
    S = None
    for m in dims:
        L = sp.diags([2.0 * np.ones(m), -np.ones(m - 1), -np.ones(m - 1)], [0, 1, -1])
        S = L if S is None else sp.kron(sp.eye(m), S) + sp.kron(L, sp.eye(S.shape[0]))
    S = sp.csr_matrix(S + sp.diags(P.uniform(S.shape[0], 71, 0.0, 2.0)))
    S.sort_indices()
    n = S.shape[0]
    b, x0 = P.uniform(n, 72), P.uniform(n, 73)

    def solve(c, jac):
        A = c.csr(S.indptr.astype(np.int32), S.indices.astype(np.int32), S.data)
        x = c.vec(x0)
        i = fsx.cg_solve(A, c.vec(b), x, fsx.Settings(maxiter=60, rtol=1e-15),
                         dinv=A.diag_inv() if jac else None)
        return x.get(), i.as_dict(), list(fsx.cg_history(c))

    launched = context_with(monkeypatch, FSX_CG_RESIDENT=0)
    parts = context_with(monkeypatch, FSX_CG_RESIDENT_ITERS=13)
    for jac in (True, False):
        want = solve(launched, jac)
        for c in (ctx, parts):
            got = solve(c, jac)
            np.testing.assert_array_equal(got[0], want[0])
            assert got[1:] == want[1:]


@pytest.mark.parametrize("symmetric", [True, False])
@pytest.mark.parametrize("n", [20_000, 150_001])
def test_resident_bits_on_general_lists(ctx, monkeypatch, n, symmetric):
    """Seven offsets without -1 and +1: the launched FP64 products run on the
    stencil layout (two rows a lane from 131072) or, not symmetric, on slice
    offsets, the FP32 ones on slice offsets; the resident solves keep their
    bits."""
    m = int(n ** 0.5)
    rng = np.random.default_rng(n)
    S = sp.diags([4.5 + rng.random(n)], [0])
    for o in (2, 7, m):
        u = -rng.uniform(0.2, 0.8, n - o)
        S = S + sp.diags([u, u if symmetric else u * rng.uniform(0.9, 1.1, n - o)], [o, -o])
    S = sp.csr_matrix(S)
    S.sort_indices()
    b, x0 = P.uniform(n, 72), P.uniform(n, 73)

    def solve(c):
        A = c.csr(S.indptr.astype(np.int32), S.indices.astype(np.int32), S.data)
        assert A.plan() == ((4, 0) if symmetric else (3, 0))
        x, before = c.vec(x0), c.counters()[1]
        i = fsx.cg_solve(A, c.vec(b), x, fsx.Settings(maxiter=40, rtol=1e-15), dinv=A.diag_inv())
        out = [x.get(), i.as_dict(), list(fsx.cg_history(c)), c.counters()[1] - before]
        A32 = A.convert(fsx.F32)
        A32.set_values_sym_scaled(A)
        x = c.vec(x0)
        r = fsx.ir_cg_rr_solve(A, A32, c.vec(b), x, 1e-10, fsx.Settings(maxiter=20, rtol=1e-2),
                               max_segments=3)
        return out + [x.get(), r.inner_iters_total]

    want, got = solve(context_with(monkeypatch, FSX_CG_RESIDENT=0)), solve(ctx)
    assert got[3] < 30 < want[3]
    np.testing.assert_array_equal(got[0], want[0])
    assert got[1:3] == want[1:3]
    np.testing.assert_array_equal(got[4], want[4])
    assert got[5] == want[5]


def test_resident_solve_inside_a_diagnostic(ctx):
    """A diagnostic may solve on another context: nothing of the resident solve
    it was called from is held meanwhile, so the inner one is resident too."""
    n = 16
    rp, ci, v, _ = diffusion(n)
    b = P.uniform(n ** 3, 94)
    s = fsx.Settings(maxiter=500, rtol=1e-9, use_zero_guess=True)

    def solve(c, diag=None):
        A = c.csr(rp, ci, v)
        d, bd, x = A.diag_inv(), c.vec(b), c.zeros(n ** 3)
        before = c.counters()[1]
        i = fsx.cg_solve_diag(A, bd, x, s, diag, dinv=d) if diag else \
            fsx.cg_solve(A, bd, x, s, dinv=d)
        return i.iters, c.counters()[1] - before, x.get()

    want = solve(ctx)
    inner, other = [], fsx.Context(0)

    def diag(x, res):
        if len(inner) < 3:
            inner.append(solve(other))
        return False

    got = solve(ctx, diag)
    assert want[1] < 20 < want[0]
    for it, k, x in inner:
        assert (it, k) == want[:2]
        np.testing.assert_array_equal(x, want[2])
    # two launches an iteration on the outer context: it stayed resident
    assert got[0] == want[0] and got[1] <= 2 * got[0] + 20
    np.testing.assert_array_equal(got[2], want[2])


def test_resident_slot_taken_between_launches(ctx, monkeypatch):
    """A diagnostic's solve (a resident launch an iteration) whose slot another
    thread's long solve takes meanwhile: it goes on in the launched loop from
    its own state, whatever the diagnostic summed on its context, same bits."""
    import threading
    import time
    n = 20
    rp, ci, v, _ = diffusion(n)
    N = n ** 3
    b = P.uniform(N, 97)
    big = P.poisson2d(512)
    s = fsx.Settings(maxiter=500, rtol=1e-9, use_zero_guess=True)
    u = [ctx.vec(P.uniform(N, 98 + k)) for k in range(4)]
    rr, rz = C.c_double(), C.c_double()

    def solve(at_five):
        A = ctx.csr(rp, ci, v)
        d, bd, x, calls = A.diag_inv(), ctx.vec(b), ctx.zeros(N), []

        def diag(xv, res):
            calls.append(res)
            fsx.check(fsx.lib().fsx_cg_update(ctx.h, 0.0, u[0].h, u[1].h, None, u[2].h, u[3].h,
                                              None, C.byref(rr), C.byref(rz)))
            if len(calls) == 5:
                at_five()
            return False

        before = ctx.counters()[1]
        i = fsx.cg_solve_diag(A, bd, x, s, diag, dinv=d)
        return x.get(), i.as_dict(), calls, ctx.counters()[1] - before

    other = context_with(monkeypatch, FSX_CG_RESIDENT_ITERS=20000)
    B = other.csr(*big)
    bb, xb = other.vec(P.uniform(512 * 512, 99)), other.zeros(512 * 512)
    long = fsx.Settings(maxiter=20000, rtol=1e-300, use_zero_guess=True)
    fsx.cg_solve(B, bb, xb, fsx.Settings(maxiter=2, rtol=1e-300, use_zero_guess=True))
    th = threading.Thread(target=fsx.cg_solve, args=(B, bb, xb, long))

    def start():
        th.start()
        time.sleep(0.03)  # the long solve's one launch takes about 190 ms

    want = solve(lambda: None)
    got = solve(start)
    th.join()
    np.testing.assert_array_equal(got[0], want[0])
    assert got[1:3] == want[1:3]
    assert got[3] > want[3] + want[1]["iters"]  # it did go on in the launched loop


@pytest.mark.parametrize("where", ["rhs", "guess", "matrix"])
def test_resident_not_finite_as_launched(ctx, monkeypatch, where):
    """A NaN or an infinity in the right-hand side, the guess or the matrix: the
    resident solve runs into it as the launched one does -- the same counts,
    history and places of NaN -- and ends."""
    n = 40
    rp, ci, v = P.poisson2d(n)
    rows = np.repeat(np.arange(n * n), np.diff(rp))
    never = context_with(monkeypatch, FSX_CG_RESIDENT=0)
    for bad in (np.nan, np.inf):
        b, x0, w = P.uniform(n * n, 61), P.uniform(n * n, 62), v.copy()
        if where == "rhs":
            b[777] = bad
        elif where == "guess":
            x0[5] = bad
        else:
            w[(rows == 801) & (ci == 801)] = bad
        for jac in (True, False):
            out = []
            for c in (ctx, never):
                A = c.csr(rp, ci, w)
                assert A.plan() == (4, 0)
                x = c.vec(x0)
                i = fsx.cg_solve(A, c.vec(b), x, fsx.Settings(maxiter=30, rtol=1e-8),
                                 dinv=A.diag_inv() if jac else None)
                out.append((x.get(), i.reason, i.iters, fsx.cg_history(c)))
            np.testing.assert_array_equal(out[0][0], out[1][0])
            assert out[0][1:3] == out[1][1:3]
            np.testing.assert_array_equal(out[0][3], out[1][3])


def test_solves_while_another_thread_captures(ctx, monkeypatch):
    """One thread captures graphs over and over (a new matrix each solve, in the
    launched loop) while another finishes small solves and reads their history:
    nothing it does touches the other's capture."""
    import threading
    rp, ci, v = P.poisson2d(24)
    b = P.uniform(24 * 24, 82)
    s = fsx.Settings(maxiter=400, rtol=1e-8, use_zero_guess=True)
    cap, sol = context_with(monkeypatch, FSX_CG_RESIDENT=0), fsx.Context(0)
    done, err, out = threading.Event(), [], []

    def capture():
        try:
            for _ in range(60):
                A = cap.csr(rp, ci, v)
                x = cap.zeros(b.size)
                out.append((fsx.cg_solve(A, cap.vec(b), x, s).iters, x.get()))
                A.destroy()
        except Exception as e:
            err.append(e)
        done.set()

    th = threading.Thread(target=capture)
    A = sol.csr(rp, ci, v)
    bd, x = sol.vec(b), sol.zeros(b.size)
    th.start()
    want = fsx.cg_solve(A, bd, x, s).iters, x.get()
    while not done.is_set():
        assert fsx.cg_solve(A, bd, x, s).iters == want[0]
        assert len(fsx.cg_history(sol)) == want[0]
    th.join()
    assert not err, err
    for it, xo in out:
        assert it == want[0]
        np.testing.assert_array_equal(xo, want[1])
