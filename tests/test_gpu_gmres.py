"""Fused device GMRES (fsx_gmres_solve) against the oracle's op::gmres::apply
(gpu).

Bar: iteration counts within +-2, restart counts consistent, x within 1e-10
relative on the convection-diffusion operator with right and left Jacobi
and without preconditioning; the restart-split identity of the reference's
gmres test (flecsolve/solvers/test/gmres.cc:88-110); settings validation
(gmres.hh:394-405); maxiter exhaustion; zero right-hand side.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from flecsolve_amd import fsx
from flecsolve_amd import problems as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n,side,jac", [(16, 1, False), (16, 1, True), (16, 0, True),
                                        (24, 1, True), (24, 0, False)])
def test_convdiff_matches_oracle(ctx, n, side, jac):
    rp, ci, v = P.convdiff3d(n, (10.0, 5.0, 2.5))
    Ao = O.Csr(rp, ci, v)
    b = P.uniform(n ** 3, 2101)
    s = dict(maxiter=600, rtol=1e-10, use_zero_guess=True, max_krylov_dim=30,
             restart=True, pre_side=side)
    xo, io, _ = O.gmres(Ao, b, np.zeros(n ** 3), O.Settings(**s),
                        P=O.prec(1, Ao.dinv()) if jac else None)
    A = ctx.csr(rp, ci, v)
    x = ctx.zeros(n ** 3)
    info = fsx.gmres_solve(A, ctx.vec(b), x, fsx.Settings(**s),
                           dinv=A.diag_inv() if jac else None)
    assert info.reason == io.reason == "converged_rtol"
    assert abs(info.iters - io.iters) <= 2, (info.iters, io.iters)
    assert abs(info.restarts - io.restarts) <= 1
    assert rel(x.get(), xo) <= 1e-10
    # same answer as the generic solver over device vectors
    xg = ctx.zeros(n ** 3)
    gi, _ = fsx.krylov("gmres", A, ctx.vec(b), xg, fsx.Settings(**s), prec=1 if jac else 0)
    assert abs(gi.iters - info.iters) <= 2
    assert rel(x.get(), xg.get()) <= 1e-10


def test_restart_split_identity(ctx):
    # flecsolve/solvers/test/gmres.cc:88-110 on the fused path
    rp, ci, v = P.poisson2d(24)
    A = ctx.csr(rp, ci, v)
    n = 576
    b = ctx.vec(O.set_random(n, 0))
    x0 = O.set_random(n, 1)
    x = ctx.vec(x0)
    ir = fsx.gmres_solve(A, b, x, fsx.Settings(maxiter=100, rtol=1e-6, max_krylov_dim=50,
                                                 restart=True))
    x = ctx.vec(x0)
    fsx.gmres_solve(A, b, x, fsx.Settings(maxiter=50, rtol=1e-6, max_krylov_dim=50,
                                          restart=True))
    i2 = fsx.gmres_solve(A, b, x, fsx.Settings(maxiter=100, rtol=1e-6, max_krylov_dim=100,
                                               restart=False))
    assert ir.restarts == 1
    assert 50 + i2.iters == ir.iters
    assert i2.res_norm_final == ir.res_norm_final


def test_validation_exhaustion_zero_rhs(ctx):
    rp, ci, v = P.convdiff3d(8, (10.0, 5.0, 2.5))
    A = ctx.csr(rp, ci, v)
    b = ctx.vec(P.uniform(512, 3))
    with pytest.raises(fsx.FsxError):   # krylov dimension above the bound
        fsx.gmres_solve(A, b, ctx.zeros(512), fsx.Settings(maxiter=200, max_krylov_dim=101,
                                                           restart=True))
    with pytest.raises(fsx.FsxError):   # no restart but maxiter > max_krylov_dim
        fsx.gmres_solve(A, b, ctx.zeros(512), fsx.Settings(maxiter=40, max_krylov_dim=30))
    info = fsx.gmres_solve(A, b, ctx.zeros(512), fsx.Settings(maxiter=5, rtol=1e-14,
                                                              max_krylov_dim=30,
                                                              restart=True,
                                                              use_zero_guess=True))
    assert (info.iters, info.reason) == (0, "diverged_iters")
    info = fsx.gmres_solve(A, ctx.zeros(512), ctx.zeros(512),
                           fsx.Settings(maxiter=5, rtol=1e-8, max_krylov_dim=30,
                                        restart=True, use_zero_guess=True))
    assert info.reason == "converged_rtol" and info.iters == 0


@pytest.mark.parametrize("dim", [1, 2, 63, 64, 65, 100])
@pytest.mark.parametrize("n", [4, 11, 17])
def test_basis_sizes_iteration_matched(ctx, dim, n):
    """The Gram-Schmidt pass at basis sizes around a wave's lanes and the
    largest, on vectors of less than a workgroup to several: cycles stopped by
    maxiter give the oracle's iterates (sums in another order: the Hessenberg
    column is off by rounding times the condition of the least-squares
    problem, so x to 1e-9), an orthogonal basis on an ill-conditioned matrix."""
    rp, ci, v = P.diffusion3d(n, P.lognormal_field(n, 2.0, 4.0, 55))
    N = n ** 3
    Ao = O.Csr(rp, ci, v)
    b = P.uniform(N, 2105)
    its = min(2 * dim, 130)
    s = dict(maxiter=its, rtol=1e-14, use_zero_guess=True, max_krylov_dim=dim, restart=True,
             pre_side=1)
    xo, io, _ = O.gmres(Ao, b, np.zeros(N), O.Settings(**s), P=O.prec(1, Ao.dinv()))
    A = ctx.csr(rp, ci, v)
    x = ctx.zeros(N)
    info = fsx.gmres_solve(A, ctx.vec(b), x, fsx.Settings(**s), dinv=A.diag_inv())
    S = sp.csr_matrix((v, ci, rp))
    ro, rg = np.linalg.norm(b - S @ xo), np.linalg.norm(b - S @ x.get())
    assert rg <= 1.01 * ro + 1e-11 * np.linalg.norm(b)
    if N > dim:  # the basis does not span the whole space
        assert info.reason == io.reason and info.restarts == io.restarts
        assert rel(x.get(), xo) <= 1e-9
