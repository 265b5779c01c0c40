"""Batched persistent CG (fsx_batch_*) against the oracle, system by system (gpu).

Each system is an independent lognormal-k diffusion problem; the oracle solves
each one separately with the reference's serial CG + Dinv.  Bar: every system
converged, iteration counts within +-2, x within 1e-10 relative.
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


def make(nsys=24, emin=3, emax=12, sigma=1.0, seed=4001):
    e, rows, rp, ci, v = P.batch(nsys, emin, emax, seed, 4100, sigma)
    b = P.uniform(int(rows[-1]), 4200)
    return e, rows, rp, ci, v, b


def local(rows, rp, ci, v, s):
    lo, hi = rows[s], rows[s + 1]
    e0, e1 = rp[lo], rp[hi]
    return (rp[lo:hi + 1] - e0).astype(np.int64), (ci[e0:e1] - lo).astype(np.int64), v[e0:e1]


def check_against_oracle(rows, rp, ci, v, b, xg, it, st, rtol=1e-10, slack=2):
    for s in range(rows.size - 1):
        sl = slice(rows[s], rows[s + 1])
        Ao = O.Csr(*local(rows, rp, ci, v, s))
        xo, io, _ = O.cg(Ao, b[sl], np.zeros(rows[s + 1] - rows[s]),
                         O.Settings(maxiter=1000, rtol=rtol, use_zero_guess=True),
                         P=O.prec(1, Ao.dinv()))
        assert st[s] == 1, (s, st[s])
        assert abs(int(it[s]) - io.iters) <= slack, (s, it[s], io.iters)
        assert rel(xg[sl], xo) <= 1e-10, s


@pytest.mark.parametrize("cfg", [(256, 2, 1), (1024, 2, 1), (256, 0, 1), (1024, 0, 1),
                                 (64, 0, 1), (256, 1, 2), (512, 1, 4), (256, 1, 8)])
def test_batched_cg_matches_oracle(ctx, cfg):
    e, rows, rp, ci, v, b = make()
    A = ctx.csr(rp, ci, v)
    assert A.plan() == (3, 0)
    A.set_plan(2)   # also build the sliced layout for mapping 0
    A.set_plan(3)
    B = fsx.Batch(A, rows)
    assert B.config()[1] == 2
    B.set_config(*cfg)
    assert B.config() == cfg
    d = A.diag_inv()
    bd, x = ctx.vec(b), ctx.zeros(b.size)
    it, st, rs = B.cg(bd, x, fsx.Settings(maxiter=1000, rtol=1e-10, use_zero_guess=True),
                      dinv=d)
    check_against_oracle(rows, rp, ci, v, b, x.get(), it, st)


def test_batched_same_result_any_order_or_config(ctx):
    # a system's arithmetic is independent of which workgroup solved it
    e, rows, rp, ci, v, b = make(40, 4, 10)
    A = ctx.csr(rp, ci, v)
    B = fsx.Batch(A, rows)
    d = A.diag_inv()
    bd = ctx.vec(b)
    outs = []
    for wg in (256, 1024):
        B.set_config(wg, 2, 1)
        x = ctx.zeros(b.size)
        it, st, rs = B.cg(bd, x, fsx.Settings(maxiter=500, rtol=1e-10, use_zero_guess=True),
                          dinv=d)
        outs.append((x.get(), it))
    # workgroup size changes the reduction tree, so compare to rounding
    assert np.abs(outs[0][1] - outs[1][1]).max() <= 2
    assert rel(outs[0][0], outs[1][0]) <= 1e-10
    # repeat with the same config: bit-identical
    x = ctx.zeros(b.size)
    it, st, rs = B.cg(bd, x, fsx.Settings(maxiter=500, rtol=1e-10, use_zero_guess=True),
                      dinv=d)
    np.testing.assert_array_equal(x.get(), outs[1][0])


def test_batched_autotune(ctx):
    e, rows, rp, ci, v, b = make(64, 4, 16, seed=77)
    A = ctx.csr(rp, ci, v)
    B = fsx.Batch(A, rows)
    d = A.diag_inv()
    bd, x = ctx.vec(b), ctx.zeros(b.size)
    ms = B.tune(bd, x, d, sample=16, iters=10)
    assert ms > 0
    wg, mapping, lanes = B.config()
    assert wg in (256, 512, 1024) and mapping in (1, 2) and lanes in (1, 2, 4, 8)
    x = ctx.zeros(b.size)
    it, st, rs = B.cg(bd, x, fsx.Settings(maxiter=1000, rtol=1e-10, use_zero_guess=True),
                      dinv=d)
    check_against_oracle(rows, rp, ci, v, b, x.get(), it, st)


@pytest.mark.parametrize("jacobi", [1, 2])
@pytest.mark.parametrize("sigma", [1.0, 2.5])
def test_batched_ir_reaches_1e10(ctx, sigma, jacobi):
    e, rows, rp, ci, v, b = make(32, 4, 14, sigma=sigma)
    A = ctx.csr(rp, ci, v)
    A32 = A.convert(fsx.F32)
    if jacobi == 2:
        A32.set_values_sym_scaled(A)
    B = fsx.Batch(A, rows)
    bd, x = ctx.vec(b), ctx.zeros(b.size)
    outer, inner, st, rs = B.ir_cg(A32, bd, x, 1e-10, fsx.Settings(maxiter=2000, rtol=1e-4),
                                   jacobi=jacobi)
    assert (st == 1).all()
    S = sp.csr_matrix((v, ci, rp))
    xg = x.get()
    for s in range(rows.size - 1):
        sl = slice(rows[s], rows[s + 1])
        r = b[sl] - (S[sl] @ xg)
        assert np.linalg.norm(r) / np.linalg.norm(b[sl]) <= 1.01e-10, s
        assert outer[s] >= 1 and inner[s] >= outer[s]


@pytest.mark.parametrize("sigma", [1.0, 2.5])
def test_batched_rr_against_model(ctx, sigma):
    """Per system, the FP32 CG with FP64 residual replacement
    (fsx_batched_rr_cg): every system at true residual <= 1e-10, each
    system's segment and FP32 iteration counts those of the CPU model in its
    two-reduction form with FP64 row sums (tests/rr_model.py; +-1 / +-3; the
    model with FP32 row sums is 5-7 iterations away on some systems, so the
    bar separates the two products), fewer FP32 iterations
    in total than the restarted refinement on the same FP32 matrix, and the
    same x bit for bit under the sliced and slice-offset mappings (both sum
    rows serially)."""
    import rr_model as M
    e, rows, rp, ci, v, b = make(32, 4, 14, sigma=sigma)
    A = ctx.csr(rp, ci, v)
    A.set_plan(2)   # the sliced layout too, for mapping 0
    A.set_plan(3)
    A32 = A.convert(fsx.F32)
    A32.set_values_sym_scaled(A)
    B = fsx.Batch(A, rows)
    bd = ctx.vec(b)
    inner = fsx.Settings(maxiter=2000, rtol=1e-2)
    outs = []
    # the same workgroup size (it sets the reduction tree), two row mappings
    for cfg in ((256, 2, 1), (256, 0, 1)):
        B.set_config(*cfg)
        x = ctx.zeros(b.size)
        outs.append((B.rr_cg(A32, bd, x, 1e-10, inner), x.get()))
    (seg, its, st, rs), xg = outs[0]
    np.testing.assert_array_equal(outs[1][1], xg)
    np.testing.assert_array_equal(outs[1][0][1], its)
    assert (st == 1).all()
    S = sp.csr_matrix((v, ci, rp))
    for k in range(rows.size - 1):
        sl = slice(rows[k], rows[k + 1])
        assert np.linalg.norm(b[sl] - S[sl] @ xg) / np.linalg.norm(b[sl]) <= 1.01e-10, k
        assert abs(rs[k] - np.linalg.norm(b[sl] - S[sl] @ xg)) <= 1e-3 * rs[k] + 1e-300
        _, msegs, mits, mst, _ = M.rr_solve(*local(rows, rp, ci, v, k), b[sl], 1e-10, 1e-2,
                                            2000, 100, single_reduction=False, acc64=True)
        assert mst == 1
        assert abs(int(seg[k]) - msegs) <= 1, (k, seg[k], msegs)
        assert abs(int(its[k]) - mits) <= 3, (k, its[k], mits)
    x2 = ctx.zeros(b.size)
    outer, inner_r, st2, _ = B.ir_cg(A32, bd, x2, 1e-10, fsx.Settings(maxiter=2000, rtol=1e-4),
                                     jacobi=2)
    assert (st2 == 1).all()
    assert its.sum() < inner_r.sum()
    with pytest.raises(fsx.FsxError):
        B.rr_cg(A32, bd, x, 1e-10, fsx.Settings(maxiter=2000, rtol=1.0))


def test_batched_edge_cases(ctx):
    e, rows, rp, ci, v, b = make(6, 2, 5)
    b[rows[2]:rows[3]] = 0.0       # zero right-hand side: converged at once
    A = ctx.csr(rp, ci, v)
    B = fsx.Batch(A, rows)
    bd, x = ctx.vec(b), ctx.zeros(b.size)
    it, st, rs = B.cg(bd, x, fsx.Settings(maxiter=200, rtol=1e-10, use_zero_guess=True),
                      dinv=A.diag_inv())
    assert it[2] == 0 and st[2] == 1
    assert (st == 1).all()
    # maxiter exhausted: iters 0, diverged_iters (cg.hh:135-136)
    it, st, rs = B.cg(bd, x, fsx.Settings(maxiter=1, rtol=1e-14, use_zero_guess=True))
    assert ((it == 0) & (st == 4) | (it == 0) & (st == 1)).all()
    # coupled systems are rejected
    rp2, ci2 = rp.copy(), ci.copy()
    ci2[rp2[rows[1]]] = rows[0]     # first row of system 1 points into system 0
    A2 = ctx.csr(rp2, ci2, v)
    with pytest.raises(fsx.FsxError):
        fsx.Batch(A2, rows)


def test_batched_full_edge_range_matches_oracle(ctx):
    """Edges spanning 8..48 as the 2048-system workload draws them, with an
    8^3 (512 rows) and a 48^3 system (110,592 rows in one workgroup): FP64
    CG + Jacobi under the autotuned mapping and under each mapping family,
    system by system against the oracle; then the FP32-inner refinement,
    every system at true residual <= 1e-10 and within 1e-8 of the oracle's
    1e-10 CG solution (each 1e-10-residual solution of these systems carries
    a forward error of up to 5e-10: the oracle's against its own rtol 1e-14
    solve)."""
    e, rows, rp, ci, v = P.batch(12, 8, 48, 4007, 4100, 1.0)
    assert 8 in e and 48 in e
    b = P.uniform(int(rows[-1]), 4200)
    A = ctx.csr(rp, ci, v)
    assert A.plan() == (3, 0)
    A.set_plan(2)   # the sliced layout too, for mapping 0
    A.set_plan(3)
    B = fsx.Batch(A, rows)
    d = A.diag_inv()
    bd = ctx.vec(b)
    s64 = fsx.Settings(maxiter=1000, rtol=1e-10, use_zero_guess=True)
    x = ctx.zeros(b.size)
    B.tune(bd, x, d, sample=12, iters=10)
    for cfg in (None, (1024, 2, 1), (256, 0, 1), (512, 1, 4)):
        if cfg is not None:
            B.set_config(*cfg)
        x = ctx.zeros(b.size)
        it, st, rs = B.cg(bd, x, s64, dinv=d)
        check_against_oracle(rows, rp, ci, v, b, x.get(), it, st)
    A32 = A.convert(fsx.F32)
    A32.set_values_sym_scaled(A)
    x = ctx.zeros(b.size)
    outer, inner, st, rs = B.ir_cg(A32, bd, x, 1e-10, fsx.Settings(maxiter=2000, rtol=1e-4),
                                   jacobi=2)
    assert (st == 1).all()
    S = sp.csr_matrix((v, ci, rp))
    xg = x.get()
    for k in range(rows.size - 1):
        sl = slice(rows[k], rows[k + 1])
        assert np.linalg.norm(b[sl] - S[sl] @ xg) / np.linalg.norm(b[sl]) <= 1.01e-10, k
        Ao = O.Csr(*local(rows, rp, ci, v, k))
        xo, io, _ = O.cg(Ao, b[sl], np.zeros(rows[k + 1] - rows[k]),
                         O.Settings(maxiter=1000, rtol=1e-10, use_zero_guess=True),
                         P=O.prec(1, Ao.dinv()))
        assert rel(xg[sl], xo) <= 1e-8, (k, e[k])


@pytest.mark.parametrize("edges", [
    (17,),                      # one system past the lockstep size, one block per slice edge
    (17, 8, 1, 5, 2),           # tiny systems beside it, none slice-aligned
    (24,) * 3 + (16,) * 5,      # one row a thread
    (48, 48, 47, 33, 9),        # two rows a thread
    (64,) * 16 + (63,) * 2,     # four rows a thread
])
def test_lockstep_matches_one_workgroup_per_system(ctx, edges):
    """Batches solved in lockstep (three launches advance every system) against
    the kernel of one workgroup per system, which a configuration set by the
    caller names: FP64 CG with and without Jacobi from zero and other guesses,
    exhausted iterations, and the FP32 CG with residual replacement.  Both run
    the same recurrences with sums in another order: iteration counts within
    two, solutions within the solves' own tolerance."""
    probs = [P.diffusion3d(e, P.lognormal_field(e, 1.0, 4.0, 900 + k))
             for k, e in enumerate(edges)]
    S = sp.block_diag([sp.csr_matrix((v, ci, rp)) for rp, ci, v in probs], format="csr")
    S.sort_indices()
    rows = np.concatenate([[0], np.cumsum([e ** 3 for e in edges])]).astype(np.int64)
    n = int(rows[-1])
    A = ctx.csr(S.indptr.astype(np.int32), S.indices.astype(np.int32), S.data)
    A.set_plan(3)
    A32 = A.convert(fsx.F32)
    A32.set_values_sym_scaled(A)
    b = P.uniform(n, 31)
    x0 = P.uniform(n, 32)
    bd, d = ctx.vec(b), A.diag_inv()
    lock, one = fsx.Batch(A, rows), fsx.Batch(A, rows)
    one.set_config(512, 2, 1)
    assert lock.lockstep() == (True, True) and one.lockstep() == (False, False)

    def both(f):
        out, launches = [], []
        for B in (lock, one):
            x, before = ctx.vec(x0), ctx.counters()[1]
            out.append((f(B, x), x.get()))
            launches.append(ctx.counters()[1] - before)
        # three launches a round, at least two chunks of eight; one launch
        assert launches[0] >= 48 and launches[1] < 10
        return out

    for dinv in (d, None):
        for s in (dict(maxiter=3000, rtol=1e-10, use_zero_guess=True),
                  dict(maxiter=3000, rtol=1e-10), dict(maxiter=7, rtol=1e-10),
                  dict(maxiter=0, rtol=1e-10), dict(maxiter=10, rtol=1e6)):
            (l, xl), (o, xo) = both(lambda B, x: B.cg(bd, x, fsx.Settings(**s), dinv=dinv))
            np.testing.assert_array_equal(l[1], o[1])
            # without a preconditioner CG on the lognormal operator loses
            # orthogonality over ~1000 iterations, and another order of the
            # sums moves its end by up to 1% (the bar of the single solves)
            assert (np.abs(l[0] - o[0]) <= (2 if dinv is not None else 2 + 0.01 * o[0])).all()
            # stopped by the iteration count: the same iterates to rounding;
            # by the residual: each within the tolerance of the solution
            assert rel(xl, xo) <= (1e-12 if s["maxiter"] <= 10 else 1e-8)
            if s["maxiter"] <= 10:
                np.testing.assert_allclose(l[2], o[2], rtol=1e-6)
            else:  # both under the tolerance of their system
                for got in (l, o):
                    assert (got[2] < 1e-10 * np.array([np.linalg.norm(b[rows[k]:rows[k + 1]])
                                                       for k in range(len(edges))])).all()
    for s, segs in ((fsx.Settings(maxiter=3000, rtol=3e-2), 100),
                    (fsx.Settings(maxiter=5, rtol=3e-2), 3), (fsx.Settings(maxiter=9, rtol=0.5), 0)):
        (l, xl), (o, xo) = both(lambda B, x: B.rr_cg(A32, bd, x, 1e-10, s, max_segments=segs))
        np.testing.assert_array_equal(l[2], o[2])
        assert np.abs(l[0] - o[0]).max() <= 1
        assert (np.abs(l[1] - o[1]) <= 3 + 0.02 * o[1]).all()
        assert rel(xl, xo) <= (1e-8 if segs == 100 else 1e-5)  # FP32 iterates short of the end
        if segs == 100:
            r = b - S @ xl
            for k in range(len(edges)):
                sl = slice(rows[k], rows[k + 1])
                assert np.linalg.norm(r[sl]) / np.linalg.norm(b[sl]) <= 1.01e-10
    # repeatable, bit for bit
    x1, x2 = ctx.vec(x0), ctx.vec(x0)
    s = fsx.Settings(maxiter=3000, rtol=1e-10)
    lock.cg(bd, x1, s, dinv=d)
    lock.cg(bd, x2, s, dinv=d)
    np.testing.assert_array_equal(x1.get(), x2.get())


def test_tuner_chooses_between_lockstep_and_one_workgroup(ctx):
    """The tuner times lockstep on the batch itself, says what it chose, and the
    solves run that: few systems with one far larger go in lockstep (three
    launches an iteration), systems of at most 4096 rows do not, a set
    configuration never does.  x keeps the systems that were not sampled."""
    def batch(edges):
        probs = [P.diffusion3d(e, P.lognormal_field(e, 1.0, 4.0, 950 + e)) for e in edges]
        S = sp.block_diag([sp.csr_matrix((v, ci, rp)) for rp, ci, v in probs], format="csr")
        S.sort_indices()
        A = ctx.csr(S.indptr.astype(np.int32), S.indices.astype(np.int32), S.data)
        rows = np.concatenate([[0], np.cumsum([e ** 3 for e in edges])]).astype(np.int64)
        return A, fsx.Batch(A, rows), int(rows[-1]), rows

    s = fsx.Settings(maxiter=400, rtol=1e-9, use_zero_guess=True)
    for edges, lock in (((40, 9, 8, 11), True), ((16, 9, 8, 11), False)):
        A, B, n, rows = batch(edges)
        d, bd = A.diag_inv(), ctx.vec(P.uniform(n, 33))
        x0 = P.uniform(n, 34)
        x = ctx.vec(x0)
        assert B.lockstep() == (lock, lock)  # by size
        for again in range(2):  # measured, then from the cache
            assert B.tune(bd, x, d, sample=1, iters=10) > 0
            assert B.lockstep() == (lock, lock)
        np.testing.assert_array_equal(x.get()[rows[1]:], x0[rows[1]:])  # the largest is sampled
        before = ctx.counters()[1]
        it, st, _ = B.cg(bd, x, s, dinv=d)
        launches = ctx.counters()[1] - before
        assert (st == 1).all()
        assert launches >= 3 * it.max() if lock else launches < 10
        x1 = x.get()
        B.set_config(512, 2, 1)
        assert B.lockstep() == (False, False)
        before = ctx.counters()[1]
        it1, st1, _ = B.cg(bd, x, s, dinv=d)
        assert ctx.counters()[1] - before < 10
        assert (st1 == 1).all() and np.abs(it1 - it).max() <= 2
        assert rel(x.get(), x1) <= 1e-8


def test_lockstep_by_size(ctx):
    """The size rule on both sides of its lines: at most 4096 rows; small
    systems enough to keep the CUs busy, for residual replacement earlier."""
    for edge, count, want in ((16, 8, (False, False)), (17, 8, (True, True)),
                              (18, 24, (True, True)), (18, 64, (True, False)),
                              (18, 140, (False, False)), (24, 64, (True, True))):
        rp, ci, v = P.diffusion3d(edge, P.lognormal_field(edge, 1.0, 4.0, 960))
        n = edge ** 3
        S = sp.csr_matrix((v, ci, rp))
        S = sp.block_diag([S] * count, format="csr")
        S.sort_indices()
        A = ctx.csr(S.indptr.astype(np.int32), S.indices.astype(np.int32), S.data)
        B = fsx.Batch(A, np.arange(count + 1, dtype=np.int64) * n)
        assert B.lockstep() == want, (edge, count)


def same_or_close(a, b, tol):
    """Equal infinities and NaN in the same places, the rest to a tolerance."""
    np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
    np.testing.assert_array_equal(a[np.isinf(a)], b[np.isinf(a)])
    ok = np.isfinite(b)
    assert np.isfinite(a[ok]).all()
    assert np.linalg.norm(a[ok] - b[ok]) <= tol * max(np.linalg.norm(b[ok]), 1e-300)


@pytest.mark.parametrize("case", ["rhs", "matrix"])
def test_lockstep_not_finite_as_one_workgroup(ctx, case):
    """Systems whose numbers run out, beside sound ones: a NaN and an infinity
    in the right-hand side, and a singular matrix whose first p.Ap is zero
    (alpha infinite).  Counts, reasons and the places of NaN and infinity are
    those of one workgroup per system."""
    if case == "rhs":
        edges = (20, 9, 17, 12)
        S = sp.block_diag([sp.csr_matrix((v, ci, rp)) for rp, ci, v in
                           (P.diffusion3d(e, P.lognormal_field(e, 1.0, 4.0, 970 + e))
                            for e in edges)], format="csr")
        rows = np.concatenate([[0], np.cumsum([e ** 3 for e in edges])]).astype(np.int64)
        b = P.uniform(int(rows[-1]), 35)
        b[rows[1] + 3], b[rows[3] - 70] = np.nan, np.inf
    else:
        m = 5000
        one = sp.kron(sp.eye(m // 2), np.ones((2, 2)))
        sound = sp.diags([np.full(m, 4.0), np.full(m - 1, -1.0), np.full(m - 1, -1.0)], [0, 1, -1])
        S = sp.block_diag([sound, one, sound], format="csr")
        rows = np.array([0, m, 2 * m, 3 * m], np.int64)
        b = P.uniform(3 * m, 36)
        b[m:2 * m] = np.tile([1.0, -1.0], m // 2)
    S = sp.csr_matrix(S)
    S.sort_indices()
    A = ctx.csr(S.indptr.astype(np.int32), S.indices.astype(np.int32), S.data)
    A.set_plan(3)
    A32 = A.convert(fsx.F32)
    A32.set_values_sym_scaled(A)
    lock, one = fsx.Batch(A, rows), fsx.Batch(A, rows)
    one.set_config(256, 2, 1)
    assert lock.lockstep() == (True, True)
    bd, d = ctx.vec(b), A.diag_inv()
    for guess in (True, False):
        for dinv in (d, None):
            s = fsx.Settings(maxiter=25, rtol=1e-6, use_zero_guess=guess)
            xl, xo = ctx.zeros(b.size), ctx.zeros(b.size)
            l, o = lock.cg(bd, xl, s, dinv=dinv), one.cg(bd, xo, s, dinv=dinv)
            np.testing.assert_array_equal(l[1], o[1])
            np.testing.assert_array_equal(l[0], o[0])
            same_or_close(l[2], o[2], 1e-6)
            same_or_close(xl.get(), xo.get(), 1e-8)
    xl, xo = ctx.zeros(b.size), ctx.zeros(b.size)
    s = fsx.Settings(maxiter=60, rtol=3e-2)
    l = lock.rr_cg(A32, bd, xl, 1e-9, s, max_segments=20)
    o = one.rr_cg(A32, bd, xo, 1e-9, s, max_segments=20)
    np.testing.assert_array_equal(l[2], o[2])
    np.testing.assert_array_equal(l[0], o[0])
    bad = o[2] != 1
    assert bad.any()
    np.testing.assert_array_equal(l[1][bad], o[1][bad])
    assert np.abs(l[1] - o[1]).max() <= 2
    same_or_close(xl.get(), xo.get(), 1e-8)


@pytest.mark.parametrize("count,edge,wg", [(200, 12, 1024), (300, 12, 256), (300, 13, 1024),
                                           (64, 11, 256), (520, 12, 256)])
def test_default_workgroup(ctx, count, edge, wg):
    """The size a batch starts with, on both sides of its lines (rows, more
    systems than CUs, than twice that)."""
    rp, ci, v = P.diffusion3d(edge, P.lognormal_field(edge, 1.0, 4.0, 980))
    S = sp.block_diag([sp.csr_matrix((v, ci, rp))] * count, format="csr")
    S.sort_indices()
    A = ctx.csr(S.indptr.astype(np.int32), S.indices.astype(np.int32), S.data)
    B = fsx.Batch(A, np.arange(count + 1, dtype=np.int64) * edge ** 3)
    assert B.config() == (wg, 2, 1)
