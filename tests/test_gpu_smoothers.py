"""Device hybrid Gauss-Seidel (fsx_gs_*, op::hybrid_gs of
flecsolve/solvers/mg/gs.hh) against the oracle (gpu).

Bar: bit-identical to the oracle's sequential sweep (the level-scheduled
kernels do each row's arithmetic in the reference's order) for forward,
backward and symmetric sweeps, one and several colours, int32 and int64
indices, rows whose columns are not sorted, and one-colour grid stencils
swept in shared-memory tiles (with partial tiles, planes, lines and
wrap-around couplings that fall back to the level copies); the level count
equals
the dependency depth the mathematics fixes (2n - 1 for the 5-point stencil
on n^2, 3n - 2 for the 7-point stencil on n^3, 1 for a diagonal matrix).
"""
import numpy as np
import pytest
import scipy.sparse as sp

from flecsolve_amd import fsx
from flecsolve_amd import problems as P
from oracle import oracle as O
from test_oracle_smoothers import random_csr

pytestmark = pytest.mark.gpu


def run_both(ctx, rp, ci, v, sweep, nrelax, ncolours, seed=1):
    n = rp.size - 1
    A = ctx.csr(rp, ci, v)
    b = P.uniform(n, seed)
    x0 = P.uniform(n, seed + 1)
    G = fsx.HybridGS(A, ncolours=ncolours)
    x = ctx.vec(x0)
    G.apply(ctx.vec(b), x, sweep=sweep, nrelax=nrelax)
    ref = O.Csr(rp, ci, v).hybrid_gs(b, x0, sweep=sweep, nrelax=nrelax, ncolours=ncolours)
    return x.get(), ref, G


@pytest.mark.parametrize("sweep", [0, 1, 2])
@pytest.mark.parametrize("nrelax", [1, 2])
def test_poisson2d_bit_exact(ctx, sweep, nrelax):
    rp, ci, v = P.poisson2d(64)
    got, ref, G = run_both(ctx, rp, ci, v, sweep, nrelax, 1)
    np.testing.assert_array_equal(got, ref)
    assert G.levels() == (2 * 64 - 1, 2 * 64 - 1)


@pytest.mark.parametrize("ncolours", [1, 5])
def test_diffusion3d_bit_exact(ctx, ncolours):
    n = 16
    rp, ci, v = P.diffusion3d(n, P.lognormal_field(n, 1.0, 4.0, 7))
    got, ref, G = run_both(ctx, rp, ci, v, 2, 2, ncolours, seed=3)
    np.testing.assert_array_equal(got, ref)
    if ncolours == 1:
        assert G.levels() == (3 * n - 2, 3 * n - 2)


@pytest.mark.parametrize("itype", [np.int32, np.int64])
@pytest.mark.parametrize("ncolours", [1, 3])
def test_random_unsorted_rows_bit_exact(ctx, itype, ncolours):
    rp, ci, v, _ = random_csr(500, 0.02, 17)
    for sweep in (0, 1, 2):
        got, ref, _ = run_both(ctx, rp.astype(itype), ci.astype(itype), v, sweep, 1,
                               ncolours, seed=5 + sweep)
        np.testing.assert_array_equal(got, ref)


def test_diagonal_is_one_level(ctx):
    n = 1000
    d = 2.0 + P.uniform(n, 4)
    rp, ci = np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32)
    got, ref, G = run_both(ctx, rp, ci, d, 2, 1, 1)
    np.testing.assert_array_equal(got, ref)
    assert G.levels() == (1, 1)


def test_graph_replay_and_value_update(ctx):
    """Replays of the captured sweep, on two different x vectors and after an
    in-place change of the matrix values, each equal the oracle."""
    n = 20
    rp, ci, v = P.diffusion3d(n, P.lognormal_field(n, 1.0, 4.0, 9))
    A = ctx.csr(rp, ci, v)
    G = fsx.HybridGS(A)
    b = P.uniform(n ** 3, 10)
    bd = ctx.vec(b)
    x0 = P.uniform(n ** 3, 11)
    Ao = O.Csr(rp, ci, v)
    for rep in range(3):
        x1, x2 = ctx.vec(x0), ctx.vec(x0 * 2.0)
        G.apply(bd, x1, sweep=2, nrelax=1)
        G.apply(bd, x2, sweep=2, nrelax=1)
        np.testing.assert_array_equal(x1.get(), Ao.hybrid_gs(b, x0, 2, 1))
        np.testing.assert_array_equal(x2.get(), Ao.hybrid_gs(b, x0 * 2.0, 2, 1))
    v2 = v * 1.5
    A.set_values(v2)
    x = ctx.vec(x0)
    G.apply(bd, x, sweep=2, nrelax=1)
    np.testing.assert_array_equal(x.get(), O.Csr(rp, ci, v2).hybrid_gs(b, x0, 2, 1))


def grid_matrix(nx, ny, nz, seed, periodic_x=False, itype=np.int32):
    """Random diagonally dominant 7-point matrix (5-point for nz = 1, 3-point
    for ny = nz = 1) on an nx x ny x nz grid in natural order, columns
    ascending; periodic_x adds the wrap-around couplings along x."""
    rng = np.random.default_rng(seed)
    n = nx * ny * nz
    rp, ci, v = [0], [], []
    for r in range(n):
        i, j, k = r % nx, (r // nx) % ny, r // (nx * ny)
        cols = {r: 0.0}
        for di, dj, dk in ((1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1)):
            a, b2, c = i + di, j + dj, k + dk
            if periodic_x and di and nx > 2:
                a %= nx
            if 0 <= a < nx and 0 <= b2 < ny and 0 <= c < nz:
                cols[a + nx * (b2 + ny * c)] = -rng.random()
        cols[r] = 7.0 + rng.random()
        for c in sorted(cols):
            ci.append(c)
            v.append(cols[c])
        rp.append(len(ci))
    return np.array(rp, itype), np.array(ci, itype), np.array(v)


@pytest.mark.parametrize("tiles", ["1", "0"])
@pytest.mark.parametrize("dims,periodic,itype", [((21, 13, 9), False, np.int32),
                                                 ((16, 8, 24), False, np.int64),
                                                 ((37, 37, 1), False, np.int32),
                                                 ((100, 1, 1), False, np.int32),
                                                 ((12, 10, 6), True, np.int32)])
def test_grid_tiles_bit_exact(ctx, monkeypatch, tiles, dims, periodic, itype):
    """One-colour stencil matrices on a grid are swept in 8^3 tiles, one
    launch per tile diagonal, cells relaxed in shared memory
    (FSX_GS_TILES=0: the level copies instead): bit-identical to the oracle's
    sequential sweep for grids that leave partial tiles in every dimension,
    a plane, a line, int64 indices, and a matrix with wrap-around couplings
    (not a grid stencil: the level copies either way); forward, backward and
    symmetric, one and two repetitions."""
    monkeypatch.setenv("FSX_GS_TILES", tiles)
    rp, ci, v = grid_matrix(*dims, seed=sum(dims), periodic_x=periodic, itype=itype)
    for sweep in (0, 1, 2):
        for nrelax in (1, 2):
            got, ref, G = run_both(ctx, rp, ci, v, sweep, nrelax, 1, seed=3 + sweep)
            np.testing.assert_array_equal(got, ref)
    if not periodic and dims[2] > 1:
        assert G.levels() == (sum(dims) - 2, sum(dims) - 2)


def pairs_matrix(n, seed):
    """Rows 2i and 2i+1 coupled, nothing else: two levels of n/2 rows each."""
    rng = np.random.default_rng(seed)
    rp, ci, v = [0], [], []
    for r in range(n):
        o = r ^ 1
        cols = sorted({r, o})
        for c in cols:
            ci.append(c)
            v.append(4.0 + rng.random() if c == r else -rng.random())
        rp.append(len(ci))
    return np.array(rp, np.int32), np.array(ci, np.int32), np.array(v)


@pytest.mark.parametrize("run_rows", ["0", "1", "7", "512"])
def test_level_runs_bit_exact(ctx, monkeypatch, run_rows):
    """Consecutive levels of at most FSX_GS_RUN_ROWS rows (at most 512) run
    in one workgroup with a barrier between levels, the next level's rows
    loaded ahead (0: a launch per level, 1: only one-row levels grouped, 512:
    every level that fits, runs split every 1024 levels): bit-identical to
    the oracle's sequential sweep on random rows (one and three colours; up
    to ~50 entries a row, past the 16 loaded at once), a chain of 2500
    one-row levels, a 3D stencil, two levels of 500 rows and two levels of
    3000 rows (a launch each)."""
    monkeypatch.setenv("FSX_GS_TILES", "0")
    monkeypatch.setenv("FSX_GS_RUN_ROWS", run_rows)
    rr = random_csr(500, 0.02, 17)[:3]
    dense = random_csr(300, 0.1, 19)[:3]
    assert np.diff(dense[0]).max() > 16 + 8
    cases = [(rr, 1), (rr, 3), (dense, 1), (dense, 2), (grid_matrix(2500, 1, 1, seed=5), 1),
             (P.diffusion3d(12, P.lognormal_field(12, 1.0, 4.0, 8)), 1),
             (pairs_matrix(1000, 6), 1), (pairs_matrix(6000, 6), 1)]
    for (rp, ci, v), ncolours in cases:
        for sweep in (0, 1, 2):
            for nrelax in (1, 2):
                got, ref, G = run_both(ctx, rp, ci, v, sweep, nrelax, ncolours, seed=7 + sweep)
                np.testing.assert_array_equal(got, ref)
    assert G.levels() == (2, 2)


def test_errors(ctx):
    rp, ci, v = P.poisson2d(8)
    A = ctx.csr(rp, ci, v)
    with pytest.raises(fsx.FsxError):
        fsx.HybridGS(A, ncolours=0)
    with pytest.raises(fsx.FsxError):
        fsx.HybridGS(A, ncolours=65)
    G = fsx.HybridGS(A)
    with pytest.raises(fsx.FsxError):
        G.apply(ctx.vec(np.ones(63)), ctx.zeros(64))
    with pytest.raises(fsx.FsxError):
        G.apply(ctx.vec(np.ones(64)), ctx.zeros(64), sweep=3)
    rect = ctx.csr(np.array([0, 1, 2], np.int32), np.array([0, 3], np.int32),
                   np.array([1.0, 1.0]), ncols=4)
    with pytest.raises(fsx.FsxError):
        fsx.HybridGS(rect)


def mirrored_csr(n, per_row, seed, long_rows=0, long_len=60):
    """Random matrix with a symmetric structure (values not), a full diagonal,
    columns ascending; `long_rows` rows couple to `long_len` others."""
    rng = np.random.default_rng(seed)
    i = rng.integers(0, n, n * per_row // 2)
    j = np.clip(i + rng.integers(-40, 41, i.size), 0, n - 1)
    for r in rng.choice(n, long_rows, replace=False):
        i = np.append(i, np.full(long_len // 2, r))
        j = np.append(j, rng.choice(n, long_len // 2, replace=False))
    S = sp.csr_matrix((np.ones(2 * i.size + n),
                       (np.r_[i, j, np.arange(n)], np.r_[j, i, np.arange(n)])), (n, n))
    S.sum_duplicates()
    S.sort_indices()
    v = rng.uniform(-1.0, 1.0, S.nnz)
    rows = np.repeat(np.arange(n), np.diff(S.indptr))
    v[S.indices == rows] = 8.0 + rng.random(n)
    return S.indptr, S.indices, v


@pytest.mark.parametrize("itype", [np.int32, np.int64])
@pytest.mark.parametrize("n,per_row,long_rows", [
    (1, 2, 0), (63, 4, 0), (65, 6, 2), (3000, 9, 5), (4000, 20, 9),
    (20478, 6, 3),   # the largest whose x fits one CU's shared memory
    (20479, 6, 3),   # the first one past it
])
def test_relaxation_in_shared_memory_bit_exact(ctx, itype, n, per_row, long_rows):
    """Small one-colour matrices run every level of every sweep in one
    workgroup (levels of more and fewer than 64 rows, rows of more than 8, 16
    and 24 entries); larger ones, and those whose structure is not symmetric,
    keep a launch or a run per level: the oracle's bits on both sides."""
    rp, ci, v = mirrored_csr(n, per_row, 100 + n, min(long_rows, n), min(60, n))
    for sweep, nrelax in ((0, 1), (1, 1), (2, 3)):
        got, ref, _ = run_both(ctx, rp.astype(itype), ci.astype(itype), v, sweep, nrelax, 1,
                               seed=9 + sweep)
        np.testing.assert_array_equal(got, ref)


def wide_level_csr(m, parts):
    """9-point matrix on m x m, numbered part by part of parts x parts rows of
    independent points: `parts`^2 levels of m^2 / parts^2 rows."""
    T = sp.diags([np.ones(m), np.ones(m - 1), np.ones(m - 1)], [0, 1, -1])
    S = sp.csr_matrix(sp.kron(T, T))
    rng = np.random.default_rng(m)
    S.data = rng.uniform(-1.0, 1.0, S.nnz)
    S = sp.csr_matrix(S + sp.diags(np.full(m * m, 12.0)))
    i = np.arange(m * m)
    order = np.argsort((i % m) % parts + parts * ((i // m) % parts), kind="stable")
    S = S[order][:, order].tocsr()
    S.sort_indices()
    return S.indptr.astype(np.int32), S.indices.astype(np.int32), S.data


@pytest.mark.parametrize("m,parts,shared", [(140, 8, True), (130, 4, False), (140, 2, False)])
def test_wide_levels_keep_their_launches(ctx, m, parts, shared):
    """Matrices whose x fits one CU's shared memory, with levels of 306, 1056
    and 4900 rows: one workgroup takes the first, every CU works on a level of
    the others.  The oracle's bits, and one copy of the matrix on the device."""
    rp, ci, v = wide_level_csr(m, parts)
    n, off = m * m, ci.size - m * m
    A = ctx.csr(rp, ci, v)
    before = fsx.alloc_stats()[1]
    G = fsx.HybridGS(A)
    held = fsx.alloc_stats()[1] - before
    levels = G.levels()[0]
    assert (n / levels <= 768) == shared
    per_row = n * (4 + 4 + 8 + 8)          # ids, lengths, diagonals and their entries
    record = n * (8 * 18 + 4)              # eight columns, values and entries
    slots = 2 * (off + n) * 20 + 8 * n     # columns, values and entries; x kept aside
    want = 2 * per_row + (2 * record if shared else slots)
    assert held <= want * 1.05 + 65536, (held, want)
    del G
    for sweep, nrelax in ((0, 1), (1, 1), (2, 2)):
        got, ref, _ = run_both(ctx, rp, ci, v, sweep, nrelax, 1, seed=19 + sweep)
        np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_shared_memory_relaxation_not_finite(ctx, bad):
    """A NaN or an infinity in b or x reaches exactly the rows it reaches in the
    sequential sweep (rows of more and fewer than 24 entries, padded ones)."""
    n = 3000
    rp, ci, v = mirrored_csr(n, 9, 3, 5)
    A = ctx.csr(rp.astype(np.int32), ci.astype(np.int32), v)
    Ao = O.Csr(rp.astype(np.int32), ci.astype(np.int32), v)
    G = fsx.HybridGS(A)
    for in_b, at in ((True, n - 3), (False, 1500), (False, 0)):
        b, x = P.uniform(n, 41), P.uniform(n, 42)
        (b if in_b else x)[at] = bad
        for sweep in (0, 1, 2):
            xd = ctx.vec(x)
            G.apply(ctx.vec(b), xd, sweep, 1)
            ref = Ao.hybrid_gs(b, x, sweep=sweep, nrelax=1)
            np.testing.assert_array_equal(xd.get(), ref)
