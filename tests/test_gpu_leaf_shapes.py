"""The panel leaf where its exchange takes several batches of loads and a
second candidate per lane: more than 64 workgroups, 32 columns, several rows
per thread; ties, winners in the last workgroups, columns without a candidate."""
import ctypes

import numpy as np
import pytest

import lu2_amd as L

pytestmark = pytest.mark.gpu


def cm_panel(a, m):
    """cm_column_decomposition_recursive on all rows of a, by lu2's rule."""
    lib = L.load_library()
    lib.cm_column_decomposition_recursive.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p,
                                                      ctypes.c_int]
    cm = np.ascontiguousarray(a.T)
    pv = np.zeros(m, np.int32)
    lib.cm_column_decomposition_recursive(len(a), cm.ctypes.data, m, pv.ctypes.data, 0)
    return pv, cm.T


def tied_panel(rows, m, seed):
    """Columns 2t and 2t+1 are nonzero only in the rows r with r % (m/2) = t from
    one place on, and column 2t holds one magnitude there: all those rows tie
    (the lowest wins), exactly, since no other row changes these columns.  The
    places are spread from the first row to near the last."""
    rng = np.random.default_rng(seed)
    a = np.zeros((rows, m))
    for t in range(m // 2):
        r = np.arange(t, rows, m // 2)
        r = r[r >= (rows - 64) * t // (m // 2 - 1)]
        a[r, 2 * t] = rng.choice([-1.0, 1.0], len(r))
        a[r, 2 * t + 1] = rng.uniform(1.0, 2.0, len(r))
    return a


# workgroups: 40 of 2 rows per thread, 74 and 128 of 4; 32 columns: 39 of one
# row per thread (the first with a second batch of loads), 79, 128 of two
SHAPES = [(20000, 16), (75000, 16), (131072, 16), (9800, 32), (20000, 32), (65536, 32)]


@pytest.mark.parametrize("rows,m", SHAPES)
def test_leaf_ties_over_many_workgroups(oracle, rows, m):
    a = tied_panel(rows, m, rows + m)
    pv, _ = cm_panel(a, m)
    po, _ = oracle.cm_panel(a, m, 0, oracle.PIV_COMPAT)
    assert po.max() >= rows - 64     # the last places reach the last rows
    assert np.array_equal(pv, po)


@pytest.mark.parametrize("rows", [9800, 20000, 65536])
def test_leaf_32_columns_over_many_workgroups(oracle, rows):
    a = np.random.default_rng(rows).uniform(-0.5, 0.5, (rows, 32))
    pv, f = cm_panel(a, 32)
    po, fo = oracle.cm_panel(a, 32, 0, oracle.PIV_COMPAT)
    assert np.array_equal(pv, po)
    assert np.abs(f - fo).max() <= 1e-12 * np.abs(fo).max() * 32


@pytest.mark.parametrize("rows,m", SHAPES)
def test_leaf_columns_without_candidate(oracle, rows, m):
    """A NaN column in the middle of the leaf: the pivots of the oracle, which
    keeps the current row where no entry compares."""
    a = np.random.default_rng(rows + m).uniform(-0.5, 0.5, (rows, m))
    a[:, 5] = np.nan
    pv, _ = cm_panel(a, m)
    po, _ = oracle.cm_panel(a, m, 0, oracle.PIV_COMPAT)
    assert np.array_equal(pv, po)


@pytest.mark.parametrize("mode", ["gepp", "compat"])
@pytest.mark.parametrize("n,nb", [(288, 32), (512, 64), (544, 32), (2080, 32)])
def test_lu_columns_without_candidate(ctx, oracle, n, nb, mode):
    gpu, ref = (L.PIV_GEPP, oracle.PIV_GEPP) if mode == "gepp" else (L.PIV_COMPAT, oracle.PIV_COMPAT)
    a0 = oracle.randomsetmat(n, n + nb)
    a0[:, 21] = np.nan
    _, piv, _ = L.solve(a0, nb, gpu, ctx)
    _, po, _ = oracle.lumcolumn(a0, nb, ref)
    assert np.array_equal(piv, po)


# ---------------------------------------------------------------------------
# A whole factorization by 32-column leaves of 73 workgroups, three batches of
# loads in FP64 and two in FP32.  Column j has one entry of 1 (two or three in
# the tied columns), the rest below 2^-2/n: no elimination changes which
# entries are the large ones, so the pivots are known beforehand.
N, NB = 18560, 64
TIED = {0: 2, 3: 3, 17: 2, 31: 2}    # columns of the first leaf with so many entries of 1


def planted():
    """The matrix in the order of its pivots (row j pivots in column j), the
    place each row has at first, and the pivots."""
    rng = np.random.default_rng(9)
    a = np.zeros((N, N + 16))
    a[:, :N + 1] = (rng.random((N, N + 1), dtype=np.float32) - np.float32(0.5)) * np.float32(0.5 / N)
    a[np.arange(N), np.arange(N)] = 1.0
    place = np.empty(N, np.int64)
    # the first leaf's pivots in turn in the last workgroups (slots of 64 and
    # more) and on both sides of the first batch's end
    last = rng.permutation(np.arange(64 * 256, N))[:16]
    batch = rng.permutation(np.arange(36 * 256, 40 * 256))[:16]
    place[0:32:2], place[1:32:2] = last, batch
    rest = np.setdiff1d(np.arange(N), place[:32])
    place[32:] = rng.permutation(rest)
    taken = set()
    for col, many in TIED.items():   # ties with rows placed below the pivot, exact when their step comes
        a[col, :32] = 0.0
        a[col, col] = 1.0
        below = np.nonzero((place > place[col]) & (np.arange(N) >= 32))[0]
        losers = [r for r in rng.permutation(below) if r not in taken][:many - 1]
        taken.update(losers)
        a[losers, :32] = 0.0
        a[losers, col] = -1.0
    at = place.copy()                # where each row stands
    row_at = np.empty(N, np.int64)
    row_at[place] = np.arange(N)
    piv = np.empty(N, np.int32)
    for j in range(N):
        p = at[j]
        piv[j] = p
        moved = row_at[j]
        row_at[p], at[moved] = moved, p
        row_at[j], at[j] = j, j
    return a, place, piv


@pytest.fixture(scope="module")
def planted_matrix():
    return planted()


def test_lu_32_column_leaves_planted_pivots(ctx, planted_matrix):
    a, place, want = planted_matrix
    shuffled = np.empty_like(a)
    shuffled[place] = a
    ctx.set_option(L.OPT_LEAF_W, 32)
    try:
        x, piv, _ = L.solve(shuffled, NB, L.PIV_GEPP, ctx)
        xs, ps, _ = L.solve(a, NB, L.PIV_GEPP, ctx)
    finally:
        ctx.set_option(L.OPT_LEAF_W, 16)   # the library default
    assert np.array_equal(piv, want)
    assert np.array_equal(ps, np.arange(N))
    assert np.array_equal(x, xs)           # an element's operations do not depend on where its row stands


def test_mixed_32_column_leaves_planted_pivots(ctx, planted_matrix):
    """FP32 leaves, whose pivots are not returned: the rows in any order give
    the bits of the rows in the order of their pivots, before and after the
    refinement."""
    a, place, _ = planted_matrix
    shuffled = np.empty_like(a)
    shuffled[place] = a
    dA, dx = ctx.alloc(a.nbytes), ctx.alloc(8 * N)
    got = []
    ctx.set_option(L.OPT_PIVMODE, L.PIV_GEPP)
    ctx.set_option(L.OPT_LEAF_W, 32)
    try:
        for m in (shuffled, a):
            dA.upload(m)
            info = ctx.solve_mixed(N, dA, N + 16, NB, dx, L.PREC_FP32)
            got.append((info["resid_hpl2_initial"], info["gmres_used"], dx.download(np.float64, N)))
    finally:
        ctx.set_option(L.OPT_LEAF_W, 16)   # the library default
        dA.free()
        dx.free()
    assert got[0][:2] == got[1][:2] and not got[0][1]
    assert np.array_equal(got[0][2], got[1][2])
