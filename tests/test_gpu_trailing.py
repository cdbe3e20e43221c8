"""Trailing-update and U12 products on both sides of the line between the
64x64 tiles and the large ones (128x128, direct-to-LDS or staged through
registers): a product with at least one 128x128 tile per CU runs the large
tile whatever the line, a small one the 64x64 tile, and an element's bits may
depend neither on the tile nor on its place in it."""
import numpy as np
import pytest

import lu2_amd as L

pytestmark = pytest.mark.gpu

# 18 x 17 tiles of 128x128, more than the device's 256 CUs, ragged and whole
RAGGED, WHOLE = (2200, 2111), (2304, 2176)
FORMS = [("f64", 1), ("f64", 0), ("f32", 1)]


def padded(a, rows, cols, dtype):
    out = np.zeros((rows, cols), dtype)
    out[:a.shape[0], :a.shape[1]] = a
    return out


def product(ctx, form, a, b, c, lower=False):
    """C - A B as the factorization's trailing update, or A B with A lower
    triangular as its U12 product, on 16-byte aligned rows."""
    prec, kernel = form
    dtype, unit = (np.float64, 2) if prec == "f64" else (np.float32, 4)
    (m, k), n = a.shape, b.shape[1]
    lda, ldb = -(-k // unit) * unit, -(-n // unit) * unit
    ops = [padded(a, m, lda, dtype), padded(b, k, ldb, dtype), padded(c, m, ldb, dtype)]
    bufs = [ctx.alloc(o.nbytes) for o in ops]
    for buf, o in zip(bufs, ops):
        buf.upload(o)
    ctx.set_option(L.OPT_TRAIL_KERNEL, kernel)
    ctx.set_option(L.OPT_DGEMM_TRAILING, 2 if lower else 1)
    try:
        gemm = ctx.dgemm_dev if prec == "f64" else ctx.sgemm_dev
        gemm(m, n, k, 1.0 if lower else -1.0, bufs[0], lda, bufs[1], ldb, 0.0 if lower else 1.0, bufs[2], ldb)
    finally:
        ctx.set_option(L.OPT_DGEMM_TRAILING, 0)
        ctx.set_option(L.OPT_TRAIL_KERNEL, 1)   # the library default
    out = bufs[2].download(dtype, m * ldb).reshape(m, ldb)
    for buf in bufs:
        buf.free()
    assert np.array_equal(out[:, n:], ops[2][:, n:])      # nothing written past column n
    return out[:, :n]


def operands(form, m, n, k, seed):
    dtype = np.float64 if form[0] == "f64" else np.float32
    rng = np.random.default_rng(seed)
    return tuple(rng.standard_normal(s).astype(dtype) for s in ((m, k), (k, n), (m, n)))


def check_bound(form, got, a, b, c):
    """|C - fl(C - AB)| <= gamma_{K+2} (|A||B| + |C|), the reference itself
    rounded in FP64."""
    u = 2.0 ** -53 if form[0] == "f64" else 2.0 ** -24
    k = a.shape[1]
    gamma = (k + 2) * u / (1 - (k + 2) * u)
    a, b, c = (x.astype(np.float64) for x in (a, b, c))
    assert np.all(np.abs(got - (c - a @ b)) <= 2 * gamma * (np.abs(a) @ np.abs(b) + np.abs(c)))


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("k", [40, 96])
@pytest.mark.parametrize("m,n", [(64, 64), (130, 66), (1, 300), (1536, 2048), (1664, 2047), (1920, 2176)])
def test_trailing_bits_do_not_depend_on_the_tile(ctx, form, k, m, n):
    """Products of 1 to 255 large tiles (192 and 208 among them, the two sides
    of the FP64 line at 3/4 of a tile per CU) against the first and the last
    rows and columns, edge tiles, of a ragged product above one tile per CU."""
    a, b, c = operands(form, *RAGGED, k, k)
    large = product(ctx, form, a, b, c)
    assert np.array_equal(large[:m, :n], product(ctx, form, a[:m], b[:, :n], c[:m, :n]))
    last = product(ctx, form, np.ascontiguousarray(a[-m:]), np.ascontiguousarray(b[:, -n:]),
                   np.ascontiguousarray(c[-m:, -n:]))
    assert np.array_equal(large[-m:, -n:], last)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("k", [40, 96])
def test_large_tiles_edge_and_interior(ctx, form, k):
    """The large tiles' bounds-checked loads do the arithmetic of their
    unchecked ones: a ragged product against one whose tiles are all interior
    (K filled up to whole stages with zeros)."""
    a, b, c = operands(form, *WHOLE, k, k + 1)
    a, b = padded(a, WHOLE[0], -(-k // 32) * 32, a.dtype), padded(b, -(-k // 32) * 32, WHOLE[1], b.dtype)
    whole = product(ctx, form, a, b, c)
    m, n = RAGGED
    ragged = product(ctx, form, np.ascontiguousarray(a[:m, :k]), np.ascontiguousarray(b[:k, :n]),
                     np.ascontiguousarray(c[:m, :n]))
    assert np.array_equal(whole[:m, :n], ragged)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("k", [17, 512])
def test_large_tiles_error_bound(ctx, form, k):
    a, b, c = operands(form, *RAGGED, k, k + 2)
    check_bound(form, product(ctx, form, a, b, c), a, b, c)


@pytest.mark.parametrize("kernel", [1, 0])
def test_u12_edge_interior_and_small(ctx, kernel):
    """The U12 product, A lower triangular, C not read: 8 x 33 large tiles,
    ragged and whole, within the product's error bound, and its first rows and
    columns as a product of their own in 64x64 tiles."""
    form, m, n = ("f64", kernel), 1000, 4200
    a, b, _ = operands(form, m, n, m, 3)
    a = np.tril(a)
    nan = np.full((1024, 4224), np.nan)
    ragged = product(ctx, form, a, b, nan[:m, :n], lower=True)
    check_bound(form, -ragged, a, b, np.zeros((m, n)))
    whole = product(ctx, form, padded(a, 1024, 1024, np.float64), padded(b, 1024, 4224, np.float64), nan, lower=True)
    assert np.array_equal(whole[:m, :n], ragged)
    for mm, nn in ((64, 64), (130, 66), (1, 300), (500, 4200)):
        small = product(ctx, form, np.ascontiguousarray(a[:mm, :mm]), np.ascontiguousarray(b[:mm, :nn]), nan[:mm, :nn],
                        lower=True)
        assert np.array_equal(ragged[:mm, :nn], small)
