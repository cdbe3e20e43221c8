"""Trailing-update and U12 products on both sides of the line between the
64x64 tiles and the large ones (128x128, direct-to-LDS or staged through
registers): a product with at least one 128x128 tile per CU runs the large
tile whatever the line, a small one the 64x64 tile, and an element's bits may
depend neither on the tile nor on its place in it."""
import numpy as np
import pytest

import lu2_amd as L

pytestmark = pytest.mark.gpu

# 18 x 17 tiles of 128x128, more than the device's 256 CUs
RAGGED = (2200, 2111)
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
