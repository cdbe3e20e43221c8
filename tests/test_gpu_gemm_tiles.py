"""Products that take another tile by their size or alignment give the bits
of the tile they stand for; the residual's sums at small and ragged sizes."""
import numpy as np
import pytest

import lu2_amd as L

pytestmark = pytest.mark.gpu


def product(ctx, a, b, c, ld):
    """C - A B with A, B and C in one matrix of row stride ld, as lu2 lays
    them out (B and C share their columns, A and C their rows)."""
    (m, k), n = a.shape, b.shape[1]
    full = np.zeros((m + k, ld))
    full[k:, :k], full[:k, k:k + n], full[k:, k:k + n] = a, b, c
    d = ctx.alloc(full.nbytes)
    d.upload(full)
    ctx.dgemm_dev(m, n, k, -1.0, d, ld, d, ld, 1.0, d, ld, offs=(8 * k * ld, 8 * k, 8 * (k * ld + k)))
    out = d.download(np.float64, full.size).reshape(full.shape)
    d.free()
    return out[k:, k:k + n].copy()


@pytest.mark.parametrize("m,n,k", [(64, 64, 16), (65, 63, 32), (128, 1, 48), (1, 130, 16), (300, 257, 64),
                                   (700, 900, 17), (16300, 17 * 128, 32)])
def test_unaligned_rows_give_the_aligned_bits(ctx, m, n, k):
    """An odd row stride (unaligned 16-byte loads) against an even one: the
    same tiles and K order, so the same bits (the last case in 128x128 tiles, with element loads)."""
    rng = np.random.default_rng(m + 3 * n + k)
    a, b, c = rng.standard_normal((m, k)), rng.standard_normal((k, n)), rng.standard_normal((m, n))
    odd, even = n + k + 1 + (n + k) % 2, n + k + (n + k) % 2
    assert odd % 2 == 1 and even % 2 == 0
    got = product(ctx, a, b, c, odd)
    u = 2.0 ** -53
    gamma = (k + 2) * u / (1 - (k + 2) * u)
    assert np.all(np.abs(got - (c - a @ b)) <= 2 * gamma * (np.abs(a) @ np.abs(b) + np.abs(c)))
    if k % 2 == 0:   # A, B and C start on 16-byte boundaries in the even layout
        assert np.array_equal(got, product(ctx, a, b, c, even))


@pytest.mark.parametrize("form", [1, 2])
@pytest.mark.parametrize("kernel", [1, 0])
@pytest.mark.parametrize("m,n,k", [(64, 64, 32), (130, 66, 64), (256, 1000, 256), (200, 2, 208)])
def test_small_trailing_products_give_the_large_tile_bits(ctx, form, kernel, m, n, k):
    """Trailing updates (form 1) and U12 products (form 2: A lower
    triangular, k = m there) below one 128x128 tile per CU against the same
    rows and columns of a product above."""
    if form == 2:
        k = m
    rng = np.random.default_rng(m + 5 * n + k)
    wide_m, wide_n = (m, 33000) if form == 2 else (4224, 2176)
    a, b = rng.standard_normal((wide_m, k)), rng.standard_normal((k, wide_n))
    if form == 2:
        a = np.tril(a)
    out = {}
    ctx.set_option(L.OPT_TRAIL_KERNEL, kernel)
    ctx.set_option(L.OPT_DGEMM_TRAILING, form)
    try:
        for tag, (mm, nn) in (("large", (wide_m, wide_n)), ("small", (m, n))):
            alpha, beta = (1.0, 0.0) if form == 2 else (-1.0, 1.0)
            da, db, dc = ctx.alloc(8 * mm * k), ctx.alloc(8 * k * nn), ctx.alloc(8 * mm * nn)
            da.upload(np.ascontiguousarray(a[:mm]))
            db.upload(np.ascontiguousarray(b[:, :nn]))
            dc.upload(np.zeros((mm, nn)))
            ctx.dgemm_dev(mm, nn, k, alpha, da, k, db, nn, beta, dc, nn)
            out[tag] = dc.download(np.float64, mm * nn).reshape(mm, nn)
            for d in (da, db, dc):
                d.free()
    finally:
        ctx.set_option(L.OPT_DGEMM_TRAILING, 0)
        ctx.set_option(L.OPT_TRAIL_KERNEL, 1)   # the library default
    assert np.array_equal(out["large"][:m, :n], out["small"])


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 65, 255, 257, 1031])
def test_residual_small_and_ragged(ctx, n):
    rng = np.random.default_rng(n)
    a = np.zeros((n, n + 16))
    a[:, :n + 1] = rng.uniform(-0.5, 0.5, (n, n + 1))
    x = rng.uniform(-0.5, 0.5, n)
    da, dx = ctx.alloc(a.nbytes), ctx.alloc(8 * n)
    da.upload(a)
    dx.upload(x)
    got = ctx.residual_dev(n, da, n + 16, dx)
    da.free()
    dx.free()
    m, b = a[:, :n], a[:, n]
    want = [np.abs(m @ x - b).max(), np.abs(m).sum(axis=1).max(), np.abs(m).sum(axis=0).max(), np.abs(x).max(),
            np.abs(x).sum(), np.abs(b).max()]
    # two n-term sums in different orders, terms below 1/2 and 1/4
    np.testing.assert_allclose(got[:6], want, rtol=0, atol=2 * n * n * 2.0 ** -53)
