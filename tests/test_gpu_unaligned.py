"""Products and factorizations on rows that are not 16-byte aligned: the bits
of the same on aligned rows."""
import numpy as np
import pytest

import lu2_amd as L

pytestmark = pytest.mark.gpu


def product(ctx, a, b, c, alpha, beta, ext):
    """alpha A B + beta C on rows of k + ext and n + ext elements."""
    (m, k), n = a.shape, b.shape[1]
    gemm = ctx.dgemm_dev if a.dtype == np.float64 else ctx.sgemm_dev
    bufs = []
    for x in (a, b, c):
        full = np.zeros((x.shape[0], x.shape[1] + ext), x.dtype)
        full[:, :x.shape[1]] = x
        bufs.append(ctx.alloc(full.nbytes))
        bufs[-1].upload(full)
    gemm(m, n, k, alpha, bufs[0], k + ext, bufs[1], n + ext, beta, bufs[2], n + ext)
    out = bufs[2].download(c.dtype, m * (n + ext)).reshape(m, n + ext)
    for buf in bufs:
        buf.free()
    return out


# an inner tile of 64x64 in every shape; K below, at and above one stage
# (FP64 16, FP32 32), and several stages with and without a remainder
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("m,n", [(64, 64), (130, 200), (641, 1088)])
@pytest.mark.parametrize("k", [1, 15, 16, 17, 32, 33, 63, 97, 500])
def test_unaligned_products_any_k(ctx, prec, m, n, k):
    dtype, unit, u = (np.float64, 2, 2.0 ** -53) if prec == "f64" else (np.float32, 4, 2.0 ** -24)
    rng = np.random.default_rng(m + n + k)
    a, b, c = (rng.standard_normal(s).astype(dtype) for s in ((m, k), (k, n), (m, n)))
    # an odd row stride of B and C (n is a multiple of the unit) against aligned rows, K filled up with zeros
    pad = (-k) % unit
    ap = np.concatenate([a, np.zeros((m, pad), dtype)], axis=1)
    bp = np.concatenate([b, np.zeros((pad, n), dtype)], axis=0)
    for alpha, beta, c0 in ((-1.0, 1.0, c), (1.0, 0.0, np.full_like(c, np.nan))):
        got = product(ctx, a, b, c0, alpha, beta, 1)
        assert not np.any(got[:, n:])                     # nothing written past column n
        got = got[:, :n]
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        cc = c.astype(np.float64) if beta else 0.0
        gamma = (k + 2) * u / (1 - (k + 2) * u)
        assert np.all(np.abs(got - (alpha * (a64 @ b64) + cc)) <= 2 * gamma * (np.abs(a64) @ np.abs(b64) + np.abs(cc)))
        assert np.array_equal(got, product(ctx, ap, bp, c0, alpha, beta, 0))


@pytest.mark.parametrize("n,nb", [(64, 32), (544, 32), (1024, 128), (2048, 256)])
def test_lu_odd_row_stride(ctx, oracle, n, nb):
    """A matrix of n + 1 columns without padding.  Its trailing updates run in
    the register-staged tiles, so its factors are those of the aligned matrix
    with these tiles chosen."""
    a0 = oracle.randomsetmat(n, n, n + 1)
    even = np.zeros((n, n + 16))
    even[:, :n + 1] = a0
    x, piv, f = L.solve(a0, nb, L.PIV_GEPP, ctx)
    ctx.set_option(L.OPT_TRAIL_KERNEL, 0)
    try:
        xe, pe, fe = L.solve(even, nb, L.PIV_GEPP, ctx)
    finally:
        ctx.set_option(L.OPT_TRAIL_KERNEL, 1)   # the library default
    assert np.array_equal(piv, pe) and np.array_equal(x, xe) and np.array_equal(f, fe[:, :n + 1])
    xo, po, _ = oracle.lumcolumn(a0, nb, oracle.PIV_GEPP)
    assert np.array_equal(piv, po)
    assert np.abs(x - xo).max() <= 1e-10 * np.abs(xo).max()
