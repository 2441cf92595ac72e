"""U8 weights: few rows on the int8 matrix cores (bytes as q - 128), many rows on the f16 ones, whose activations keep 22 bits of every value whatever its row holds."""
import numpy as np
import pytest

import fastnn_amd
from fastnn_amd import lib as flib

pytestmark = pytest.mark.gpu


def exact(pw, a, n, k, bias):
    kb = -(-k // 4) * 4
    q = np.ascontiguousarray(pw.words).view(np.uint8)[:n * kb].reshape(n, kb)[:, :k].astype(np.float64)
    a = a.astype(np.float64)
    return (a @ q.T) * pw.scales.astype(np.float64) + pw.zeros.astype(np.float64) * a.sum(1, keepdims=True) + bias


def weights(rng, n, k):
    """Ranges that lie anywhere: around zero, off it, on one side, of one value, a few values far out."""
    w = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    w[1::7] += 0.3
    w[2::7] = np.abs(w[2::7]) + 2.0
    w[3::7] = -1.0
    w[4, 0] = 30.0
    return w


def off(got, want):
    return float(np.linalg.norm(got - want) / np.linalg.norm(want))


# (9 to 16 rows: where the option asks for them)
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 8, 9, 12, 13, 16])
@pytest.mark.parametrize("tiles", [0, 3])
@pytest.mark.parametrize("k,n", [(64, 16), (528, 100), (2048, 40), (2576, 264)])
def test_few_rows(m, tiles, k, n):
    """30-bit activations and 64-bit sums: what is left is the rounding of the sum and of the bias added to it, 2^-24 each at most; the f16 kernels are 1.3e-7 to 3e-7 off."""
    rng = np.random.default_rng(m * 1000 + k)
    pw = fastnn_amd.quantize_weights(flib.DT_U8, weights(rng, n, k))
    a = rng.standard_normal((m, k)).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    bad = a.copy()
    bad[m - 1, k // 2] = np.nan
    large = a.copy()
    large[:, k // 3] = 200.0
    with fastnn_amd.HipContext(0) as ctx:
        h = ctx.register(pw)
        ctx.set_option(flib.OPT_FRAGMENT, -1)
        ctx.set_option(flib.OPT_STREAM_MAX_M, 0)
        ctx.set_option(flib.OPT_GEMV_INT8_MAX_M, 16)
        ctx.set_option(flib.OPT_GEMV_ROW_TILES, tiles)
        want = exact(pw, a, n, k, bias)
        got = ctx.qmatmul(h, a, n, bias=bias)
        assert off(got, want) < 1.2e-7
        assert off(ctx.qmatmul(h, large, n, bias=bias), exact(pw, large, n, k, bias)) < 1.2e-7
        other = ctx.qmatmul(h, bad, n, bias=bias)
        assert np.isnan(other[m - 1]).all() and np.array_equal(other[:-1], got[:-1])
        ctx.set_option(flib.OPT_GEMV_INT8, 0)
        assert not np.array_equal(ctx.qmatmul(h, a, n, bias=bias), got)
        ctx.release(h)


@pytest.mark.parametrize("form", [1, 2, 4, 1 | 2 << 3, 1 | 4 << 3, 2 | 4 << 3])
@pytest.mark.parametrize("m,k,n", [(33, 200, 129), (130, 2600, 260), (1090, 130, 3900)])
def test_register_tiles(form, m, k, n):
    """U8 has none of those: asked for them, a call is what it is without.  4e-7 of the result's norm at most with the values drawn here."""
    rng = np.random.default_rng(m + form)
    pw = fastnn_amd.quantize_weights(flib.DT_U8, weights(rng, n, k))
    a = rng.standard_normal((m, k)).astype(np.float32)
    a[5] = 0.0
    bias = rng.standard_normal(n).astype(np.float32)
    bad = a.copy()
    bad[7, k - 1] = np.inf
    keep = np.setdiff1d(np.arange(m), [7])
    with fastnn_amd.HipContext(0) as ctx:
        h = ctx.register(pw)
        ctx.set_option(flib.OPT_FRAGMENT, -1)
        plain = ctx.qmatmul(h, a, n, bias=bias)
        ctx.set_option(flib.OPT_FRAGMENT, 1 << 14 | form)
        want = exact(pw, a, n, k, bias)
        got = ctx.qmatmul(h, a, n, bias=bias)
        assert off(got, want) < 4e-7 and got.tobytes() == plain.tobytes()
        broken = ctx.qmatmul(h, bad, n, bias=bias)
        assert not np.isfinite(broken[7]).any() and np.array_equal(broken[keep], got[keep])
        ctx.release(h)


@pytest.mark.parametrize("value", [0.0, 50.0, 200.0, 1e4])
def test_rows_with_one_large_value(value):
    """Digit planes below the row's largest value would leave the others 23 - log2(value) bits: 2.5e-6 of the result's norm off at 200.  Hi and lo halves keep 22
    bits of each; what is left is their f32 sums, 2.8e-7 to 5.7e-7 measured."""
    m, k, n = 512, 4096, 4096
    rng = np.random.default_rng(1)
    pw = fastnn_amd.quantize_weights(flib.DT_U8, (rng.standard_normal((n, k)) * 0.05).astype(np.float32))
    a = rng.standard_normal((m, k)).astype(np.float32)
    if value:
        a[:, 77] = value
    sel = np.arange(0, m, 16)
    with fastnn_amd.HipContext(0) as ctx:
        h = ctx.register(pw)
        assert off(ctx.qmatmul(h, a, n)[sel], exact(pw, a[sel], n, k, 0.0)) < 9e-7
        ctx.release(h)


@pytest.mark.parametrize("form", [1, 2, 4, 1 | 2 << 3])
def test_long_rows_with_the_tiles_asked_for(form):
    """A lane and the zero point's steps are up to 384 together: 384 * 128 * K passes 2^31 from K = 43691 on (in 32-bit sums -128849 for 134324).  The sums are f32, of products of one sign, added 16 and more at a time: 45000 / 16
    additions, each half of 2^-24 of the sum off at most, 8.4e-5 where all err to one side."""
    m, k, n = 40, 45000, 64
    q = np.full((n, k), 255, np.uint8)       # 1.5, and one weight of 0.5
    q[:, 7] = 0
    words = np.concatenate([q.reshape(-1).view(np.uint32), np.zeros(16, np.uint32)])
    pw = fastnn_amd.PackedWeight(flib.DT_U8, n, k, words, np.full(n, 1 / 255, np.float32), np.full(n, 0.5, np.float32))
    a = np.full((m, k), 1.99, np.float32)
    with fastnn_amd.HipContext(0) as ctx:
        h = ctx.register(pw)
        ctx.set_option(flib.OPT_FRAGMENT, 1 << 14 | form)
        assert off(ctx.qmatmul(h, a, n), exact(pw, a, n, k, 0.0)) < 8.4e-5
        ctx.release(h)
