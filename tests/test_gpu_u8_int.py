"""U8 weights on the int8 matrix cores (bytes as q - 128, the zero point's whole steps added to the integer sums): the vector kernel and the register tiles."""
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


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("k,n", [(64, 16), (528, 100), (2048, 40), (2576, 264)])
def test_few_rows(m, k, n):
    """30-bit activations and 64-bit sums: nothing but the rounding of the result to 32 bits is left, 2^-24 a value."""
    rng = np.random.default_rng(m * 1000 + k)
    pw = fastnn_amd.quantize_weights(flib.DT_U8, weights(rng, n, k))
    a = rng.standard_normal((m, k)).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    bad = a.copy()
    bad[m - 1, k // 2] = np.nan
    with fastnn_amd.HipContext(0) as ctx:
        h = ctx.register(pw)
        ctx.set_option(flib.OPT_FRAGMENT, -1)
        want = exact(pw, a, n, k, bias)
        assert off(ctx.qmatmul(h, a, n, bias=bias), want) < 3e-7
        got = ctx.qmatmul(h, bad, n, bias=bias)
        assert np.isnan(got[m - 1]).all() and (m == 1 or off(got[:-1], want[:-1]) < 3e-7)
        ctx.release(h)


@pytest.mark.parametrize("form", [1, 2, 4, 1 | 2 << 3, 1 | 4 << 3, 2 | 4 << 3])
@pytest.mark.parametrize("m,k,n", [(33, 200, 129), (130, 2600, 260), (1090, 130, 3900)])
def test_register_tiles(form, m, k, n):
    """Activations of 24 bits: 2^-23 of a row's largest value each, 4e-7 of the result's norm at most with the values drawn here."""
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
        ctx.set_option(flib.OPT_FRAGMENT, 1 << 14 | form)
        want = exact(pw, a, n, k, bias)
        got = ctx.qmatmul(h, a, n, bias=bias)
        assert off(got, want) < 4e-7
        broken = ctx.qmatmul(h, bad, n, bias=bias)
        assert not np.isfinite(broken[7]).any() and np.array_equal(broken[keep], got[keep])
        ctx.release(h)


@pytest.mark.parametrize("form", [1, 2, 4, 1 | 2 << 3])
def test_long_rows_with_the_tiles_asked_for(form):
    """A lane and the zero point's shift are up to 384 together: 384 * 128 * K passes 2^31 from K = 43691 on, so that longer rows are another kernel's whatever the
    option asks for (in 32-bit sums -128849 for 134324).  The sums are f32 then, of products of one sign, added 16 and more at a time: 45000 / 16
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
