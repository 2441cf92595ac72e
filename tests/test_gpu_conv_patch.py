"""The quantised Conv2d from an int8 patch in LDS, in every shape its launch can take."""
import numpy as np
import pytest

import fastnn_amd
from fastnn_amd import lib as flib
from gpu_common import assert_close, to_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with fastnn_amd.HipContext(0) as c:
        yield c


# batch, channels, height, width, output channels, kernel (h, w), stride, padding, dilation, groups
GEOMETRIES = [
    (2, 3, 45, 61, 16, 3, 3, 2, 1, 1, 1),     # up to four channels; 16 output channels share a block's lanes
    (1, 4, 33, 29, 20, 7, 7, 2, 3, 1, 1),     # ... two chunks per kernel row
    (1, 2, 30, 24, 33, 5, 6, 1, 2, 2, 1),     # ... dilated, a second chunk of two columns, a block of one channel
    (2, 16, 24, 20, 16, 3, 3, 1, 1, 1, 1),    # one chunk per tap: an odd number of chunks
    (1, 17, 21, 19, 130, 3, 3, 1, 1, 1, 1),   # a chunk of one channel, five blocks of channels, no multiple of four columns
    (2, 48, 20, 20, 64, 1, 1, 1, 0, 1, 1),    # 1x1 as one row of pixels; an odd number of chunks with halves of a wave on their own
    (3, 64, 5, 5, 128, 1, 1, 1, 0, 1, 1),     # fewer pixels than a block
    (1, 36, 17, 23, 40, 3, 3, 2, 0, 1, 2),    # groups, rows and columns of the input that no tap reaches
    (2, 40, 12, 14, 96, 1, 1, 2, 0, 1, 1),    # 1x1 with a stride
    (1, 512, 9, 9, 32, 3, 3, 1, 1, 1, 1),     # K = 4608: does not fit the LDS whole
    (2, 150, 11, 13, 72, 3, 3, 1, 1, 1, 1),   # ten chunks, the last of six channels: segments of two, four and two, eight and two; an even K
    (1, 230, 9, 10, 40, 1, 5, 2, 2, 2, 1),    # fifteen chunks of five taps: the last segment is one chunk, the last step half a one
    (2, 72, 30, 31, 24, 5, 5, 1, 2, 1, 1),    # five chunks of 25 taps
]
FORMS = [0] + [128 + a + 4 * b + 16 * w + 32 * t for w in (0, 1) for a in range(4) for b in range(4) if a + b <= 2 + w for t in (0, 1, 3)]
# ... with the channels in segments of two, four and eight chunks of 16
FORMS += [f + 256 * s for f in FORMS[1:] if f >> 5 & 3 != 3 for s in (1, 2, 3)]
# ... with one, two and four blocks of output channels a wave, which fetches their weights itself
FORMS += [f + 2048 * s for f in FORMS[1:] if f < 256 and f >> 5 & 3 == 0 and (f & 3) + (f >> 2 & 3) == 2 + (f >> 4 & 1) for s in (1, 2, 3)]


@pytest.mark.parametrize("wdt", [flib.DT_I8, flib.DT_I4])
@pytest.mark.parametrize("geo", GEOMETRIES)
def test_every_shape_gives_the_same_integers_and_floats(ctx, orc, geo, wdt):
    """Accumulators equal the oracle's bit for bit, outputs within a few last places of its exp (1e-5), and the same bits for
    every shape of the launch and for the operand kernel + GEMM pair."""
    b, c, h, w, oc, kh, kw, stride, pad, dil, groups = geo
    rng = np.random.default_rng(77 + c + oc)
    kk = c // groups * kh * kw
    x = rng.uniform(-0.3, 1, (b, c, h, w)).astype(np.float32)
    x[1 % b] *= 3.0   # images with different ranges
    bias = (rng.standard_normal(oc) * 0.05).astype(np.float32)
    pw = fastnn_amd.quantize_weights(wdt, (rng.standard_normal((oc, kk)) * np.sqrt(2.0 / kk)).astype(np.float32))
    args = (kh, kw, stride, pad, dil, groups)
    want, want_acc, _, _ = orc.qconv2d_i8(x, to_oracle(orc, pw), *args, bias=bias, act=flib.ACT_SILU, want_acc=True)
    handle = ctx.register(pw)
    try:
        ctx.set_option(flib.OPT_CONV_IMPLICIT, 2)
        before = ctx.one_launch_convs
        pair, pair_acc = ctx.qconv2d(handle, x, oc, *args, bias=bias, act=flib.ACT_SILU, want_acc=True)
        assert np.array_equal(pair_acc, want_acc)
        assert ctx.one_launch_convs == before
        ctx.set_option(flib.OPT_CONV_IMPLICIT, 1)
        ran = set()
        for form in FORMS:
            ctx.set_option(flib.OPT_CONV_PATCH, form)
            before = ctx.one_launch_convs
            got, acc = ctx.qconv2d(handle, x, oc, *args, bias=bias, act=flib.ACT_SILU, want_acc=True)
            assert np.array_equal(acc, want_acc), form
            assert np.array_equal(got, pair), form
            if ctx.one_launch_convs > before:
                ran.add(form)
        # the launch ran: by rule, with K shared by waves and not (all of them over pixels and channels), four waves and eight
        segments = {f >> 8 & 7 for f in ran if f} - {0}
        assert segments == {s for s in (1, 2, 3) if -(-c // groups // 16) > 1 << s and c // groups > 4}
        assert any(f >> 11 for f in ran)
        if kk < 4000:
            shared = {f for f in ran if f and (f & 3) + (f >> 2 & 3) < 2 + (f >> 4 & 1)}
            assert 0 in ran and shared and ran - shared - {0}
            assert {f >> 4 & 1 for f in ran if f} == {0, 1}
        assert_close(pair, want, 1e-5)
    finally:
        ctx.set_option(flib.OPT_CONV_IMPLICIT, 0)
        ctx.set_option(flib.OPT_CONV_PATCH, 0)
        ctx.release(handle)


@pytest.mark.parametrize("geo", [(1, 512, 40, 40, 16, 3), (2, 320, 33, 30, 24, 5), (1, 1024, 60, 50, 40, 3), (4, 96, 100, 100, 8, 7), (8, 512, 38, 38, 512, 1)])
def test_layers_with_more_weights_than_lds_holds_run_as_one_launch(ctx, orc, geo):
    """A long K under few output channels, many channels under many pixels: by rule one launch, with the pair's bits."""
    b, c, h, w, oc, k = geo
    rng = np.random.default_rng(3 + c)
    x = rng.uniform(-0.3, 1, (b, c, h, w)).astype(np.float32)
    pw = fastnn_amd.quantize_weights(flib.DT_I8, (rng.standard_normal((oc, c * k * k)) * 0.02).astype(np.float32))
    handle = ctx.register(pw)
    before = ctx.one_launch_convs
    got, acc = ctx.qconv2d(handle, x, oc, k, k, 1, k // 2, 1, 1, act=flib.ACT_SILU, want_acc=True)
    assert ctx.one_launch_convs == before + 1
    try:
        ctx.set_option(flib.OPT_CONV_IMPLICIT, 2)
        pair, pair_acc = ctx.qconv2d(handle, x, oc, k, k, 1, k // 2, 1, 1, act=flib.ACT_SILU, want_acc=True)
    finally:
        ctx.set_option(flib.OPT_CONV_IMPLICIT, 0)
        ctx.release(handle)
    assert np.array_equal(acc, pair_acc) and np.array_equal(got, pair)


def test_a_weight_used_with_another_kernel_geometry(ctx, orc):
    """One weight as 3x3 over 4 channels, then as 1x1 over 36: its copy is in the order of the first, the second is left to the pair."""
    rng = np.random.default_rng(5)
    pw = fastnn_amd.quantize_weights(flib.DT_I8, (rng.standard_normal((24, 36)) * 0.2).astype(np.float32))
    handle = ctx.register(pw)
    ctx.set_option(flib.OPT_CONV_IMPLICIT, 1)
    for _ in range(2):
        for c, k in ((4, 3), (36, 1)):
            before = ctx.one_launch_convs
            x = rng.uniform(-1, 1, (1, c, 10, 12)).astype(np.float32)
            args = (k, k, 1, k // 2, 1, 1)
            want, want_acc, _, _ = orc.qconv2d_i8(x, to_oracle(orc, pw), *args, want_acc=True)
            got, acc = ctx.qconv2d(handle, x, 24, *args, want_acc=True)
            assert np.array_equal(acc, want_acc)
            assert_close(got, want, 1e-5)
            assert ctx.one_launch_convs - before == (1 if k == 3 else 0)
    ctx.set_option(flib.OPT_CONV_IMPLICIT, 0)
    ctx.release(handle)


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_not_a_number_and_infinities_as_in_the_pair(ctx, value):
    rng = np.random.default_rng(6)
    x = rng.uniform(-1, 1, (2, 20, 14, 12)).astype(np.float32)
    x[0, 3, 5, 7] = value
    pw = fastnn_amd.quantize_weights(flib.DT_I8, (rng.standard_normal((40, 180)) * 0.1).astype(np.float32))
    handle = ctx.register(pw)
    res = []
    try:
        for option in (1, 2):
            ctx.set_option(flib.OPT_CONV_IMPLICIT, option)
            before = ctx.one_launch_convs
            res.append(ctx.qconv2d(handle, x, 40, 3, 3, 1, 1, 1, 1, act=flib.ACT_RELU, want_acc=True))
            assert ctx.one_launch_convs - before == 2 - option
    finally:
        ctx.set_option(flib.OPT_CONV_IMPLICIT, 0)
        ctx.release(handle)
    assert np.array_equal(res[0][1], res[1][1])
    assert res[0][0].tobytes() == res[1][0].tobytes()
