"""The f32 Conv2d of more than 2048 output pixels, whose f16 operand comes straight from the image, against im2col rows and their preparation."""
import ctypes as C

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


# batch, channels, height, width, output channels, kernel (h, w), stride, padding, dilation
GEOMETRIES = [
    # 64 pixels a workgroup
    (1, 3, 64, 33, 16, 3, 3, 1, 1, 1),      # one k block, part of it padding; 2112 pixels end on no tile
    (2, 17, 66, 71, 20, 3, 3, 2, 1, 1),     # 153 values; blocks of pixels that span two images
    (3, 32, 29, 31, 130, 1, 1, 1, 0, 1),    # 1x1
    (1, 6, 61, 57, 33, 5, 2, 1, 3, 2),      # dilated, a kernel that is not square, more padding than it reaches
    (3, 8, 97, 95, 40, 2, 3, 3, 0, 1),      # rows and columns that no tap reaches
    (1, 72, 259, 257, 8, 3, 3, 1, 1, 1),    # more than 65536 pixels, 11 k blocks: two of them read twice
    # 16 pixels
    (1, 64, 50, 47, 48, 3, 3, 1, 1, 1),     # nine k blocks in three steps
    (2, 90, 40, 41, 24, 3, 3, 1, 1, 1),     # 810 values in four
    (1, 40, 46, 47, 20, 8, 8, 1, 3, 1),     # 2560 values: a step of four k blocks read twice
    (3, 230, 33, 31, 16, 1, 1, 1, 0, 1),    # 1x1, one step
]


def both(ctx, handle, x, oc, args, **kw):
    got = ctx.qconv2d(handle, x, oc, *args, 1, **kw)
    ctx.set_option(flib.OPT_FRAGMENT, 1)    # (no tile of the fragment kernels: the call runs on im2col rows)
    try:
        return got, ctx.qconv2d(handle, x, oc, *args, 1, **kw)
    finally:
        ctx.set_option(flib.OPT_FRAGMENT, 0)


@pytest.mark.parametrize("wdt", [flib.DT_U8, flib.DT_F8, flib.DT_F8R, flib.DT_F4, flib.DT_I4CB])
@pytest.mark.parametrize("geo", GEOMETRIES)
def test_operand_from_the_image_equals_prepared_rows(ctx, orc, geo, wdt):
    """The operand's halves are the same bits, so is every product; a row sum, which zero points (U8, FP4) multiply, may differ in its
    last place (f32 of a double against f32 sums: 1e-6 of the sum of magnitudes, as the stated 2e-5 against the oracle)."""
    b, c, h, w, oc, kh, kw, stride, pad, dil = geo
    rng = np.random.default_rng(5 + c + oc)
    kk = c * kh * kw
    x = rng.uniform(-0.3, 1, (b, c, h, w)).astype(np.float32)
    bias = (rng.standard_normal(oc) * 0.05).astype(np.float32)
    pw = fastnn_amd.quantize_weights(wdt, (rng.standard_normal((oc, kk)) * np.sqrt(2.0 / kk)).astype(np.float32))
    args = (kh, kw, stride, pad, dil)
    want = orc.qconv2d_float(x, to_oracle(orc, pw), *args, 1, bias=bias, act=flib.ACT_SILU)
    assert b * want.shape[2] * want.shape[3] > 2048
    handle = ctx.register(pw)
    got, rows = both(ctx, handle, x, oc, args, bias=bias, act=flib.ACT_SILU)
    assert_close(got, want, 2e-5)
    if wdt in (flib.DT_U8, flib.DT_F4):
        assert_close(got, rows, 2e-6)
    else:
        assert np.array_equal(got, rows)
    single, rows = both(ctx, handle, x, oc, args, bias=bias, act=flib.ACT_SILU, flags=flib.FLAG_ACT_F16_SINGLE)
    assert_close(single, rows, 2e-6)


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_not_a_number_and_infinities_as_in_the_rows(ctx, value):
    rng = np.random.default_rng(9)
    x = rng.standard_normal((1, 16, 50, 48)).astype(np.float32)
    x[0, 3, 20, 21] = value
    handle = ctx.register(fastnn_amd.quantize_weights(flib.DT_F8, rng.standard_normal((24, 144)).astype(np.float32)))
    got, rows = both(ctx, handle, x, 24, (3, 3, 1, 1, 1))
    assert np.array_equal(got, rows, equal_nan=True)


def test_no_room_for_rows_of_results_that_go_straight_to_the_image():
    """1 -> 128 channels over 512 x 512 pixels: the operand is 64 values of two halves a pixel (64 MiB), the result 128 MiB in the caller's memory."""
    def free():
        bytes_free, total = C.c_size_t(), C.c_size_t()
        assert c.lib.hipMemGetInfo(C.byref(bytes_free), C.byref(total)) == 0
        return bytes_free.value

    with fastnn_amd.HipContext(0) as c:
        handle = c.register(fastnn_amd.quantize_weights(flib.DT_F8, np.ones((128, 9), np.float32)))
        x, y = c.to_device(np.ones((512, 512), np.float32)), c.alloc(128 * 512 * 512 * 4)
        c.sync()
        before = free()
        rc = c.lib.fnn_hip_qconv2d(c.handle, handle, x.ptr, 1, 1, 512, 512, 3, 3, 1, 1, 1, 1, None, flib.ACT_NONE, y.ptr, None, flib.FLAG_DEVICE_PTRS)
        c.sync()
        assert rc == 0 and before - free() < 100 << 20
        got = y.download(np.float32, 128 * 512 * 512).reshape(128, 512, 512)
        assert (got[:, 1:-1, 1:-1] == 9).all() and (got[:, 0, 0] == 4).all()
        c.release(handle)
