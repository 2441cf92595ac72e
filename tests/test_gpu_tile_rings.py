"""The rings of stages of the tiled MatMul kernels where a workgroup's K range is shorter than the ring, as long, and a stage longer:
stages past the range are not requested."""
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


def weight(rng, dt, n, k):
    return fastnn_amd.quantize_weights(dt, (rng.standard_normal((n, k)) * 0.05).astype(np.float32))


# stages of 128 values: one to six, a last one that is not full; tile forms 0 to 2, K whole and in splits, one column tile and several, more than one
# round of workgroups
@pytest.mark.parametrize("dt", [flib.DT_I8, flib.DT_I4])
@pytest.mark.parametrize("m,n,k", [(m, n, k) for m, n in ((100, 130), (256, 300)) for k in (64, 128, 250, 384, 512, 640, 700, 1100)] + [(2100, 2200, 250)])
def test_i8_activations(ctx, orc, dt, m, n, k):
    """Exact sums, and the formula to 1e-6 of the largest result (a few roundings of f32)."""
    rng = np.random.default_rng(k + m)
    pw = weight(rng, dt, n, k)
    payload = orc.quantize_activations(rng.standard_normal((m, k)).astype(np.float32))
    want, want_acc = orc.qmatmul_i8act(to_oracle(orc, pw), payload, m, want_acc=True)
    h = ctx.register(pw)
    try:
        ctx.set_option(flib.OPT_FRAGMENT, -1)
        for shape in (-1, 0, 1, 2):
            for split in (0, 2, 3):
                ctx.set_option(flib.OPT_TILE_SHAPE, shape)
                ctx.set_option(flib.OPT_TILE_SPLIT, split)
                got, acc = ctx.qmatmul_i8act(h, payload, m, n, want_acc=True)
                assert np.array_equal(acc, want_acc), (shape, split)
                assert_close(got, want, 1e-6, f"shape {shape} split {split}")
    finally:
        for option, value in ((flib.OPT_FRAGMENT, 0), (flib.OPT_TILE_SHAPE, -1), (flib.OPT_TILE_SPLIT, 0)):
            ctx.set_option(option, value)
        ctx.release(h)


# 256 tiles of 128 x 128, and 240: every CU has one, and the 8-bit tiles run on three stages up to 16 of them, on four waves and four stages beyond
@pytest.mark.parametrize("m,n,k", [(2000, 2040, 100), (2000, 2040, 380), (2000, 2040, 2048), (2000, 2040, 2050), (2000, 1920, 2300)])
def test_i8_activations_on_every_cu(ctx, orc, m, n, k):
    """The sums of the first and the last rows equal the oracle's, all of them those of the four-wave tiles."""
    rng = np.random.default_rng(k + n)
    pw = weight(rng, flib.DT_I8, n, k)
    payload = np.frombuffer(orc.quantize_activations(rng.standard_normal((m, k)).astype(np.float32)), np.uint8)
    h = ctx.register(pw)
    try:
        ctx.set_option(flib.OPT_FRAGMENT, -1)
        outs = []
        for shape in (0, 1):
            ctx.set_option(flib.OPT_TILE_SHAPE, shape)
            outs.append(ctx.qmatmul_i8act(h, payload, m, n, want_acc=True))
        assert np.array_equal(outs[0][1], outs[1][1])
        assert_close(outs[0][0], outs[1][0], 1e-6, "all rows")
        for first in (0, m - 20):
            part = np.concatenate([payload[:8], payload[8 + first * k:8 + (first + 20) * k]])
            want, want_acc = orc.qmatmul_i8act(to_oracle(orc, pw), part, 20, want_acc=True)
            assert np.array_equal(outs[1][1][first:first + 20], want_acc)
            assert_close(outs[1][0][first:first + 20], want, 1e-6, f"rows {first} ..")
    finally:
        ctx.set_option(flib.OPT_FRAGMENT, 0)
        ctx.set_option(flib.OPT_TILE_SHAPE, -1)
        ctx.release(h)


# f16 tiles (stages of 64 values, rings of three to six) and digit planes (128 values, three to six)
@pytest.mark.parametrize("dt", [flib.DT_I8, flib.DT_I4, flib.DT_U4, flib.DT_F8])
@pytest.mark.parametrize("k", [60, 128, 190, 256, 384, 500, 640, 770])
def test_f32_activations(ctx, orc, dt, k):
    """2e-5 of the largest result, as for every f32-activation MatMul."""
    rng = np.random.default_rng(k + 50 * dt)
    m, n = 70, 200
    pw = weight(rng, dt, n, k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    a[m // 2] = 0.0
    want = orc.qmatmul(to_oracle(orc, pw), a, order=2)
    h = ctx.register(pw)
    try:
        ctx.set_option(flib.OPT_FRAGMENT, -1)
        for planes in ((0, 3, 4) if dt in (flib.DT_I8, flib.DT_I4, flib.DT_U4) else (0,)):
            for shape in (-1, 0, 1, 2):
                for stages in (0, 3, 5):
                    for option, value in ((flib.OPT_DIGIT_PLANES, planes), (flib.OPT_TILE_SHAPE, shape), (flib.OPT_TILE_STAGES, stages)):
                        ctx.set_option(option, value)
                    assert_close(ctx.qmatmul(h, a, n), want, 2e-5, f"planes {planes} shape {shape} stages {stages}")
    finally:
        for option, value in ((flib.OPT_FRAGMENT, 0), (flib.OPT_DIGIT_PLANES, 0), (flib.OPT_TILE_SHAPE, -1), (flib.OPT_TILE_STAGES, 0)):
            ctx.set_option(option, value)
        ctx.release(h)
