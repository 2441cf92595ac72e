"""The MatMul kernels on fragment-major operands (FNN_OPT_FRAGMENT) against the oracle, at the edges of their tiles: rows and
columns around multiples of 16, K around the k blocks (64 or 128 values), the pieces of 256 values and the eight waves."""
import ctypes as C

import numpy as np
import pytest

import fastnn_amd
from fastnn_amd import lib as flib
from gpu_common import assert_close, to_oracle

pytestmark = pytest.mark.gpu
TYPES = [flib.DT_I8, flib.DT_I4, flib.DT_U8, flib.DT_U4, flib.DT_F8, flib.DT_F8R, flib.DT_F4]
SHAPES = [(mb, nb, sp, 0) for mb, nb in ((1, 1), (1, 2), (2, 2), (2, 4), (3, 4), (4, 4)) for sp in (1, 3)] + [(1, nb, 1, 1) for nb in (1, 2, 4)]


@pytest.fixture(scope="module")
def ctx():
    with fastnn_amd.HipContext(0) as c:
        yield c


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("m,k,n", [(1, 63, 15), (16, 128, 16), (17, 1000, 33), (31, 1025, 64), (49, 2048, 130), (65, 2600, 257), (130, 515, 68)])
def test_every_shape_of_the_fragment_kernels(ctx, orc, dt, m, k, n):
    rng = np.random.default_rng(9000 + dt * 7 + m)
    pw = fastnn_amd.quantize_weights(dt, (rng.standard_normal((n, k)) * 0.05).astype(np.float32))
    a = rng.standard_normal((m, k)).astype(np.float32)
    a[:, ::61] *= 100.0
    a[m // 2] = 0.0
    bias = (rng.standard_normal(n) * 0.1).astype(np.float32)
    want = orc.qmatmul(to_oracle(orc, pw), a, order=2, bias=bias, act=flib.ACT_SILU)
    h = ctx.register(pw)
    try:
        results = []
        for mb, nb, sp, direct in [(0, 0, 0, 0)] + SHAPES:
            ctx.set_option(flib.OPT_FRAGMENT, direct << 15 | sp << 8 | nb << 4 | mb)
            got = ctx.qmatmul(h, a, n, bias=bias, act=flib.ACT_SILU)
            assert_close(got, want, 2e-5, f"{mb}x{nb} splits {sp} direct {direct}")
            if sp == 1 and (direct or mb * nb <= 4) and k <= 1024:
                results.append(got)
        for r in results[1:]:      # the same segments of K: the same bits, whoever converts the activations
            assert np.array_equal(r, results[0])
    finally:
        ctx.set_option(flib.OPT_FRAGMENT, 0)
        ctx.release(h)


@pytest.mark.parametrize("dt", [flib.DT_I8, flib.DT_I4, flib.DT_U4])
@pytest.mark.parametrize("m,k,n", [(17, 63, 15), (31, 200, 129), (33, 1000, 257), (65, 2600, 260), (130, 515, 140)])
def test_every_form_of_the_wave_tiles(ctx, orc, dt, m, k, n):
    """Rows around 32 and 64, columns around 128 and 256, K around the rings of six or eight steps of 32 and their split."""
    rng = np.random.default_rng(9100 + dt * 7 + m)
    pw = fastnn_amd.quantize_weights(dt, (rng.standard_normal((n, k)) * 0.05).astype(np.float32))
    a = rng.standard_normal((m, k)).astype(np.float32)
    a[:, ::61] *= 100.0
    a[m // 2] = 0.0
    bias = (rng.standard_normal(n) * 0.1).astype(np.float32)
    want = orc.qmatmul(to_oracle(orc, pw), a, order=2, bias=bias, act=flib.ACT_SILU)
    h = ctx.register(pw)
    try:
        for waves in (1, 2, 4):
            ctx.set_option(flib.OPT_FRAGMENT, 1 << 14 | waves)
            assert_close(ctx.qmatmul(h, a, n, bias=bias, act=flib.ACT_SILU), want, 2e-5, f"{waves} waves a tile")
    finally:
        ctx.set_option(flib.OPT_FRAGMENT, 0)
        ctx.release(h)


@pytest.mark.parametrize("dt", [flib.DT_I8, flib.DT_I4])
@pytest.mark.parametrize("m,k,n", [(1, 63, 15), (17, 1000, 33), (31, 1026, 64), (65, 2600, 257), (130, 515, 68)])
def test_every_shape_of_the_integer_fragment_kernels(ctx, orc, dt, m, k, n):
    rng = np.random.default_rng(9200 + dt * 7 + m)
    pw = fastnn_amd.quantize_weights(dt, (rng.standard_normal((n, k)) * 0.05).astype(np.float32))
    payload = orc.quantize_activations(rng.standard_normal((m, k)).astype(np.float32))
    want, want_acc = orc.qmatmul_i8act(to_oracle(orc, pw), payload, m, want_acc=True)
    h = ctx.register(pw)
    try:
        for mb, nb in ((1, 1), (1, 2), (2, 2), (2, 4), (4, 4)):
            for sp in (1, 3):
                for direct in (0, 1):
                    ctx.set_option(flib.OPT_FRAGMENT, direct << 15 | sp << 8 | nb << 4 | mb)
                    got, acc = ctx.qmatmul_i8act(h, payload, m, n, want_acc=True)
                    assert np.array_equal(acc, want_acc), f"{mb}x{nb} splits {sp} direct {direct}"
                    assert_close(got, want, 2e-5, f"{mb}x{nb} splits {sp} direct {direct}")
    finally:
        ctx.set_option(flib.OPT_FRAGMENT, 0)
        ctx.release(h)


@pytest.mark.parametrize("m,k,n", [(17, 2050, 2100), (33, 4096, 1100), (64, 2050, 2100), (95, 4096, 1100)])
def test_int8_weights_keep_four_digit_planes(ctx, m, k, n):
    """The sizes whose activations are four digit planes: exact sums, so what is left is the rounding of the recombination
    (four conversions, three multiply-adds, the scale, the K split's additions: at most 14 roundings of 2.4e-8 rms each,
    9e-8 in all).  f16 hi + lo rows with f32 sums are 1.2e-7 off and more."""
    rng = np.random.default_rng(9300 + m)
    pw = fastnn_amd.quantize_weights(flib.DT_I8, (rng.standard_normal((n, k)) * 0.05).astype(np.float32))
    pw.zeros = np.zeros(0, np.float32)
    lanes = pw.words[:n * (-(-k // 4))].view(np.int8).reshape(n, -1)[:, :k].astype(np.float64)
    h = ctx.register(pw)
    try:
        for scale in (1.0, 100.0):
            a = rng.standard_normal((m, k)).astype(np.float32)
            a[:, ::61] *= scale
            want = a.astype(np.float64) @ lanes.T * pw.scales.astype(np.float64)
            got = ctx.qmatmul(h, a, n)
            assert np.linalg.norm(got - want) <= 9e-8 * np.linalg.norm(want), (scale, np.linalg.norm(got - want) / np.linalg.norm(want))
    finally:
        ctx.release(h)


@pytest.mark.parametrize("m,k,n", [(1, 301, 40), (16, 1003, 72), (33, 1003, 72), (64, 6005, 72), (48, 2048, 64)])
def test_row_sums_of_the_fragment_kernels(ctx, m, k, n):
    """The zero-point term alone (scale 0, zero 1): every column is its row's sum.  Three levels of f32 additions per eight
    values, the sum of a piece of K and the result; with K split the sums of two halves and their sum: at most seven roundings
    of 2.4e-8 rms, 6.4e-8 of sqrt(K) times the rms of a value, and three times the 5 % by which the rms over 1000 rows scatters."""
    rng = np.random.default_rng(9400 + m)
    pw = fastnn_amd.quantize_weights(flib.DT_U8, (rng.standard_normal((n, k)) * 0.05).astype(np.float32))
    pw.scales, pw.zeros = np.zeros(n, np.float32), np.ones(n, np.float32)
    h = ctx.register(pw)
    try:
        # (named forms only: by rule the call may be another kernel's, with the sums of that kernel)
        for shape in [1 << 8 | 1 << 4 | 1, 2 << 8 | 2 << 4 | 2, 1 << 8 | 4 << 4 | 4] + ([1 << 15 | 1 << 4 | 1] if k <= 2048 else []):
            ctx.set_option(flib.OPT_FRAGMENT, shape)
            square, calls = 0.0, -(-1000 // m)
            for _ in range(calls):
                a = rng.standard_normal((m, k)).astype(np.float32)
                off = ctx.qmatmul(h, a, n)[:, 0] - a.astype(np.float64).sum(1)
                square += (off ** 2).mean() / k / calls
            assert square ** 0.5 <= 7.4e-8, (hex(shape), square ** 0.5)
    finally:
        ctx.set_option(flib.OPT_FRAGMENT, 0)
        ctx.release(h)


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("m,k,n", [(1, 63, 15), (17, 1000, 33), (33, 1025, 70), (65, 2600, 257), (40, 2048, 2112)])
def test_results_do_not_depend_on_the_copy_of_the_weight(ctx, dt, m, k, n):
    """The registered rows instead of the fragment-major copy: the same bits, for every form, K that ends inside a 64-byte block
    and rows of not-a-number next to others (the last block's words past a row are the next row's)."""
    rng = np.random.default_rng(9500 + dt * 7 + m)
    pw = fastnn_amd.quantize_weights(dt, (rng.standard_normal((n, k)) * 0.05).astype(np.float32))
    if dt == flib.DT_F8:
        pw.words[n // 2 * (-(-k // 4))] = 0x7f
    a = rng.standard_normal((m, k)).astype(np.float32)
    forms = [0, 1 << 8 | 1 << 4 | 1, 3 << 8 | 2 << 4 | 2, 1 << 8 | 4 << 4 | 4] + [1 << 15 | nb << 4 | 1 for nb in (1, 2, 4)]
    if dt in (flib.DT_I8, flib.DT_I4, flib.DT_U4):
        forms += [1 << 14 | w for w in (1, 2, 4)]
    h = ctx.register(pw)
    try:
        results = []
        for copy in (0, 2, 1, 2):   # none; none built (as without memory for one); built; the built one
            ctx.set_option(flib.OPT_GEMV_TILE_MAJOR, copy)
            for i, form in enumerate(forms):
                ctx.set_option(flib.OPT_FRAGMENT, form)
                got = ctx.qmatmul(h, a, n)
                if copy == 0:
                    results.append(got)
                else:
                    assert got.tobytes() == results[i].tobytes(), hex(form)
        if dt == flib.DT_F8:
            assert np.isnan(results[0][:, n // 2]).all() and np.isnan(results[0]).sum() == m
    finally:
        ctx.set_option(flib.OPT_FRAGMENT, 0)
        ctx.set_option(flib.OPT_GEMV_TILE_MAJOR, 1)
        ctx.release(h)


def test_a_weight_has_one_copy_beside_its_words(ctx):
    """Decode, few-row, tile and prefill kernels read the same fragment-major copy: a weight of 32 MB that has served them all
    takes 64 MB and its side tables."""
    def free():      # (the runtime that the library is linked with)
        f, t = C.c_size_t(), C.c_size_t()
        assert ctx.lib.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    n = k = 8192
    pw = fastnn_amd.quantize_weights(flib.DT_I4, np.tile(np.random.default_rng(9600).standard_normal((n, 64)).astype(np.float32) * 0.05, (1, k // 64)))
    a, out = ctx.to_device(np.ones((512, k), np.float32)), ctx.alloc(512 * n * 4)
    taken = []
    for _ in range(2):      # (the first one grows the workspaces)
        ctx.sync()
        before = free()
        h = ctx.register(pw)
        for m in (1, 8, 16, 24, 64, 512):
            ctx.qmatmul_dev(h, a.ptr, m, out.ptr)
        ctx.set_option(flib.OPT_FRAGMENT, -1)
        for m in (24, 64, 512):
            ctx.qmatmul_dev(h, a.ptr, m, out.ptr)
        ctx.set_option(flib.OPT_FRAGMENT, 0)
        ctx.sync()
        taken.append(before - free())
    assert taken[1] < 80 << 20, [t >> 20 for t in taken]


@pytest.mark.parametrize("dt,m,k,n", [(flib.DT_I8, 17, 5120, 5120), (flib.DT_U8, 23, 9984, 4416), (flib.DT_F4, 22, 11904, 4608), (flib.DT_U4, 161, 10880, 2688),
                                      (flib.DT_F8, 32, 2048, 8192), (flib.DT_I4, 64, 4096, 11008)])
def test_calls_that_the_other_kernels_do_faster_stay_with_them(ctx, dt, m, k, n):
    """Sizes at which the fragment kernels measured 1.3 to 1.7 times the time of the streaming kernel or of the LDS tiles (the last
    two 1.1 times, with weights from memory): the bits are those of the other kernel."""
    rng = np.random.default_rng(9700)
    w = np.tile((rng.standard_normal((n, 96)) * 0.05).astype(np.float32), (1, -(-k // 96)))[:, :k]
    a = rng.standard_normal((m, k)).astype(np.float32)
    h = ctx.register(fastnn_amd.quantize_weights(dt, w))
    try:
        got = ctx.qmatmul(h, a, n)
        ctx.set_option(flib.OPT_FRAGMENT, -1)
        assert np.array_equal(got, ctx.qmatmul(h, a, n))
    finally:
        ctx.set_option(flib.OPT_FRAGMENT, 0)
        ctx.release(h)


@pytest.mark.parametrize("dt", [flib.DT_I8, flib.DT_I4, flib.DT_U4])
@pytest.mark.parametrize("m,k,n", [(330, 1024, 2300), (600, 640, 5000)])
def test_wave_tiles_over_many_tiles(ctx, dt, m, k, n):
    """Tiles by the hundred, in stripes of four row tiles with a shorter last one, dealt to eight XCDs in unequal shares; rows of
    infinity and not-a-number come out as such in every column and touch no other row."""
    rng = np.random.default_rng(9800 + dt + m)
    pw = fastnn_amd.quantize_weights(dt, (rng.standard_normal((n, k)) * 0.05).astype(np.float32))
    a = rng.standard_normal((m, k)).astype(np.float32)
    h = ctx.register(pw)
    try:
        want = a.astype(np.float64) @ ctx.dequant(h, n, k).T.astype(np.float64)
        bad = a.copy()
        bad[3, k // 2], bad[m - 1, 0] = np.inf, np.nan
        good = np.setdiff1d(np.arange(m), [3, m - 1])
        for waves in (1, 2, 4):
            ctx.set_option(flib.OPT_FRAGMENT, 1 << 14 | waves)
            got = ctx.qmatmul(h, a, n)
            assert_close(got, want, 2e-5, f"{waves} waves a tile")
            off = ctx.qmatmul(h, bad, n)
            assert not np.isfinite(off[[3, m - 1]]).any() and off[good].tobytes() == got[good].tobytes()
    finally:
        ctx.set_option(flib.OPT_FRAGMENT, 0)
        ctx.release(h)


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("m,k,n", [(20, 1000, 70), (33, 512, 4000)])
def test_rows_that_are_not_finite_in_the_fragment_kernels(ctx, dt, m, k, n):
    rng = np.random.default_rng(9900 + dt + m)
    pw = fastnn_amd.quantize_weights(dt, (rng.standard_normal((n, k)) * 0.05).astype(np.float32))
    a = rng.standard_normal((m, k)).astype(np.float32)
    bad = a.copy()
    bad[3, k // 2], bad[17, k - 1], bad[m - 1, 0] = np.inf, -np.inf, np.nan
    good = np.setdiff1d(np.arange(m), [3, 17, m - 1])
    h = ctx.register(pw)
    try:
        for form in [1 << 8 | 1 << 4 | 1, 2 << 8 | 2 << 4 | 2, 1 << 8 | 4 << 4 | 3] + [1 << 15 | nb << 4 | 1 for nb in (1, 2, 4)]:
            ctx.set_option(flib.OPT_FRAGMENT, form)
            got, off = ctx.qmatmul(h, a, n), ctx.qmatmul(h, bad, n)
            assert not np.isfinite(off[[3, 17, m - 1]]).any() and off[good].tobytes() == got[good].tobytes(), hex(form)
    finally:
        ctx.set_option(flib.OPT_FRAGMENT, 0)
        ctx.release(h)
