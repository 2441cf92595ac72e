"""Codebook MatMul of 5 to 16 rows in one launch (16 weight rows and all of K a workgroup)."""
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


def codebook_weight(rng, n, k):
    kp, bpr = -(-k // 8), -(-k // 32)
    words = rng.integers(0, 1 << 32, n * kp, dtype=np.uint32).reshape(n, kp)
    if k % 8:   # nibbles past the end of a row are zero, as the packer leaves them
        words[:, -1] &= np.uint32((1 << (4 * (k % 8))) - 1)
    scales = rng.uniform(0.01, 0.2, n * bpr).astype(np.float32)
    table = np.sort(rng.uniform(-1, 1, 16)).astype(np.float32)
    return fastnn_amd.PackedWeight(flib.DT_I4CB, n, k, np.concatenate([words.reshape(-1), np.zeros(16, np.uint32)]), scales, np.zeros(0, np.float32), 32, table)


# one k block and less, blocks of 32 that end early, one and several pieces a wave, columns that fill no block of 16
@pytest.mark.parametrize("k,n", [(31, 15), (128, 16), (300, 700), (1003, 333), (1024, 1024), (2050, 130), (4100, 257), (9000, 48)])
@pytest.mark.parametrize("m", [5, 8, 9, 16])
def test_against_the_oracle(ctx, orc, m, k, n):
    """2e-5 of the largest result, as for every f32-activation MatMul; the error against 64 bits is about 1.5e-7."""
    rng = np.random.default_rng(100 * m + k)
    pw = codebook_weight(rng, n, k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    a[:, ::61] *= 100.0
    a[m // 2] = 0.0
    bias = (rng.standard_normal(n) * 0.1).astype(np.float32)
    want = orc.qmatmul(to_oracle(orc, pw), a, order=2, bias=bias, act=flib.ACT_SILU)
    handle = ctx.register(pw)
    got = ctx.qmatmul(handle, a, n, bias=bias, act=flib.ACT_SILU)
    assert_close(got, want, 2e-5)
    # the same bits from the registered words, where the weight has no copy in fragment order
    other = ctx.register(pw)
    try:
        ctx.set_option(flib.OPT_GEMV_TILE_MAJOR, 0)
        assert ctx.qmatmul(other, a, n, bias=bias, act=flib.ACT_SILU).tobytes() == got.tobytes()
    finally:
        ctx.set_option(flib.OPT_GEMV_TILE_MAJOR, 1)
    ctx.release(handle)
    ctx.release(other)


@pytest.mark.parametrize("m", [6, 13])
def test_values_that_are_no_numbers(ctx, m):
    """An infinity or a not-a-number stays in its row (activations), its weights' columns (table), and a table entry that no weight of a
    row uses does not reach it, not even as the padding of a row that ends inside a block."""
    rng = np.random.default_rng(9)
    k, n = 205, 40
    pw = codebook_weight(rng, n, k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    handle = ctx.register(pw)
    clean = ctx.qmatmul(handle, a, n)
    bad = a.copy()
    bad[2, 17] = np.inf
    bad[4, 3] = np.nan
    got = ctx.qmatmul(handle, bad, n)
    keep = [i for i in range(m) if i not in (2, 4)]
    assert np.array_equal(got[keep], clean[keep])
    assert not np.isfinite(got[2]).any() and np.isnan(got[4]).all()
    ctx.release(handle)
    words = pw.words[:n * 26].reshape(n, 26).copy()
    words |= np.uint32(0x11111111)   # no index 0 ...
    words[:, -1] &= np.uint32((1 << (4 * (k % 8))) - 1)
    words[7, 5] &= np.uint32(0xfffffff0)   # ... but in one row
    table = pw.codebook.copy()
    table[0] = np.nan
    pn = fastnn_amd.PackedWeight(flib.DT_I4CB, n, k, np.concatenate([words.reshape(-1), np.zeros(16, np.uint32)]), pw.scales, pw.zeros, 32, table)
    handle = ctx.register(pn)
    got = ctx.qmatmul(handle, a, n)
    assert np.isnan(got[:, 7]).all() and np.isfinite(np.delete(got, 7, axis=1)).all()
    ctx.release(handle)


# K that ends anywhere in a lane's group of eight values (or four): what lies behind a row's last value is the next row's first
@pytest.mark.parametrize("k", [204, 205, 206, 207, 208, 300, 1004])
@pytest.mark.parametrize("m", [6, 13])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, -3.4e38, 1e30])
def test_the_first_values_of_a_row_do_not_reach_the_row_before(ctx, m, k, value):
    rng = np.random.default_rng(k)
    n = 40
    pw = codebook_weight(rng, n, k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    handle = ctx.register(pw)
    clean = ctx.qmatmul(handle, a, n)
    for row in (1, m - 1):
        bad = a.copy()
        bad[row, :4] = value
        got = ctx.qmatmul(handle, bad, n)
        assert np.delete(got, row, axis=0).tobytes() == np.delete(clean, row, axis=0).tobytes(), row
    ctx.release(handle)


# beside values of a normal row one of every 128 is larger, on weights that are zero: what the others are held in shows.  (shape: as FNN_OPT_STREAM_SHAPE names it; by rule
# the first four are the kernel's of 5 to 16 rows, the last one is the form for wide outputs)
@pytest.mark.parametrize("m,k,n,shape", [(5, 1003, 333, 0), (8, 1024, 1024, 0), (9, 1024, 1024, 0), (16, 1003, 333, 0), (16, 1152, 300, 0x92), (32, 1152, 300, 0x192),
                                         (48, 1152, 300, 0x91), (64, 1152, 300, 0x291), (57, 4224, 5121, 0)])
def test_small_values_beside_large_ones(ctx, m, k, n, shape):
    """Two f16 halves hold 22 bits of every value down to 2^-29 of a piece's largest: 2^-23 of each value and of each table entry, and f32 sums, 1.1e-7 to 1.6e-7 of the
    result's norm measured at any size of the large ones, 3e-7 allowed."""
    rng = np.random.default_rng(m + k)
    pw = codebook_weight(rng, n, k)
    kp, table, zero = -(-k // 8), pw.codebook.copy(), 7
    table[zero] = 0.0
    words = pw.words[:n * kp].reshape(n, kp).copy()
    large = np.arange(5, k, 128)
    for c in large:
        words[:, c // 8] = words[:, c // 8] & ~np.uint32(15 << 4 * (c % 8)) | np.uint32(zero << 4 * (c % 8))
    values = table[words[:, :, None] >> 4 * np.arange(8, dtype=np.uint32) & 15].reshape(n, -1)[:, :k].astype(np.float64)
    values *= np.repeat(pw.scales.reshape(n, -1), 32, axis=1)[:, :k]
    handle = ctx.register(fastnn_amd.PackedWeight(flib.DT_I4CB, n, k, np.concatenate([words.reshape(-1), np.zeros(16, np.uint32)]), pw.scales, pw.zeros, 32, table))
    try:
        if shape:
            ctx.set_option(flib.OPT_FRAGMENT, -1)
            ctx.set_option(flib.OPT_STREAM_SHAPE, shape)
        for value in (1.0, 2.0 ** 10, 2.0 ** 17, 2.0 ** 24, 2.0 ** 28):
            a = rng.standard_normal((m, k)).astype(np.float32)
            a[:, large] = value
            want = a.astype(np.float64) @ values.T
            got = ctx.qmatmul(handle, a, n)
            assert np.linalg.norm(got - want) < 3e-7 * np.linalg.norm(want), value
            if shape:       # (the named form has run)
                ctx.set_option(flib.OPT_STREAM_MAX_M, 0)
                assert ctx.qmatmul(handle, a, n).tobytes() != got.tobytes()
                ctx.set_option(flib.OPT_STREAM_MAX_M, 32)
    finally:
        ctx.set_option(flib.OPT_FRAGMENT, 0)
        ctx.set_option(flib.OPT_STREAM_SHAPE, 0)
        ctx.set_option(flib.OPT_STREAM_MAX_M, 32)
    ctx.release(handle)


@pytest.mark.parametrize("m,k,n", [(6, 1024, 512), (16, 1024, 512), (8, 1003, 333), (13, 1003, 333)])
def test_activations_at_the_end_of_the_range(ctx, m, k, n):
    """Results of 3e38 times weights below 0.2 are numbers, and so are those of activations of 1e-37 (2e-5 of the largest, as above)."""
    rng = np.random.default_rng(m + k)
    pw = codebook_weight(rng, n, k)
    weights = ctx.dequant(handle := ctx.register(pw), n, k).astype(np.float64)
    for value in (3e38, 1e-37):
        a = (rng.standard_normal((m, k)) * 1e-3).astype(np.float32) * np.float32(value)
        a[m - 1, 5] = value
        assert_close(ctx.qmatmul(handle, a, n), a.astype(np.float64) @ weights.T, 2e-5)
    ctx.release(handle)


# up to four rows whose K or addresses fit no 16 bytes (the last two: columns beyond 8192): one chunk of 512 and less, several, blocks of 32 that end early, eight waves' slices
@pytest.mark.parametrize("k,n", [(1, 1), (7, 3), (31, 15), (300, 700), (513, 9), (1003, 333), (2050, 130), (4100, 257), (9001, 48), (1024, 40), (512, 8200), (2080, 8200)])
@pytest.mark.parametrize("m", [1, 2, 3, 4])
def test_few_rows_of_any_length(ctx, orc, m, k, n):
    """2e-5 of the largest result; sums in 32 bits of at most 9001 / 16 products each are 5e-6 off.  K = 1024 with activations off a 16-byte line."""
    rng = np.random.default_rng(100 * m + k)
    pw = codebook_weight(rng, n, k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    a[:, ::61] *= 100.0
    bias = (rng.standard_normal(n) * 0.1).astype(np.float32)
    want = orc.qmatmul(to_oracle(orc, pw), a, order=2, bias=bias, act=flib.ACT_SILU)
    handle = ctx.register(pw)
    if k == 1024:
        x, b, out = ctx.to_device(np.concatenate([np.zeros(1, np.float32), a.reshape(-1)])), ctx.to_device(bias), ctx.alloc(m * n * 4)
        ctx.qmatmul_dev(handle, x.ptr + 4, m, out.ptr, b.ptr, act=flib.ACT_SILU)
        ctx.sync()
        got = out.download(np.float32, m * n).reshape(m, n)
    else:
        got = ctx.qmatmul(handle, a, n, bias=bias, act=flib.ACT_SILU)
    assert_close(got, want, 2e-5)
    ctx.release(handle)


def test_few_rows_that_are_no_numbers(ctx):
    """A table entry that no weight of a row uses does not reach it, not even as the padding of a row that ends inside a block."""
    rng = np.random.default_rng(10)
    k, n = 205, 40
    pw = codebook_weight(rng, n, k)
    words = pw.words[:n * 26].reshape(n, 26) | np.uint32(0x11111111)   # no index 0 ...
    words[:, -1] &= np.uint32((1 << (4 * (k % 8))) - 1)
    words[7, 5] &= np.uint32(0xfffffff0)   # ... but in one row
    table = pw.codebook.copy()
    table[0] = np.nan
    pn = fastnn_amd.PackedWeight(flib.DT_I4CB, n, k, np.concatenate([words.reshape(-1), np.zeros(16, np.uint32)]), pw.scales, pw.zeros, 32, table)
    handle = ctx.register(pn)
    for m in (1, 3, 4):
        a = rng.standard_normal((m, k)).astype(np.float32)
        a[m - 1, 9] = np.inf
        got = ctx.qmatmul(handle, a, n)
        assert np.isnan(got[:, 7]).all() and np.isfinite(np.delete(got[:m - 1], 7, axis=1)).all()
        assert not np.isfinite(got[m - 1]).any()
    ctx.release(handle)


@pytest.mark.parametrize("m", [5, 16, 17, 33, 48, 49, 64])
@pytest.mark.parametrize("k,n", [(1152, 8200), (2432, 11001), (4224, 5121)])
def test_wide_outputs(ctx, orc, m, k, n):
    """One launch of two workgroups a CU, K in whole and in ragged rounds (2e-5 of the largest result, as above)."""
    rng = np.random.default_rng(100 * m + k)
    pw = codebook_weight(rng, n, k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    a[m // 2] = 0.0
    bias = (rng.standard_normal(n) * 0.1).astype(np.float32)
    handle = ctx.register(pw)
    assert_close(ctx.qmatmul(handle, a, n, bias=bias), orc.qmatmul(to_oracle(orc, pw), a, order=2, bias=bias), 2e-5)
    ctx.release(handle)


# (splits << 8 | 128, low halves scaled | row tiles a wave << 4 | k-values of a round / 256; 0: none, the tiles take it)
@pytest.mark.parametrize("m,k,n,shape", [(16, 4224, 11008, 5 << 8 | 1 << 4 | 2), (32, 2432, 11001, 5 << 8 | 1 << 4 | 2), (48, 2432, 11001, 5 << 8 | 1 << 4 | 1),
                                         (64, 4224, 5121, 9 << 8 | 128 | 1 << 4 | 1), (33, 8448, 10368, 6 << 8 | 2 << 4 | 2), (37, 9856, 1248, 0), (60, 7296, 1664, 0)])
def test_the_form_that_wide_outputs_run_in(ctx, m, k, n, shape):
    """By rule the bits are those of the form named, and the other kernels', whose sums have another order, are 4e-5 of the largest result off at most (2e-5 each)."""
    rng = np.random.default_rng(m + k)
    pw = codebook_weight(rng, n, k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    handle = ctx.register(pw)
    got = ctx.qmatmul(handle, a, n)
    try:
        ctx.set_option(flib.OPT_FRAGMENT, -1)      # (not the kernel for 5 to 16 rows)
        ctx.set_option(flib.OPT_STREAM_SHAPE, shape)
        named = ctx.qmatmul(handle, a, n)
        ctx.set_option(flib.OPT_STREAM_MAX_M, 0)
        tiles = ctx.qmatmul(handle, a, n)
    finally:
        ctx.set_option(flib.OPT_FRAGMENT, 0)
        ctx.set_option(flib.OPT_STREAM_SHAPE, 0)
        ctx.set_option(flib.OPT_STREAM_MAX_M, 32)
    assert got.tobytes() == named.tobytes()
    assert (got.tobytes() == tiles.tobytes()) == (shape == 0)
    assert_close(got, tiles, 4e-5)
    ctx.release(handle)
