"""Transfers between host arrays and the device (csrc/host_io.hip): the staging memory's edges, arrays in pinned memory as inputs,
several outputs, and calls that fail half way.  All of it moves bytes: results are compared exactly."""
import gc

import numpy as np
import pytest

import fastnn_amd
from fastnn_amd import lib as flib
from fastnn_amd.backend import ExecutablePlan, HipBackend

pytestmark = pytest.mark.gpu
SMALL = 1 << 20       # up to here a copy kernel in the stream, beyond it the copy engine


@pytest.fixture(scope="module")
def be():
    return HipBackend(0)


@pytest.fixture(scope="module")
def ctx():
    with fastnn_amd.HipContext(0) as c:
        yield c


def _bytes(rng, n):
    return rng.integers(0, 256, n, dtype=np.uint8)


def pinned(a):
    out = flib.result_array(a.shape, a.dtype)
    out[...] = a
    return out


@pytest.mark.parametrize("n", [1, 3, 15, 16, 17, 255, 4099, 32768, SMALL - 1, SMALL, SMALL + 1, SMALL + 16, (8 << 20) - 1, 8 << 20,
                               (8 << 20) + 5, (9 << 20) + 3, 33 << 20])
@pytest.mark.parametrize("offset", [0, 1, 4])
def test_every_size_and_alignment_survives_the_round_trip(ctx, n, offset):
    """Around the staging memory, the first transfer of a large input (8 MB) and its blocks of 512 KB."""
    rng = np.random.default_rng(n)
    data = _bytes(rng, n)
    buf = ctx.alloc(n + 64)
    try:
        buf.upload(np.full(n + 64, 7, np.uint8))
        buf.upload(data, offset)
        assert np.array_equal(buf.download(np.uint8, n, offset), data)
        around = buf.download(np.uint8, n + 64)
        assert (around[:offset] == 7).all() and (around[offset + n:] == 7).all()
        buf.upload(pinned(data[::-1].copy()), offset)     # from pinned memory
        host = np.empty(n, np.uint8)                      # to ordinary memory
        ctx._check(ctx.lib.fnn_hip_download(ctx.handle, host.ctypes.data, buf.ptr + offset, n))
        assert np.array_equal(host, data[::-1])
    finally:
        buf.free()


def test_staging_that_fills_up_between_two_waits(be):
    """Writes into the arena do not wait: 60 of 50 KB need the 1 MB of staging memory three times over, and every one may
    reuse its source on return."""
    rng = np.random.default_rng(1)
    n, count = 50_001, 60
    parts = [_bytes(rng, n) for _ in range(count)]
    be.allocate_arena(count * 50_048)
    for mem in (np.empty(n, np.uint8), pinned(np.zeros(n, np.uint8)), pinned(np.zeros(n + SMALL, np.uint8))[:n]):
        for i, p in enumerate(parts):
            mem[:] = p
            be.write_arena(i * 50_048, mem)
            mem[:] = 0xEE
        for i, p in enumerate(parts):
            assert np.array_equal(be.read_arena(i * 50_048, n), p), i


def test_forward_with_many_inputs_and_outputs_of_every_kind(be):
    """One call, one wait: small and large inputs and outputs, ordinary and pinned, more small ones than the staging memory holds."""
    rng = np.random.default_rng(2)
    sizes = [17, 300_000, 300_000, 300_000, 400_001, SMALL, SMALL + 16, 9 << 20, 5, 200_000]
    offsets = np.cumsum([0] + [(s + 255) // 256 * 256 for s in sizes])
    be.allocate_arena(int(offsets[-1]))
    plan = ExecutablePlan(int(offsets[-1]))
    for turn in range(4):
        data = [_bytes(rng, s) for s in sizes]
        ins = [(int(o), pinned(d) if (i + turn) % 2 else d.copy()) for i, (o, d) in enumerate(zip(offsets, data))]
        outs = [(int(o), flib.result_array(s, np.uint8) if (i + turn // 2) % 2 else np.zeros(s, np.uint8)) for i, (o, s) in enumerate(zip(offsets, sizes))]
        be.forward(plan, ins, outs)
        for (_, src), (_, got), d in zip(ins, outs, data):
            assert np.array_equal(got, d) and np.array_equal(src, d)
            src[...] = 0       # the call is over: its arrays are the caller's again
            assert np.array_equal(got, d)


def test_results_of_one_forward_are_the_inputs_of_the_next(be):
    """Pinned results as inputs, the same array as input and output, results dropped while others live."""
    rng = np.random.default_rng(3)
    n = 3 << 20
    be.allocate_arena(4 * n)
    plan = ExecutablePlan(4 * n)
    x = pinned(_bytes(rng, n))
    want = x.copy()
    kept = []
    for i in range(12):
        y = flib.result_array(n, np.uint8)
        be.forward(plan, [(i % 4 * n, x)], [(i % 4 * n, y)])
        assert np.array_equal(y, want)
        if i % 3 == 0:
            kept.append(y)
        y = flib.result_array(n, np.uint8) if i % 2 else y
        y[...] = want
        y[i] ^= 0xFF
        want[i] ^= 0xFF
        kept and i % 3 == 0 and kept.__setitem__(-1, kept[-1].copy())
        x = y
        gc.collect()
    be.forward(plan, [(0, x)], [(0, x)])
    assert np.array_equal(x, want)


@pytest.mark.parametrize("large", [False, True])
def test_a_forward_that_fails_half_way_leaves_nothing_behind(be, large):
    """The second output lies outside the arena: the call fails, writes no result afterwards, and the next one is whole."""
    rng = np.random.default_rng(4)
    n = (4 << 20) if large else 40_000
    be.allocate_arena(2 * n)
    plan = ExecutablePlan(2 * n)
    data = _bytes(rng, n)
    for mem in (lambda: np.zeros(n, np.uint8), lambda: pinned(np.zeros(n, np.uint8))):
        src, first, second = pinned(data), mem(), mem()
        with pytest.raises(flib.FnnError):
            be.forward(plan, [(0, src)], [(0, first), (2 * n - 8, second)])
        seen = first.copy()
        src[...] = 0x55
        other = _bytes(rng, n)
        got = mem()
        be.forward(plan, [(n, other)], [(n, got)])
        assert np.array_equal(got, other) and np.array_equal(first, seen) and not second.any()
        with pytest.raises(flib.FnnError):
            be.forward(plan, [(0, src), (2 * n, src)], [(0, first)])     # an input outside it
        be.forward(plan, [(0, data)], [(0, got)])
        assert np.array_equal(got, data)


def test_a_call_refused_after_its_input_was_taken(ctx):
    """FNN_FLAG_ACT_QUANT on U8 weights is refused behind the transfer of a pinned input: the array is the caller's again at once."""
    rng = np.random.default_rng(5)
    m, k, n = 700, 1024, 64
    pw = fastnn_amd.quantize_weights(flib.DT_U8, (rng.standard_normal((n, k)) * 0.05).astype(np.float32))
    h = ctx.register(pw)
    a = pinned(rng.standard_normal((m, k)).astype(np.float32))
    try:
        want = ctx.qmatmul(h, a.copy(), n)
        with pytest.raises(flib.FnnError):
            ctx.qmatmul(h, a, n, flags=flib.FLAG_ACT_QUANT)
        b = a.copy()
        a[...] = np.nan
        assert np.array_equal(ctx.qmatmul(h, b, n), want)
    finally:
        ctx.release(h)
