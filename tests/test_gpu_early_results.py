"""Results that leave for host memory while the rest of a forward pass runs: they are the bytes that the finished pass holds, whichever
instruction writes them last, wherever they go, pass after pass and with the results asked for changing between passes."""
import time

import numpy as np
import pytest

from fastnn_amd import lib as flib
from fastnn_amd.backend import ExecutablePlan, HipBackend

pytestmark = pytest.mark.gpu
LEAST = 512 << 10     # bytes of a result from which on it leaves early


class Chain:
    """x -> relu -> v0, v0 + x -> v1, v1 + x -> v2, ...: each value its own slot."""

    def __init__(self, values, count=10):
        self.n, self.count = values, count
        self.x = (0, values * 4)
        self.v = [((i + 1) * self.step, values * 4) for i in range(count)]
        self.arena = (count + 1) * self.step

    @property
    def step(self):
        return (self.n * 4 + 63) // 64 * 64

    def plan(self, again=None):
        p = ExecutablePlan(self.arena)
        p.call_kernel("relu_f32", [self.x], self.v[0], [self.n])
        for a, b in zip(self.v, self.v[1:]):
            p.call_kernel("add_f32", [a, self.x], b, [self.n])
        if again is not None:     # a late write into an early value
            p.call_kernel("relu_f32", [self.v[-1]], self.v[again], [self.n])
            for _ in range(6):
                p.call_kernel("add_f32", [self.v[-1], self.x], self.v[-2], [self.n])
        return p

    def expect(self, x, again=None):
        out = [np.maximum(x, 0)]
        for _ in self.v[1:]:
            out.append(out[-1] + x)
        if again is not None:
            out[again] = np.maximum(out[-1], 0)
            out[-2] = out[-1] + x
        return out


def result(kind, n):
    return flib.result_array((n,)) if kind == "pinned" else np.empty(n, np.float32)


@pytest.mark.parametrize("replay", [True, False])
@pytest.mark.parametrize("kind", ["pinned", "ordinary"])
@pytest.mark.parametrize("values", [LEAST // 4 - 4, LEAST // 4, LEAST // 4 + 1, 1 << 20])
def test_results_on_their_way(values, kind, replay):
    chain = Chain(values)
    rng = np.random.default_rng(values)
    with HipBackend(0) as be:
        be.allocate_arena(chain.arena)
        be.set_graph_replay(replay)
        for again in (None, 1):
            plan = chain.plan(again)
            for call, asked in enumerate([(1, 4, 9), (1, 4, 9), (1, 4, 9), (9, 0), (2,), (4, 1, 3, 5, 2, 8), (1, 4, 9), (3,), (1,), (0, 1, 2)]):
                x = rng.standard_normal(values).astype(np.float32)
                out = [result(kind, values) for _ in asked]
                be.forward(plan, [(chain.x[0], x)], [(chain.v[i][0], o) for i, o in zip(asked, out)])
                want = chain.expect(x, again)
                for i, o in zip(asked, out):
                    assert o.tobytes() == want[i].tobytes(), (again, call, i)
                if call == 6:       # a pass on its own between two of them
                    be.dispatch(plan)
                    assert be.read_arena(*chain.v[9], np.float32).tobytes() == want[9].tobytes()
            plan.close()


def test_results_in_the_same_pinned_memory():
    """The result named later is the one that stays, and the input may lie there as well."""
    n = 1 << 18
    chain = Chain(n)
    with HipBackend(0) as be:
        be.allocate_arena(chain.arena)
        plan = chain.plan()
        for _ in range(3):
            buffer = flib.result_array((2 * n,))
            buffer[:n] = np.random.default_rng(1).standard_normal(n).astype(np.float32)
            want = chain.expect(buffer[:n].copy())
            be.forward(plan, [(chain.x[0], buffer[:n])], [(chain.v[9][0], buffer[:n]), (chain.v[1][0], buffer[n // 2:n // 2 + n])])
            assert np.array_equal(buffer[:n // 2], want[9][:n // 2]) and np.array_equal(buffer[n // 2:n // 2 + n], want[1])
        plan.close()


def test_a_plan_that_another_backend_has_cut():
    n = 1 << 18
    chain = Chain(n)
    plan = chain.plan()
    x = np.random.default_rng(2).standard_normal(n).astype(np.float32)
    want = chain.expect(x)
    with HipBackend(0) as a, HipBackend(0) as b:
        for be in (a, b):
            be.allocate_arena(chain.arena)
        for _ in range(3):
            out = flib.result_array((n,))
            a.forward(plan, [(chain.x[0], x)], [(chain.v[1][0], out)])
            assert out.tobytes() == want[1].tobytes()
            b.write_arena(chain.x[0], x)
            b.dispatch(plan)
            assert b.read_arena(*chain.v[9], np.float32).tobytes() == want[9].tobytes()
        # ... and recorded there, where nobody has asked for a mark so far: its results leave at marks that are there all the same
        for _ in range(3):
            b.dispatch(plan)
        assert plan.replayed
        took = []
        for _ in range(6):
            out = flib.result_array((n,))
            start = time.perf_counter()
            b.forward(plan, [(chain.x[0], x)], [(chain.v[1][0], out)])
            took.append(time.perf_counter() - start)
            assert out.tobytes() == want[1].tobytes()
        assert min(took) < 3e-3, took      # (0.2 ms; a wait for a mark that never comes is many times that)
        plan.close()


@pytest.mark.parametrize("past", [4, 64, 4096])
def test_a_pinned_result_that_ends_outside_the_arena(past):
    """It begins in a tensor that leaves early and ends past the arena: refused as every such read is, nothing leaves, and the next pass is whole."""
    n = 1 << 18
    chain = Chain(n)
    end = (chain.arena, n * 4)          # the arena's last tensor, written first
    plan = ExecutablePlan(chain.arena + chain.step)
    plan.call_kernel("relu_f32", [chain.x], end, [n])
    plan.call_kernel("relu_f32", [chain.x], chain.v[0], [n])
    for a, b in zip(chain.v, chain.v[1:]):
        plan.call_kernel("add_f32", [a, chain.x], b, [n])
    x = np.random.default_rng(4).standard_normal(n).astype(np.float32)
    want = np.maximum(x, 0)
    with HipBackend(0) as be:
        be.allocate_arena(chain.arena + chain.step)
        for _ in range(4):
            whole, longer = flib.result_array((n,)), flib.result_array((n + past // 4,))
            whole[...] = longer[...] = 7.0
            with pytest.raises(flib.FnnError) as e:
                be.forward(plan, [(chain.x[0], x)], [(end[0], whole), (end[0], longer)])
            assert "outside the arena" in str(e.value)
            assert (longer == 7.0).all() and (whole == 7.0).all()
            be.forward(plan, [(chain.x[0], x)], [(end[0], whole)])
            assert whole.tobytes() == want.tobytes()
        plan.close()


@pytest.mark.parametrize("first", [1, 4, 9])
def test_results_for_ordinary_memory_beside_early_ones(first):
    """Pinned results that leave early, large ones for ordinary memory and small ones in one call, in any order."""
    n = 1 << 19
    chain = Chain(n)
    rng = np.random.default_rng(first)
    asked = [first] + [i for i in (0, 1, 2, 4, 9) if i != first]
    with HipBackend(0) as be:
        be.allocate_arena(chain.arena)
        plan = chain.plan()
        for call in range(4):
            x = rng.standard_normal(n).astype(np.float32)
            out = [result("pinned" if (i + call) % 2 else "ordinary", n) for i in asked]
            small = np.empty(100, np.float32)
            be.forward(plan, [(chain.x[0], x)], [(chain.v[i][0], o) for i, o in zip(asked, out)] + [(chain.v[3][0], small)])
            want = chain.expect(x)
            for i, o in zip(asked, out):
                assert o.tobytes() == want[i].tobytes(), (call, i)
            assert small.tobytes() == want[3][:100].tobytes()
        plan.close()


def test_a_mark_that_is_long_in_coming():
    """A pass whose first result is final after some 9 ms: the wait for it pauses (without, the processor time is the pass's; 0.65 of it measured), and the result is whole."""
    n, calls = 1 << 24, 240
    size = n * 4
    plan = ExecutablePlan(4 * size)
    plan.call_kernel("relu_f32", [(0, size)], (size, size), [n])
    for i in range(calls):
        a, b = ((1, 2) if i % 2 == 0 else (2, 1))
        plan.call_kernel("add_f32", [(a * size, size), (0, size)], (b * size, size), [n])
    plan.call_kernel("relu_f32", [(size, size)], (3 * size, size), [n])
    for _ in range(8):
        plan.call_kernel("add_f32", [(size, size), (0, size)], (2 * size, size), [n])
    x = np.random.default_rng(5).integers(0, 3, n).astype(np.float32)      # (whole numbers: the sums are exact)
    with HipBackend(0) as be:
        be.allocate_arena(4 * size)
        be.write_arena(0, x)
        share = []
        for _ in range(6):
            out = flib.result_array((n,))
            took, cpu = time.perf_counter(), time.process_time()
            be.forward(plan, [(0, x[:64])], [(3 * size, out)])
            share.append((time.process_time() - cpu) / (time.perf_counter() - took))
            assert np.array_equal(out, x * (calls + 1))
        assert min(share[2:]) < 0.9, share       # (the first ones allocate)
        plan.close()
