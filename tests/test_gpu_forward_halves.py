"""A forward pass in two halves of its images (transfers of one half beside the kernels of the other) leaves the bytes that the whole
pass leaves: in the outputs, in every other value, call after call; plans that do not work image by image go whole."""
import numpy as np
import pytest

import fastnn_amd
from fastnn_amd import lib as flib
from fastnn_amd.aot import AotExecutor
from fastnn_amd.backend import ExecutablePlan, HipBackend, meta_of

pytestmark = pytest.mark.gpu


def node(op, inputs, outputs, **attributes):
    return {"name": outputs[0], "op_type": op, "inputs": "[" + ", ".join(inputs) + "]", "outputs": "[" + ", ".join(outputs) + "]",
            **{k: str(v) for k, v in attributes.items()}}


def graph(rng, size):
    """Every kind of instruction that is halved: Conv (with an Add, with a Concat behind it), Split, MaxPool, Concat, Resize, Silu, Add."""
    params = {"w1": rng.standard_normal((16, 3, 3, 3)).astype(np.float32), "b1": rng.standard_normal(16).astype(np.float32),
              "w2": rng.standard_normal((8, 8, 3, 3)).astype(np.float32) * 0.2, "w3": rng.standard_normal((8, 24, 1, 1)).astype(np.float32) * 0.2}
    nodes = [node("Conv", ["x", "w1", "b1"], ["c1"], strides=2, pads=1, group=1), node("Silu", ["c1"], ["s1"]), node("Split", ["s1"], ["l", "r"], axis=1),
             node("Conv", ["r", "w2"], ["c2"], strides=1, pads=1, group=1), node("Add", ["c2", "r"], ["a"]),
             node("MaxPool", ["a"], ["p"], kernel_shape=5, strides=1, pads=2), node("Concat", ["r", "l", "p"], ["k"], axis=1),
             node("Conv", ["k", "w3"], ["c3"], strides=1, pads=0, group=1), node("Relu", ["c3"], ["out"]),
             node("Resize", ["out"], ["up"], mode="nearest", scale_h=2, scale_w=2)]
    return nodes, params


def executor(rng, batch, size, quantize=8, outputs=("up", "out")):
    nodes, params = graph(rng, size)
    return AotExecutor(nodes, params, ["x"], list(outputs), {"x": [batch, 3, size, size]}, quantize=quantize)


@pytest.mark.parametrize("quantize", [8, 4])
@pytest.mark.parametrize("batch,size", [(2, 640), (6, 352), (16, 224)])
def test_the_same_bytes(batch, size, quantize):
    rng = np.random.default_rng(batch)
    ex = executor(np.random.default_rng(7), batch, size, quantize)
    whole = executor(np.random.default_rng(7), batch, size, quantize)
    whole.set_graph_replay(False)
    try:
        for call in range(6):     # the first two go whole, the second as a graph, the others as the graphs of their halves
            x = rng.standard_normal((batch, 3, size, size)).astype(np.float32) * (call + 1)
            got, want = ex.forward({"x": x}), whole.forward({"x": x})
            assert not whole._plan.halved and ex._plan.halved == (call > 1)
            assert ex.replayed == (call > 0)
            for name in want:
                assert got[name].tobytes() == want[name].tobytes(), (call, name)
            for name in ("l", "a", "p", "k"):
                assert ex.read_output(name).tobytes() == whole.read_output(name).tobytes(), (call, name)
            # between the passes: the whole plan on other inputs, and on these again
            if call == 3:
                y = x[::-1].copy()
                ex.write_inputs({"x": y})
                ex.dispatch()
                whole.write_inputs({"x": y})
                whole.dispatch()
                assert ex.read_output("up").tobytes() == whole.read_output("up").tobytes()
    finally:
        ex.close()
        whole.close()


def test_what_goes_whole():
    """An odd number of images, one image, floating-point weights (their kernels add in an order that depends on the batch), few bytes."""
    for batch, size, quantize in ((3, 640, 8), (1, 1024, 8), (2, 640, "f8"), (2, 64, 8)):
        ex = executor(np.random.default_rng(7), batch, size, quantize)
        x = np.random.default_rng(1).standard_normal((batch, 3, size, size)).astype(np.float32)
        first = ex.forward({"x": x})
        for _ in range(3):
            again = ex.forward({"x": x})
            assert not ex._plan.halved
            assert all(again[n].tobytes() == first[n].tobytes() for n in first)
        ex.close()


def test_results_in_memory_of_the_input():
    """The caller may have the results written over its input: that pass goes whole."""
    batch, size = 2, 640
    rng = np.random.default_rng(3)
    ex = executor(np.random.default_rng(7), batch, size, outputs=("up",))
    x = rng.standard_normal((batch, 3, size, size)).astype(np.float32)
    want = ex.forward({"x": x})["up"].copy()
    slots = [ex._values[n].slot[0] for n in ("x", "up")]
    buffer = np.empty(max(x.size, want.size), np.float32)
    for _ in range(4):
        buffer[:x.size] = x.reshape(-1)
        ex._backend.forward(ex._plan, [(slots[0], buffer[:x.size])], [(slots[1], buffer[:want.size])])
        assert not ex._plan.halved
        assert buffer[:want.size].tobytes() == want.tobytes()
    ex.close()


class TwoImages:
    """x -> Conv 1x1 -> c -> Relu -> r on two images of three channels, as a plan that goes in halves; `take` lays further slots out."""

    C, SIZE = 4, 640

    def __init__(self):
        rng = np.random.default_rng(11)
        self.top = 0
        self.pw = fastnn_amd.quantize_weights(flib.DT_I8, (rng.standard_normal((self.C, 3)) * 0.4).astype(np.float32))
        self.pw2 = fastnn_amd.quantize_weights(flib.DT_I8, (rng.standard_normal((self.C, self.C)) * 0.4).astype(np.float32))
        plane = 2 * self.SIZE * self.SIZE * 4
        self.x, self.c, self.r, self.z = (self.take(n * plane) for n in (3, self.C, self.C, self.C))
        self.w, self.w2 = self.take(self.pw.words.nbytes), self.take(self.pw2.words.nbytes)
        self.rng = rng

    def take(self, nbytes):
        off = self.top
        self.top += (nbytes + 63) // 64 * 64
        return (off, nbytes)

    def conv(self, src, channels, w, pw, dst, bias=()):
        return ("conv2d_i8", [src, w, *bias], dst, [1, 0, 1, 1, channels, self.SIZE, self.SIZE, 1, 1], meta_of(pw, [self.C, channels, 1, 1]))

    def plan(self):
        p = ExecutablePlan(self.top).write_const(self.w[0], self.pw.words).write_const(self.w2[0], self.pw2.words)
        p.call_kernel(*self.conv(self.x, 3, self.w, self.pw, self.c))
        return p.call_kernel("relu_f32", [self.c], self.r, [self.c[1] // 4])

    def input(self):
        return self.rng.standard_normal(self.x[1] // 4).astype(np.float32)

    def pass_(self, be, plan, x, outputs):
        out = [np.empty(s[1] // 4, np.float32) for s in outputs]
        be.forward(plan, [(self.x[0], x)], [(s[0], o) for s, o in zip(outputs, out)])
        return out

    def same_as_whole(self, be, plan, outputs, halved, extend=None, passes=4):
        """`passes` passes on new inputs equal those of a plan that never goes in halves; the later ones go in halves or not, as said."""
        with HipBackend(0) as other:
            other.allocate_arena(self.top)
            other.set_graph_replay(False)
            whole = self.plan()
            if extend:
                whole.call_kernel(*extend)
            for i in range(passes):
                x = self.input()
                got, want = self.pass_(be, plan, x, outputs), self.pass_(other, whole, x, outputs)
                assert all(g.tobytes() == w.tobytes() for g, w in zip(got, want)), i
            assert plan.halved == halved
            whole.close()


def test_an_instruction_added_after_halved_passes():
    """The new instruction reads the last bytes of the input as a constant (a bias): what could be halved before it no longer can."""
    t = TwoImages()
    with HipBackend(0) as be:
        be.allocate_arena(t.top)
        plan = t.plan()
        t.same_as_whole(be, plan, [t.r], halved=True)
        extend = t.conv(t.r, t.C, t.w2, t.pw2, t.z, [(t.x[0] + t.x[1] - 4 * t.C, 4 * t.C)])
        plan.call_kernel(*extend)
        t.same_as_whole(be, plan, [t.z], halved=False, extend=extend)
        plan.close()


def test_a_tensor_inside_the_input():
    """The second image is read as a tensor of its own: its first half would be read while the input's second half arrives."""
    t = TwoImages()
    second = (t.x[0] + t.x[1] // 2, t.x[1] // 2)
    s_y = t.take(second[1])
    with HipBackend(0) as be:
        be.allocate_arena(t.top)
        extend = ("relu_f32", [second], s_y, [second[1] // 4])
        plan = t.plan().call_kernel(*extend)
        t.same_as_whole(be, plan, [t.r, s_y], halved=False, extend=extend)
        plan.close()


def test_results_that_overlap():
    """Two results in overlapping memory of the caller: the later one wins, in every byte, as when the pass goes whole."""
    t = TwoImages()
    n = t.c[1] // 4
    with HipBackend(0) as be:
        be.allocate_arena(t.top)
        plan = t.plan()
        for _ in range(4):
            x = t.input()
            buffer = np.empty(n + n // 2, np.float32)
            be.forward(plan, [(t.x[0], x)], [(t.c[0], buffer[:n]), (t.r[0], buffer[n // 2:])])
            c, r = (be.read_arena(*s, np.float32) for s in (t.c, t.r))
            assert np.array_equal(buffer[:n // 2], c[:n // 2]) and np.array_equal(buffer[n // 2:], r)
        assert not plan.halved
        plan.close()


@pytest.mark.parametrize("forward", [True, False])
def test_recorded_passes_run_the_kernels_that_their_calls_choose(forward):
    """Passes on the operand kernel + GEMM pair, then one launch a convolution asked for: a pass that is recorded at once (as the halves of a
    pass are, and a plan after a change of options) has the copies of its weights all the same."""
    t = TwoImages()
    with HipBackend(0) as be:
        be.allocate_arena(t.top)
        plan = t.plan()
        run = (lambda: t.pass_(be, plan, x, [t.r])[0]) if forward else (lambda: (be.write_arena(t.x[0], x), be.dispatch(plan), be.read_arena(*t.r, np.float32))[2])
        x = t.input()
        be.set_option(flib.OPT_CONV_IMPLICIT, 2)
        want = [run() for _ in range(2)]
        assert plan.replayed and plan.one_launch_convs == 0
        be.set_option(flib.OPT_CONV_IMPLICIT, 1)
        got = [run() for _ in range(2)]
        assert plan.replayed and plan.halved == forward and plan.one_launch_convs == 1
        assert all(np.array_equal(g, want[0]) for g in want + got)
        plan.close()
