"""The work that users of this framework have it do, as measurable cases.

A case is a dict of plain values.  `prepare` makes what a user's program has in hand before the call (activations, the
packed weight or the compiled executor), `run` is one pass through the public entry points, `work` counts the bytes and
operations the pass cannot do without, and `tolerance` says how far two correct implementations may be apart.

kind      entry point                                        inputs and outputs
matmul    HipContext.qmatmul_dev                             device memory
call      HipContext.qmatmul                                 numpy arrays
i8act     fnn_hip_quantize_activations + fnn_hip_qmatmul_i8act   device memory
mlp       AotExecutor.forward, a stack of MLP blocks         numpy arrays
vision    AotExecutor.forward, a YOLOv8n-shaped graph        numpy arrays
quantise  quantize_weights_kn                                numpy arrays
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import fastnn_amd
from fastnn_amd import lib as flib
from fastnn_amd.aot import AotExecutor

DTYPES = {"i8": flib.DT_I8, "i4": flib.DT_I4, "u8": flib.DT_U8, "u4": flib.DT_U4, "f8": flib.DT_F8, "f8r": flib.DT_F8R,
          "f4": flib.DT_F4, "i4cb": flib.DT_I4CB}
BITS = {"i8": 8, "i4": 4, "u8": 8, "u4": 4, "f8": 8, "f8r": 8, "f4": 4, "i4cb": 4}
ACTS = {"none": flib.ACT_NONE, "relu": flib.ACT_RELU, "gelu": flib.ACT_GELU, "silu": flib.ACT_SILU}
# the largest listed MatMul bounds the drawn ones
MOST_MACS = 2048 * 4096 * 11008


def listed():
    return [
        # a small layer called from Python with numpy arrays, one row: all latency
        {"name": "call_i8_1024_m1", "kind": "call", "dtype": "i8", "m": 1, "k": 1024, "n": 1024, "bias": True, "act": "relu"},
        # token decode: one activation row against a feed-forward weight, bias and SiLU fused (the benchmark's default)
        {"name": "decode_i4_4096x11008_m1", "kind": "matmul", "dtype": "i4", "m": 1, "k": 4096, "n": 11008, "bias": True, "act": "silu"},
        # a small decode batch against codebook weights
        {"name": "decode_i4cb_4096_m8", "kind": "matmul", "dtype": "i4cb", "m": 8, "k": 4096, "n": 4096, "bias": False, "act": "none"},
        # sizes that fit no tile: a batch of 77 rows, K and N no multiple of anything
        {"name": "ragged_u4_1003x3333_m77", "kind": "matmul", "dtype": "u4", "m": 77, "k": 1003, "n": 3333, "bias": True, "act": "gelu"},
        # prefill of a short prompt, 8-bit weights
        {"name": "prefill_i8_4096_m256", "kind": "matmul", "dtype": "i8", "m": 256, "k": 4096, "n": 4096, "bias": False, "act": "none"},
        # prefill of a long prompt, 4-bit weights: the largest product
        {"name": "prefill_i4_4096x11008_m2048", "kind": "matmul", "dtype": "i4", "m": 2048, "k": 4096, "n": 11008, "bias": True, "act": "silu"},
        # activations quantised on the device and multiplied as integers
        {"name": "i8act_2048x8192_m512", "kind": "i8act", "dtype": "i8", "m": 512, "k": 2048, "n": 8192},
        # one token through a stack of MLP blocks, 4-bit weights
        {"name": "mlp_i4_4x2048_t1", "kind": "mlp", "dtype": "i4", "tokens": 1, "d": 2048, "f": 8192, "layers": 4},
        # 64 tokens through the same stack, FP8 weights
        {"name": "mlp_f8_4x2048_t64", "kind": "mlp", "dtype": "f8", "tokens": 64, "d": 2048, "f": 8192, "layers": 4},
        # object detection backbone and neck, one camera frame and a batch
        {"name": "vision_i8_640_b1", "kind": "vision", "dtype": "i8", "size": 640, "batch": 1},
        {"name": "vision_i8_640_b16", "kind": "vision", "dtype": "i8", "size": 640, "batch": 16},
        # a layer's weight on its way into the framework: [K, N] floats to packed words (host work)
        {"name": "quantise_i4_4096x11008", "kind": "quantise", "dtype": "i4", "k": 4096, "n": 11008},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extent(rng, lo, hi):
    """A matrix extent: most are multiples of 64, some fit nothing."""
    v = _log_int(rng, lo, hi)
    return v if rng.random() < 0.35 else max(64, v // 64 * 64)


def draw(rng):
    kind = rng.choices(("matmul", "call", "i8act", "mlp", "vision", "quantise"), (9, 2, 2, 3, 2, 2))[0]
    if kind in ("matmul", "call", "i8act"):
        while True:
            m, k, n = _log_int(rng, 1, 64 if kind == "call" else 2048), _extent(rng, 256, 8192), _extent(rng, 256, 16384)
            if m * k * n <= MOST_MACS:
                break
        if kind == "i8act":
            return {"kind": kind, "dtype": rng.choice(("i8", "i4")), "m": m, "k": k, "n": n}
        return {"kind": kind, "dtype": rng.choice(sorted(DTYPES)), "m": m, "k": k, "n": n, "bias": rng.random() < 0.5, "act": rng.choice(sorted(ACTS))}
    if kind == "mlp":
        d = _extent(rng, 256, 2048)
        return {"kind": kind, "dtype": rng.choice(("i8", "i4", "u8", "u4", "f8", "f8r", "f4")), "tokens": _log_int(rng, 1, 512), "d": d,
                "f": 4 * d, "layers": rng.randint(1, 4)}
    if kind == "vision":
        size = 32 * rng.randint(5, 20)
        return {"kind": kind, "dtype": rng.choice(("i8", "i8", "f8")), "size": size, "batch": _log_int(rng, 1, 16)}
    dt = rng.choice(sorted(DTYPES))
    hi = 1024 if dt == "i4cb" else 4096      # (the codebook is learned over all values: seconds for a large matrix)
    return {"kind": kind, "dtype": dt, "k": _extent(rng, 256, hi), "n": _extent(rng, 256, hi)}


# ---- inputs

_context = None


def context():
    """The program's one context."""
    global _context
    if _context is None:
        _context = fastnn_amd.HipContext(0)
    return _context


class Weight:
    """A packed weight registered with the context for as long as the object lives."""

    def __init__(self, packed):
        self.ctx = context()
        self.handle = self.ctx.register(packed)

    def __del__(self):
        self.ctx.release(self.handle)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(gen, *shape):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32)


def _trained_like(gen, rows, cols):
    """Weights as training leaves them: a narrow normal distribution and a few values far out."""
    w = _normal(gen, rows, cols) * 0.02
    far = torch.rand(rows, cols, generator=gen, device="cuda") < 0.001
    return torch.where(far, w * 4, w)


def _codebook_packed(w, block=32):
    """A codebook weight as a program loads it from storage: one scale for each block of 32 values along a row and a
    16-entry table over the normalised values (their 16 quantiles here: learning the table is a matter of seconds)."""
    rows, inner = w.shape
    blocks = -(-inner // block)
    padded = torch.nn.functional.pad(w, (0, blocks * block - inner)).view(rows, blocks, block)
    scales = padded.abs().amax(dim=2)
    norm = (padded / scales.clamp_min(1e-30).unsqueeze(2)).view(rows, -1)[:, :inner]
    sample = norm.reshape(-1)[: 1 << 20].sort().values
    table = sample[((torch.arange(16, device=w.device) + 0.5) / 16 * sample.numel()).long()]
    index = torch.bucketize(norm, (table[1:] + table[:-1]) / 2)
    words = -(-inner // 8)
    nibbles = torch.nn.functional.pad(index, (0, words * 8 - inner)).view(rows, words, 8)
    packed = (nibbles << (4 * torch.arange(8, device=w.device))).sum(dim=2)
    packed = torch.where(packed >= 1 << 31, packed - (1 << 32), packed).to(torch.int32).reshape(-1).cpu().numpy().view(np.uint32)
    return fastnn_amd.PackedWeight(flib.DT_I4CB, rows, inner, np.concatenate([packed, np.zeros(16, np.uint32)]),
                                   scales.reshape(-1).cpu().numpy(), np.zeros(0, np.float32), block, table.cpu().numpy())


def _packed(dtype, gen, n, k):
    w = _trained_like(gen, n, k)
    return _codebook_packed(w) if dtype == "i4cb" else fastnn_amd.quantize_weights(DTYPES[dtype], w.cpu().numpy())


def _mlp_graph(case, gen):
    """x -> x + W2 gelu(W1 x + b1) + b2, `layers` times."""
    d, f = case["d"], case["f"]
    nodes, params, x = [], {}, "x"
    for i in range(case["layers"]):
        for name, rows, cols in ((f"up{i}", d, f), (f"down{i}", f, d)):
            params[name] = (_normal(gen, rows, cols) / math.sqrt(rows)).cpu().numpy()
            params[name + "_b"] = (_normal(gen, cols) * 0.02).cpu().numpy()
        def node(op, inputs, out):
            nodes.append({"name": out, "op_type": op, "inputs": "[" + ", ".join(inputs) + "]", "outputs": f"[{out}]"})
            return out
        h = node("Gelu", [node("Add", [node("MatMul", [x, f"up{i}"], f"u{i}"), f"up{i}_b"], f"ub{i}")], f"g{i}")
        y = node("Add", [node("MatMul", [h, f"down{i}"], f"v{i}"), f"down{i}_b"], f"vb{i}")
        x = node("Add", [y, x], f"x{i}")
    return nodes, params, [x]


def _conv_layers():
    """The vision graph's convolutions: (input channels, input size as a fraction of the image, output channels, kernel, stride)."""
    layers = []

    def conv(c, down, oc, k, s):
        layers.append((c, down, oc, k, s))

    def c2f(c1, c2, n, down):
        conv(c1, down, c2, 1, 1)
        for _ in range(2 * n):
            conv(c2 // 2, down, c2 // 2, 3, 1)
        conv((2 + n) * c2 // 2, down, c2, 1, 1)

    conv(3, 1, 16, 3, 2), conv(16, 2, 32, 3, 2), c2f(32, 32, 1, 4)
    conv(32, 4, 64, 3, 2), c2f(64, 64, 2, 8)
    conv(64, 8, 128, 3, 2), c2f(128, 128, 2, 16)
    conv(128, 16, 256, 3, 2), c2f(256, 256, 1, 32)
    conv(256, 32, 128, 1, 1), conv(512, 32, 256, 1, 1)
    c2f(384, 128, 1, 16), c2f(192, 64, 1, 8)
    conv(64, 8, 64, 3, 2), c2f(192, 128, 1, 16)
    conv(128, 16, 128, 3, 2), c2f(384, 256, 1, 32)
    return layers


def _vision_graph(gen):
    """Backbone and neck of a YOLOv8n-shaped detector (Conv + SiLU, C2f blocks, a pooling pyramid, nearest resizes)."""
    nodes, params, count = [], {}, [0]

    def node(op, inputs, outputs=1, **attributes):
        names = []
        for _ in range(outputs):
            count[0] += 1
            names.append(f"v{count[0]}")
        nodes.append({"name": names[0], "op_type": op, "inputs": "[" + ", ".join(inputs) + "]", "outputs": "[" + ", ".join(names) + "]",
                      **{k: str(v) for k, v in attributes.items()}})
        return names if outputs > 1 else names[0]

    def conv(x, c, oc, k, s):
        w = f"w{len(params)}"
        params[w] = (_normal(gen, oc, c, k, k) * math.sqrt(2.0 / (c * k * k))).cpu().numpy()
        params[w + "_b"] = (_normal(gen, oc) * 0.05).cpu().numpy()
        return node("Silu", [node("Conv", [x, w, w + "_b"], strides=s, pads=k // 2, group=1)])

    def c2f(x, c1, c2, n, shortcut):
        parts = list(node("Split", [conv(x, c1, c2, 1, 1)], outputs=2, axis=1))
        for _ in range(n):
            y = conv(conv(parts[-1], c2 // 2, c2 // 2, 3, 1), c2 // 2, c2 // 2, 3, 1)
            parts.append(node("Add", [parts[-1], y]) if shortcut else y)
        return conv(node("Concat", parts, axis=1), (2 + n) * c2 // 2, c2, 1, 1)

    def up(x):
        return node("Resize", [x], mode="nearest", scale_h=2, scale_w=2)

    x = c2f(conv(conv("x", 3, 16, 3, 2), 16, 32, 3, 2), 32, 32, 1, True)
    p3 = c2f(conv(x, 32, 64, 3, 2), 64, 64, 2, True)
    p4 = c2f(conv(p3, 64, 128, 3, 2), 128, 128, 2, True)
    x = c2f(conv(p4, 128, 256, 3, 2), 256, 256, 1, True)
    pools = [conv(x, 256, 128, 1, 1)]
    for _ in range(3):
        pools.append(node("MaxPool", [pools[-1]], kernel_shape=5, strides=1, pads=2))
    p5 = conv(node("Concat", pools, axis=1), 512, 256, 1, 1)
    n4 = c2f(node("Concat", [up(p5), p4], axis=1), 384, 128, 1, False)
    n3 = c2f(node("Concat", [up(n4), p3], axis=1), 192, 64, 1, False)
    m4 = c2f(node("Concat", [conv(n3, 64, 64, 3, 2), n4], axis=1), 192, 128, 1, False)
    n5 = c2f(node("Concat", [conv(m4, 128, 128, 3, 2), p5], axis=1), 384, 256, 1, False)
    return nodes, params, [n3, m4, n5]


def _executor(case, graph, shape):
    nodes, params, outputs = graph
    quantize = {"i8": 8, "i4": 4}.get(case["dtype"], case["dtype"])
    return AotExecutor(nodes, params, ["x"], outputs, {"x": shape}, quantize=quantize)


def prepare(case, seed):
    gen, kind = _generator(seed), case["kind"]
    if kind in ("mlp", "vision"):
        if kind == "mlp":
            shape = [case["tokens"], case["d"]]
            graph = _mlp_graph(case, gen)
            x = _normal(gen, *shape).cpu().numpy()
        else:
            shape = [case["batch"], 3, case["size"], case["size"]]
            graph = _vision_graph(gen)
            x = torch.rand(*shape, generator=gen, device="cuda").cpu().numpy()
        return {"kind": kind, "executor": _executor(case, graph, shape), "x": x}
    if kind == "quantise":
        return {"kind": kind, "dtype": DTYPES[case["dtype"]], "w": _trained_like(gen, case["k"], case["n"]).cpu().numpy()}
    m, k, n = case["m"], case["k"], case["n"]
    state = {"kind": kind, "ctx": context(), "weight": Weight(_packed(case["dtype"], gen, n, k)), "m": m, "k": k, "n": n}
    x = _normal(gen, m, k)
    if kind == "i8act":
        state.update(x=x, payload=torch.zeros(8 + m * k + 16, dtype=torch.uint8, device="cuda"), out=torch.empty(m, n, device="cuda"))
        torch.cuda.synchronize()      # (the context has a stream of its own)
        return state
    bias = _normal(gen, n) * 0.01 if case["bias"] else None
    state["act"] = ACTS[case["act"]]
    if kind == "call":
        state.update(x=x.cpu().numpy(), bias=None if bias is None else bias.cpu().numpy())
        return state
    state.update(x=x, bias=bias, out=torch.empty(m, n, device="cuda"))
    torch.cuda.synchronize()
    return state


def run(state):
    kind = state["kind"]
    if kind == "matmul":
        bias = state["bias"]
        state["ctx"].qmatmul_dev(state["weight"].handle, state["x"].data_ptr(), state["m"], state["out"].data_ptr(),
                                 0 if bias is None else bias.data_ptr(), state["act"])
        return state["out"]
    if kind == "call":
        return state["ctx"].qmatmul(state["weight"].handle, state["x"], state["n"], state["bias"], state["act"])
    if kind in ("mlp", "vision"):
        return state["executor"].forward({"x": state["x"]})
    if kind == "quantise":
        packed = fastnn_amd.quantize_weights_kn(state["dtype"], state["w"])
        return [packed.words.view(np.int32), packed.scales, packed.zeros] + ([] if packed.codebook is None else [packed.codebook])
    ctx, lib, vp = state["ctx"], state["ctx"].lib, C.c_void_p
    x, payload, out, m, k = state["x"], state["payload"], state["out"], state["m"], state["k"]
    rc = lib.fnn_hip_quantize_activations(ctx.handle, vp(x.data_ptr()), m * k, 0.0, 0.0, vp(payload.data_ptr()), flib.FLAG_DEVICE_PTRS)
    rc = rc or lib.fnn_hip_qmatmul_i8act(ctx.handle, state["weight"].handle, vp(payload.data_ptr()), m, vp(out.data_ptr()), None, flib.FLAG_DEVICE_PTRS)
    if rc:
        raise flib.FnnError(rc, lib.fnn_hip_last_error(ctx.handle).decode())
    return [payload, out]


def _weight_bytes(dtype, n, k):
    if dtype == "i4cb":
        return n * k // 2 + 4 * n * -(-k // 32) + 64
    return n * k * BITS[dtype] // 8 + (4 if dtype in ("f8", "f8r") else 8) * n


def work(case):
    kind, dt = case["kind"], case["dtype"]
    if kind == "mlp":
        t, d, f, layers = case["tokens"], case["d"], case["f"], case["layers"]
        weights = layers * (_weight_bytes(dt, f, d) + _weight_bytes(dt, d, f) + 4 * (d + f))
        return {"bytes": weights + 2 * 4 * t * d, "flops": 4 * t * d * f * layers}
    if kind == "vision":
        b, size = case["batch"], case["size"]
        flops, weights = 0, 0
        for c, down, oc, k, s in _conv_layers():
            flops += 2 * b * (size // down // s) ** 2 * c * k * k * oc
            weights += _weight_bytes(dt, oc, c * k * k) + 4 * oc
        pixels = size * size
        outputs = pixels // 64 * 64 + pixels // 256 * 128 + pixels // 1024 * 256
        return {"bytes": weights + 4 * b * (3 * pixels + outputs), "flops": flops}
    k, n = case["k"], case["n"]
    if kind == "quantise":
        return {"bytes": 4 * k * n + _weight_bytes(dt, n, k), "flops": 0}
    m = case["m"]
    side = 5 * m * k if kind == "i8act" else 4 * m * k + (4 * n if case["bias"] else 0)
    return {"bytes": _weight_bytes(dt, n, k) + side + 4 * m * n, "flops": 2 * m * k * n}


def tolerance(case):
    kind = case["kind"]
    if kind == "quantise":
        return "exact"
    if kind == "vision":
        # 8-bit convolutions round the activations of every layer to 256 levels: a last-bit difference moves a value to the
        # next level now and then, and through the layers behind it; the others accumulate in f32
        return {"rel": 2e-2} if case["dtype"] == "i8" else {"rel": 1e-4}
    return {"rel": 3e-5 if kind == "mlp" else 1e-5}
