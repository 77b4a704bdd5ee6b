"""Performance cases: the work that programs have the backend do, one pass each
through the public entry points (Device, DeviceProgram), with the inputs, the
compiled graph and the re-laid weights that such a program keeps at hand.

listed() names twelve cases, from an 8 us MLP forward to a 137 GFLOP product;
draw() gives more of the same kinds, over the sizes and options each kind is
used with, odd ones among them.  exact() is the same result from plain torch in
64 bits.
"""
import math
import weakref

import numpy as np
import torch
import torch.nn.functional as F

from lancius_amd import (ACT_GELU, ACT_NONE, ACT_RELU, DEVICE_GRAPH, Device, DeviceProgram, abi, graph_lib, graphs)

MOST_FLOPS = 2.0 * 4096 ** 3  # a drawn case does no more than the largest listed one
ACTS = {"none": ACT_NONE, "relu": ACT_RELU, "gelu": ACT_GELU}

_device = None


def device():
    """One context on GPU 0's null stream, torch's default stream too."""
    global _device
    if _device is None:
        _device = Device(0)
    return _device


# ---- the cases ----------------------------------------------------------------


def listed():
    return [
        # one small classifier request batch: the MNIST example's forward graph, launch latency
        {"name": "mlp_forward", "kind": "mlp_forward", "batch": 64, "d_in": 784, "hidden": 256, "classes": 10},
        # one step of the MNIST training example: loss and every gradient, a dozen small launches
        {"name": "mlp_train", "kind": "mlp_train", "batch": 64, "d_in": 784, "hidden": 128, "classes": 10,
         "recorded": False},
        # one step of the CIFAR-10 training example: small convolutions, pooling, their gradients
        {"name": "cnn_train", "kind": "cnn_train", "batch": 32, "recorded": False},
        # a whole transformer encoder block over four sequences, as one graph
        {"name": "block_forward", "kind": "block", "batch": 4, "S": 1024, "d": 1024, "H": 16, "F": 4096},
        # a linear layer over a ragged batch of tokens, no size a multiple of a tile
        {"name": "linear_ragged", "kind": "linear", "M": 1537, "K": 1000, "N": 2999, "bias": True, "act": "gelu",
         "residual": False},
        # the large square product of the benchmark
        {"name": "linear_large", "kind": "linear", "M": 4096, "K": 4096, "N": 4096, "bias": False, "act": "none",
         "residual": False},
        # that layer's backward pass: dX = dY W^T, dW = X^T dY, db
        {"name": "linear_backward", "kind": "linear_backward", "M": 2048, "K": 1024, "N": 4096},
        # prefill of a grouped-query layer with a history of keys, ragged lengths
        {"name": "attention_prefill", "kind": "attention", "batch": 3, "S_q": 700, "S_kv": 1500, "H_q": 32,
         "H_kv": 8, "D": 128, "causal": True},
        # one decode step of a serving batch whose sequences differ in length
        {"name": "attention_decode", "kind": "decode", "batch": 16, "S_kv": 4096, "H_q": 32, "H_kv": 8, "D": 128},
        # a mid-network 3x3 convolution with bias and ReLU, its filter packed once
        {"name": "conv_forward", "kind": "conv", "batch": 32, "C_in": 64, "H": 56, "W": 56, "C_out": 128, "k": 3,
         "stride": 1, "act": "relu", "packed": True},
        # the two gradients of that convolution
        {"name": "conv_backward", "kind": "conv_backward", "batch": 32, "C_in": 64, "H": 56, "W": 56, "C_out": 128,
         "k": 3, "stride": 1},
        # a quantized linear layer: the activation quantized in the call, the int8 weight packed once
        {"name": "int8_linear", "kind": "int8_linear", "M": 4096, "K": 4096, "N": 4096, "bias": True, "act": "none"},
    ]


def _log(rng, lo, hi, step=1):
    """A size from lo to hi, spread over its logarithm; a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step, int(round(v / step)) * step)


def _size(rng, lo, hi):
    """A matrix size: half of them multiples of 64 as models have them, half of any value."""
    return _log(rng, max(lo, 64), hi, 64) if rng.random() < 0.5 else _log(rng, lo, hi)


def _draw_kind(rng, kind):
    if kind == "mlp_forward":
        return {"batch": _log(rng, 1, 256), "d_in": _log(rng, 32, 2048), "hidden": _log(rng, 16, 512),
                "classes": _log(rng, 2, 100)}
    if kind == "mlp_train":
        return {"batch": _log(rng, 8, 512), "d_in": _log(rng, 32, 2048), "hidden": _log(rng, 16, 512),
                "classes": _log(rng, 2, 100), "recorded": rng.random() < 0.5}
    if kind == "cnn_train":
        return {"batch": _log(rng, 1, 128), "recorded": rng.random() < 0.5}
    if kind == "block":
        h, hd = rng.choice([4, 8, 12, 16]), rng.choice([32, 64, 128])
        return {"batch": rng.randint(1, 6), "S": _log(rng, 33, 1024), "d": h * hd, "H": h, "F": 4 * h * hd}
    if kind == "linear":
        return {"M": _size(rng, 1, 8192), "K": _size(rng, 48, 8192), "N": _size(rng, 10, 8192),
                "bias": rng.random() < 0.7, "act": rng.choice(["none", "none", "relu", "gelu"]),
                "residual": rng.random() < 0.3}
    if kind == "linear_backward":
        return {"M": _size(rng, 16, 8192), "K": _size(rng, 48, 4096), "N": _size(rng, 10, 4096)}
    if kind == "attention":
        h_kv = rng.choice([2, 4, 8, 16])
        s_q = _log(rng, 16, 2048)
        return {"batch": _log(rng, 1, 8), "S_q": s_q, "S_kv": s_q + rng.choice([0, 0, _log(rng, 1, 1024)]),
                "H_q": h_kv * rng.choice([1, 1, 2, 4]), "H_kv": h_kv, "D": rng.choice([32, 64, 64, 96, 128]),
                "causal": rng.random() < 0.7}
    if kind == "decode":
        h_kv = rng.choice([2, 4, 8, 16])
        return {"batch": _log(rng, 1, 64), "S_kv": _log(rng, 64, 8192), "H_q": h_kv * rng.choice([1, 2, 4, 8]),
                "H_kv": h_kv, "D": rng.choice([64, 96, 128])}
    if kind in ("conv", "conv_backward"):
        k = rng.choice([1, 3, 3, 5, 7])
        aligned = rng.random() < 0.7
        case = {"batch": _log(rng, 1, 32), "C_in": _log(rng, 16, 256, 16) if aligned else _log(rng, 3, 64),
                "H": _log(rng, 7, 112), "W": _log(rng, 7, 112),
                "C_out": _log(rng, 16, 256, 16) if aligned else _log(rng, 6, 256), "k": k,
                "stride": rng.choice([1, 1, 2])}
        if kind == "conv":
            case.update(act=rng.choice(["none", "relu"]), packed=aligned and rng.random() < 0.7)
        return case
    return {"M": _size(rng, 1, 8192), "K": _size(rng, 48, 8192), "N": _size(rng, 10, 8192),
            "bias": rng.random() < 0.7, "act": rng.choice(["none", "relu", "gelu"])}


def draw(rng):
    while True:
        kind = rng.choice(listed())["kind"]
        case = {"kind": kind, **_draw_kind(rng, kind)}
        w = work(case)
        # memory-bound kinds are held to the bytes of the largest decode step as well
        if w["flops"] <= MOST_FLOPS and w["bytes"] <= 600e6:
            return case


# ---- what a program has in hand ------------------------------------------------


class _Memory:
    """A device address as an array that torch can view without a copy; the
    view keeps the owner of the memory alive."""

    def __init__(self, ptr, shape, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (int(ptr), False),
                                         "version": 2, "strides": None}


class _Program:
    """A compiled graph with its inputs uploaded, closed with the last reference to it."""

    def __init__(self, bg, feeds, flags=0):
        lib = graph_lib()
        lib.lancius_graph_set_dtype(bg.g, abi.DTYPE_FP32)
        sched = lib.lancius_ir_schedule(bg.g)
        plan = lib.lancius_build_memory_plan(sched, bg.g)
        self.prog = DeviceProgram(device(), bg.g, sched, plan, flags)
        for name in bg.inputs:
            self.prog.upload(bg.node(name), feeds[name])
        sinks = [(name, self.prog.buffer(bg.node(name)), abi.node_shape(bg.node(name))) for name in bg.outputs]
        lib.lancius_memory_plan_destroy(plan)
        lib.lancius_schedule_destroy(sched)
        bg.destroy()
        weakref.finalize(self, DeviceProgram.close, self.prog)
        self.sinks = sinks

    def outputs(self):
        return {name: torch.as_tensor(_Memory(ptr, shape, self), device="cuda") for name, ptr, shape in self.sinks}


def _graph_state(case, bg, feeds, flags=0):
    program = _Program(bg, feeds, flags)
    return {"case": case, "program": program.prog, "out": program.outputs()}


def _host(seed):
    return np.random.Generator(np.random.PCG64(seed))


def _cuda(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * std


def _int8(g, *shape):
    """Quantized weights: N(0, 1) values on the symmetric grid of their largest magnitude."""
    w = torch.randn(*shape, generator=g, device="cuda")
    return torch.round(w * (127.0 / w.abs().max())).to(torch.int8)


def _mlp_feeds(c, seed):
    r = _host(seed)
    b, k, h, n = c["batch"], c["d_in"], c["hidden"], c["classes"]
    feeds = {"W1": r.standard_normal((k, h), np.float32) * np.float32(math.sqrt(2.0 / k)),
             "b1": r.standard_normal((1, h), np.float32) * np.float32(0.05),
             "W2": r.standard_normal((h, n), np.float32) * np.float32(math.sqrt(2.0 / h)),
             "b2": r.standard_normal((1, n), np.float32) * np.float32(0.05)}
    x = r.standard_normal((b, k), np.float32)
    y = np.zeros((b, n), np.float32)
    y[np.arange(b), r.integers(0, n, b)] = 1.0
    if c["kind"] == "mlp_forward":
        return {"x": x, **feeds}
    return {"X": x, "Y": y, **feeds}


def _cnn_feeds(c, seed):
    r = _host(seed)

    def layer(fan_in, *shape):
        return r.standard_normal(shape, np.float32) * np.float32(math.sqrt(2.0 / fan_in))

    b = c["batch"]
    y = np.zeros((b, 10), np.float32)
    y[np.arange(b), r.integers(0, 10, b)] = 1.0
    return {"X": r.standard_normal((b, 3, 32, 32), np.float32), "W1": layer(75, 16, 3, 5, 5),
            "W2": layer(400, 32, 16, 5, 5), "W3": layer(2048, 2048, 120), "b1": 0.05 * layer(2, 1, 120),
            "W4": layer(120, 120, 10), "b2": 0.05 * layer(2, 1, 10), "Y": y}


def _block_feeds(c, seed):
    r = _host(seed)
    d, f = c["d"], c["F"]

    def matrix(rows, cols):
        return r.standard_normal((rows, cols), np.float32) * np.float32(1.0 / math.sqrt(rows))

    def vector(n, mean=0.0):
        return r.standard_normal((1, n), np.float32) * np.float32(0.05) + np.float32(mean)

    feeds = {"g1": vector(d, 1.0), "be1": vector(d), "Wq": matrix(d, d), "bq": vector(d), "Wk": matrix(d, d),
             "bk": vector(d), "Wv": matrix(d, d), "bv": vector(d), "Wo": matrix(d, d), "bo": vector(d),
             "g2": vector(d, 1.0), "be2": vector(d), "W1": matrix(d, f), "bf1": vector(f), "W2": matrix(f, d),
             "bf2": vector(d)}
    for s in range(c["batch"]):
        feeds[f"x{s}"] = r.standard_normal((c["S"], d), np.float32)
    return feeds


def _linear_inputs(c, seed):
    g = _cuda(seed)
    M, K, N = c["M"], c["K"], c["N"]
    s = {"x": _normal(g, M, K)}
    if c["kind"] == "int8_linear":
        s["w"] = _int8(g, K, N)
        s["scale"] = 4.5 / (127.0 * math.sqrt(K))
    else:
        s["w"] = _normal(g, K, N, std=1.0 / math.sqrt(K))
    if c["kind"] == "linear_backward":
        s["dy"] = _normal(g, M, N, std=0.01)
        return s
    s["bias"] = _normal(g, N, std=0.1) if c["bias"] else None
    s["residual"] = _normal(g, M, N) if c.get("residual") else None
    return s


def _attention_inputs(c, seed):
    g = _cuda(seed)
    b, d = c["batch"], c["D"]
    if c["kind"] == "decode":
        lens = torch.randint(max(1, c["S_kv"] // 4), c["S_kv"] + 1, (b,), generator=g, device="cuda",
                             dtype=torch.int32)
        return {"q": _normal(g, b, c["H_q"], d), "k": _normal(g, b, c["S_kv"], c["H_kv"], d),
                "v": _normal(g, b, c["S_kv"], c["H_kv"], d), "lens": lens}
    return {"q": _normal(g, b, c["S_q"], c["H_q"], d), "k": _normal(g, b, c["S_kv"], c["H_kv"], d),
            "v": _normal(g, b, c["S_kv"], c["H_kv"], d)}


def _conv_out(c):
    p = c["k"] // 2
    return (c["H"] + 2 * p - c["k"]) // c["stride"] + 1, (c["W"] + 2 * p - c["k"]) // c["stride"] + 1


def _conv_inputs(c, seed):
    g = _cuda(seed)
    fan_in = c["C_in"] * c["k"] ** 2
    s = {"x": _normal(g, c["batch"], c["C_in"], c["H"], c["W"]),
         "w": _normal(g, c["C_out"], c["C_in"], c["k"], c["k"], std=math.sqrt(2.0 / fan_in))}
    if c["kind"] == "conv":
        s["bias"] = _normal(g, c["C_out"], std=0.1)
    else:
        s["dy"] = _normal(g, c["batch"], c["C_out"], *_conv_out(c), std=0.01)
    return s


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "mlp_forward":
        bg = graphs.build_mlp(graph_lib(), c["batch"], c["d_in"], c["hidden"], c["classes"])
        return _graph_state(c, bg, _mlp_feeds(c, seed))
    if kind in ("mlp_train", "cnn_train"):
        lib = graph_lib()
        if kind == "mlp_train":
            fwd, feeds = graphs.build_mlp_ce(lib, c["batch"], c["d_in"], c["hidden"], c["classes"]), _mlp_feeds(c, seed)
        else:
            fwd, feeds = graphs.build_cnn_ce(lib, c["batch"]), _cnn_feeds(c, seed)
        return _graph_state(c, graphs.build_training(lib, fwd), feeds, DEVICE_GRAPH if c["recorded"] else 0)
    if kind == "block":
        bg = graphs.build_block(graph_lib(), c["batch"], c["S"], c["d"], c["H"], c["F"])
        return _graph_state(c, bg, _block_feeds(c, seed))
    dev = device()
    if kind in ("linear", "linear_backward", "int8_linear"):
        s = _linear_inputs(c, seed)
        if kind == "linear_backward":
            s.update(dx=torch.empty_like(s["x"]), dw=torch.empty_like(s["w"]), db=s["x"].new_empty(c["N"]))
        else:
            s["y"] = s["x"].new_empty(c["M"], c["N"])
        if kind == "int8_linear":
            s["packed"] = torch.empty(dev.i8_packed_bytes(c["K"], c["N"]), dtype=torch.int8, device="cuda")
            dev.i8_pack_weight(s["packed"].data_ptr(), s["w"].data_ptr(), c["K"], c["N"])
    elif kind in ("attention", "decode"):
        s = _attention_inputs(c, seed)
        s["y"] = torch.empty_like(s["q"])
    else:
        s = _conv_inputs(c, seed)
        if kind == "conv":
            s["y"] = s["x"].new_empty(c["batch"], c["C_out"], *_conv_out(c))
            if c["packed"]:
                nbytes = dev.conv2d_packed_bytes(c["C_out"], c["C_in"], c["k"], c["k"])
                s["packed"] = torch.empty(nbytes // 4, device="cuda")
                dev.conv2d_pack_weight(s["packed"].data_ptr(), s["w"].data_ptr(), c["C_out"], c["C_in"], c["k"],
                                       c["k"])
        else:
            s.update(dx=torch.empty_like(s["x"]), dw=torch.empty_like(s["w"]))
    return {"case": c, **s}


# ---- one pass -----------------------------------------------------------------


def _ptr(t):
    return None if t is None else t.data_ptr()


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if "program" in s:
        s["program"].run()
        return s["out"]
    dev = device()
    if kind == "linear":
        dev.gemm(_ptr(s["y"]), _ptr(s["x"]), _ptr(s["w"]), c["M"], c["K"], c["N"], _ptr(s["bias"]), ACTS[c["act"]],
                 _ptr(s["residual"]))
        return s["y"]
    if kind == "int8_linear":
        dev.gemm_i8p(_ptr(s["y"]), _ptr(s["x"]), _ptr(s["packed"]), s["scale"], c["M"], c["K"], c["N"],
                     _ptr(s["bias"]), ACTS[c["act"]])
        return s["y"]
    if kind == "linear_backward":
        M, K, N = c["M"], c["K"], c["N"]
        dev.gemm_ex(_ptr(s["dx"]), _ptr(s["dy"]), _ptr(s["w"]), M, N, K, trans_b=True)
        dev.gemm_ex(_ptr(s["dw"]), _ptr(s["x"]), _ptr(s["dy"]), K, M, N, trans_a=True)
        dev.sum_axis0(_ptr(s["db"]), _ptr(s["dy"]), M, N)
        return {"dx": s["dx"], "dw": s["dw"], "db": s["db"]}
    if kind == "attention":
        dev.attention_gqa(_ptr(s["y"]), _ptr(s["q"]), _ptr(s["k"]), _ptr(s["v"]), c["batch"], c["S_q"], c["S_kv"],
                          c["H_q"], c["H_kv"], c["D"], c["causal"])
        return s["y"]
    if kind == "decode":
        dev.attention_decode(_ptr(s["y"]), _ptr(s["q"]), _ptr(s["k"]), _ptr(s["v"]), _ptr(s["lens"]), c["batch"],
                             c["S_kv"], c["H_q"], c["H_kv"], c["D"])
        return s["y"]
    k, stride, pad = c["k"], c["stride"], c["k"] // 2
    if kind == "conv":
        conv, w = (dev.conv2d_packed, s["packed"]) if c["packed"] else (dev.conv2d, s["w"])
        conv(_ptr(s["y"]), _ptr(s["x"]), _ptr(w), _ptr(s["bias"]), c["batch"], c["C_in"], c["H"], c["W"], c["C_out"],
             k, k, stride, pad, ACTS[c["act"]])
        return s["y"]
    ho, wo = _conv_out(c)
    dims = (c["batch"], c["C_in"], c["H"], c["W"], c["C_out"], ho, wo, k, k, stride, pad)
    dev.conv2d_bwd_input(_ptr(s["dx"]), _ptr(s["dy"]), _ptr(s["w"]), *dims)
    dev.conv2d_bwd_weight(_ptr(s["dw"]), _ptr(s["dy"]), _ptr(s["x"]), *dims)
    return {"dx": s["dx"], "dw": s["dw"]}


# ---- what a pass cannot do without ----------------------------------------------


def _pairs(c):
    """Query-key pairs of one head of one sequence."""
    if not c["causal"]:
        return c["S_q"] * c["S_kv"]
    return sum(c["S_kv"] - c["S_q"] + i + 1 for i in range(c["S_q"]))


def work(case):
    c, kind = case, case["kind"]
    if kind == "mlp_forward" or kind == "mlp_train":
        b, k, h, n = c["batch"], c["d_in"], c["hidden"], c["classes"]
        weights, product = k * h + h + h * n + n, 2.0 * b * (k * h + h * n)
        if kind == "mlp_forward":
            return {"bytes": 4.0 * (b * k + weights + b * n), "flops": product}
        return {"bytes": 4.0 * (2 * b * k + 2 * weights + b * n + 1), "flops": 3 * product}
    if kind == "cnn_train":
        b = c["batch"]
        weights = 16 * 75 + 32 * 400 + 2048 * 120 + 120 + 1200 + 10
        product = 2.0 * b * (16 * 1024 * 75 + 32 * 256 * 400 + 2048 * 120 + 1200)
        return {"bytes": 4.0 * (2 * b * 3072 + 2 * weights + b * 10 + 1), "flops": 3 * product}
    if kind == "block":
        b, S, d, f = c["batch"], c["S"], c["d"], c["F"]
        weights = 4 * d * d + 2 * d * f + 9 * d + f
        return {"bytes": 4.0 * (2 * b * S * d + weights),
                "flops": b * (2.0 * S * (4 * d * d + 2 * d * f) + 4.0 * d * S * (S + 1) / 2)}
    if kind in ("linear", "int8_linear", "linear_backward"):
        M, K, N = c["M"], c["K"], c["N"]
        if kind == "linear_backward":
            return {"bytes": 4.0 * (2 * M * K + 2 * K * N + M * N + N), "flops": 4.0 * M * N * K}
        nbytes = 4.0 * (M * K + M * N + (N if c["bias"] else 0)) + K * N * (1.0 if kind == "int8_linear" else 4.0)
        return {"bytes": nbytes + (4.0 * M * N if c.get("residual") else 0.0), "flops": 2.0 * M * N * K}
    if kind == "attention":
        b, d = c["batch"], c["D"]
        return {"bytes": 8.0 * b * d * (c["S_q"] * c["H_q"] + c["S_kv"] * c["H_kv"]),
                "flops": 4.0 * b * c["H_q"] * d * _pairs(c)}
    if kind == "decode":
        b, d, mean = c["batch"], c["D"], 0.625 * c["S_kv"]  # lengths are uniform over the upper three quarters
        return {"bytes": 8.0 * b * d * (c["H_q"] + mean * c["H_kv"]), "flops": 4.0 * b * c["H_q"] * d * mean}
    ho, wo = _conv_out(c)
    x, w, y = c["batch"] * c["C_in"] * c["H"] * c["W"], c["C_out"] * c["C_in"] * c["k"] ** 2, c["batch"] * c["C_out"] * ho * wo
    flops = 2.0 * y * c["C_in"] * c["k"] ** 2
    if kind == "conv":
        return {"bytes": 4.0 * (x + w + y), "flops": flops}
    return {"bytes": 4.0 * (2 * x + 2 * w + y), "flops": 2 * flops}


# About four times the largest distance from exact() that the draws show.  Long
# fp32 sums (K up to 8192, a filter gradient over every pixel) are the largest;
# the quantized product is exact up to its last rounding.
TOLERANCE = {"mlp_forward": 1.5e-6, "block": 2e-6, "linear": 5e-6, "linear_backward": 5e-6, "attention": 3e-6,
             "decode": 1e-6, "conv": 5e-6, "conv_backward": 5e-6, "int8_linear": 3e-7,
             # 2e-6 too, unless a ReLU or a pooling window decides between values that differ by less than
             # a rounding: the other choice is as correct and moves a gradient by one element's share
             "mlp_train": 1e-2, "cnn_train": 1e-2}


def tolerance(case):
    return {"rel": TOLERANCE[case["kind"]]}


# ---- the same results in 64 bits -------------------------------------------------


def _act(y, act):
    return F.relu(y) if act == "relu" else F.gelu(y, approximate="tanh") if act == "gelu" else y


def _leaf(feeds):
    return {k: torch.from_numpy(v).double().requires_grad_() for k, v in feeds.items()}


def _exact_train(c, seed):
    if c["kind"] == "mlp_train":
        t = _leaf(_mlp_feeds(c, seed))
        logits = F.relu(t["X"] @ t["W1"] + t["b1"]) @ t["W2"] + t["b2"]
    else:
        t = _leaf(_cnn_feeds(c, seed))
        h = F.max_pool2d(F.relu(F.conv2d(t["X"], t["W1"], padding=2)), 2)
        h = F.max_pool2d(F.relu(F.conv2d(h, t["W2"], padding=2)), 2)
        logits = F.relu(h.flatten(1) @ t["W3"] + t["b1"]) @ t["W4"] + t["b2"]
    loss = -(t["Y"].detach() * F.log_softmax(logits, 1)).sum(1).mean()
    loss.backward()
    return {"loss": loss.detach().reshape(1, 1), **{"d" + k: v.grad for k, v in t.items() if k != "Y"}}


def _softmax_attention(q, k, v, causal):
    """q [S_q, H, D], k and v [S_kv, H, D] in float64; query i sits at key S_kv - S_q + i."""
    q, k, v = q.transpose(0, 1).contiguous(), k.permute(1, 2, 0).contiguous(), v.transpose(0, 1).contiguous()
    s = torch.matmul(q, k) / math.sqrt(q.shape[-1])
    if causal:
        keep = torch.ones(s.shape[-2:], dtype=torch.bool, device=s.device).tril(s.shape[-1] - s.shape[-2])
        s = s.masked_fill(~keep, float("-inf"))
    return torch.matmul(s.softmax(-1), v).transpose(0, 1).contiguous()


def _exact_block(c, seed):
    t = {k: torch.from_numpy(v).cuda().double() for k, v in _block_feeds(c, seed).items()}
    S, d, H = c["S"], c["d"], c["H"]
    out = {}
    for s in range(c["batch"]):
        x = t[f"x{s}"]
        h = F.layer_norm(x, (d,), t["g1"][0], t["be1"][0], 1e-5)
        q, k, v = ((h @ t["W" + n] + t["b" + n]).reshape(S, H, d // H) for n in "qkv")
        x1 = _softmax_attention(q, k, v, True).reshape(S, d) @ t["Wo"] + t["bo"] + x
        h = F.layer_norm(x1, (d,), t["g2"][0], t["be2"][0], 1e-5)
        out[f"y{s}"] = F.gelu(h @ t["W1"] + t["bf1"], approximate="tanh") @ t["W2"] + t["bf2"] + x1
    return out


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "mlp_forward":
        t = {k: torch.from_numpy(v).double() for k, v in _mlp_feeds(c, seed).items()}
        return {"softmax": (F.relu(t["x"] @ t["W1"] + t["b1"]) @ t["W2"] + t["b2"]).softmax(1)}
    if kind in ("mlp_train", "cnn_train"):
        return _exact_train(c, seed)
    if kind == "block":
        return _exact_block(c, seed)
    if kind in ("linear", "int8_linear", "linear_backward"):
        s = _linear_inputs(c, seed)
        x, w = s["x"].double(), s["w"].double()
        if kind == "linear_backward":
            dy = s["dy"].double()
            return {"dx": dy @ w.t(), "dw": x.t() @ dy, "db": dy.sum(0)}
        if kind == "int8_linear":
            scale = x.abs().max() / 127.0
            q = x / scale
            y = ((torch.sign(q) * torch.floor(q.abs() + 0.5)) @ w) * (scale * s["scale"])
        else:
            y = x @ w
        if s["bias"] is not None:
            y = y + s["bias"].double()
        y = _act(y, c["act"])
        return y if s["residual"] is None else y + s["residual"].double()
    if kind in ("attention", "decode"):
        s = _attention_inputs(c, seed)
        group = c["H_q"] // c["H_kv"]
        out = []
        for b in range(c["batch"]):
            n = int(s["lens"][b]) if kind == "decode" else c["S_kv"]
            q = s["q"][b].double()
            k, v = (s[t][b, :n].double().repeat_interleave(group, 1) for t in "kv")
            if kind == "decode":
                out.append(_softmax_attention(q[None], k, v, False)[0])
            else:
                out.append(_softmax_attention(q, k, v, c["causal"]))
        return torch.stack(out)
    s = _conv_inputs(c, seed)
    k, pad, stride = c["k"], c["k"] // 2, c["stride"]
    w = s["w"].double().reshape(c["C_out"], -1)
    ys, dxs, dw = [], [], torch.zeros_like(w)
    for x, dy in zip(s["x"].double(), s["dy"].double() if "dy" in s else s["x"]):
        cols = F.unfold(x[None], k, padding=pad, stride=stride)[0]
        if kind == "conv":
            ys.append(_act(w @ cols + s["bias"].double()[:, None], c["act"]).reshape(c["C_out"], *_conv_out(c)))
        else:
            dy = dy.reshape(c["C_out"], -1)
            dw += dy @ cols.t()
            dxs.append(F.fold((w.t() @ dy)[None], x.shape[-2:], k, padding=pad, stride=stride)[0])
    if kind == "conv":
        return torch.stack(ys)
    return {"dx": torch.stack(dxs), "dw": dw.reshape(s["w"].shape)}
