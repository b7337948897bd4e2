"""The workloads this framework is timed on: programs built with NetBuilder, compiled with
Computation.build_and_compile and executed, as a user's program does it.  A program keeps its compiled computation,
its weights and its input tensors on the GPU; one pass is one execution.

`listed()` are fixed cases, `draw(rng)` gives another one of the same kinds and ranges.  The kinds:

  add_relu      relu(scale * (a + b)), a chain of element-wise operators over an image batch
  row_ops       softmax, layer norm, row sum and argmax over the last axis
  matmul        one product, any operand transposed, batched or not
  linear_train  a linear layer's training step: y = x W + b, dx, dW, db
  conv_train    a convolution block's training step: convolution, batch norm, relu, max pooling or not, and the
                gradients of all of them
  resnet50      ResNet-50 v1.5 inference, const weights
  transformer   one transformer block with const weights: a whole prompt (past = 0), or new tokens that attend to
                `past` cached ones
  top_k         the k largest scores of every row with their indices
"""
import math

import numpy as np
import torch

from cinn_amd import runtime
from cinn_amd.common import BFloat16, DefaultAMDGPUTarget, Float
from cinn_amd.frontend import Computation, NetBuilder

_BYTES = {"float32": 4, "float16": 2, "bfloat16": 2}
_TORCH = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16, "int32": torch.int32,
          "int64": torch.int64}


def listed():
    return [
        # the first framework configuration's operators over an image batch: launch and memory bound
        {"name": "add_relu_f32_b32", "kind": "add_relu", "n": 32, "c": 3, "h": 224, "w": 224, "dtype": "float32"},
        # normalisation and scoring operators of a large activation: memory bound
        {"name": "row_ops_f32_4096", "kind": "row_ops", "rows": 4096, "cols": 4096, "dtype": "float32"},
        # the large square product of the benchmark
        {"name": "matmul_bf16_4096", "kind": "matmul", "batch": 1, "m": 4096, "n": 4096, "k": 4096, "ta": False,
         "tb": False, "dtype": "bfloat16"},
        # an ordinary single-precision product whose extents are no powers of two
        {"name": "matmul_f32_1000", "kind": "matmul", "batch": 1, "m": 1000, "n": 1000, "k": 1000, "ta": False,
         "tb": False, "dtype": "float32"},
        # training step of a transformer's first feed-forward layer; the token count is not a multiple of any tile
        {"name": "linear_train_f16_4100", "kind": "linear_train", "tokens": 4100, "inp": 768, "out": 3072,
         "dtype": "float16"},
        # training step of a 3x3 layer of an image network's first stage, the framework's default layout
        {"name": "conv_train_f16_56_nchw", "kind": "conv_train", "n": 32, "c": 64, "h": 56, "w": 56, "f": 64, "k": 3,
         "stride": 1, "pool": False, "layout": "NCHW", "dtype": "float16"},
        # training step of a strided layer with pooling behind it, odd extents, channels last, single precision
        {"name": "conv_train_f32_odd_nhwc", "kind": "conv_train", "n": 8, "c": 96, "h": 35, "w": 41, "f": 200, "k": 3,
         "stride": 2, "pool": True, "layout": "NHWC", "dtype": "float32"},
        # offline inference of a whole network, replayed as a graph
        {"name": "resnet50_f16_b32", "kind": "resnet50", "batch": 32, "image": 224, "graph": True, "dtype": "float16"},
        # one request at a time: launch latency and small grids
        {"name": "resnet50_f16_b1", "kind": "resnet50", "batch": 1, "image": 224, "graph": False, "dtype": "float16"},
        # prefill: a batch of whole prompts through a block
        {"name": "transformer_f16_prefill", "kind": "transformer", "batch": 8, "tokens": 512, "past": 0, "hidden": 768,
         "heads": 12, "graph": False, "dtype": "float16"},
        # decode: one new token per sequence against a cache
        {"name": "transformer_f16_decode", "kind": "transformer", "batch": 8, "tokens": 1, "past": 511, "hidden": 768,
         "heads": 12, "graph": True, "dtype": "float16"},
        # top-5 of a thousand classes for a large batch of scores
        {"name": "top_k_2048x1000", "kind": "top_k", "rows": 2048, "cols": 1000, "k": 5, "dtype": "float32"},
    ]


def _log(rng, low, high):
    """a whole number between low and high, spread over its logarithm"""
    return int(min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _pick_case(rng):
    kind = rng.choice(["add_relu", "row_ops", "matmul", "linear_train", "conv_train", "conv_train", "resnet50",
                       "transformer", "transformer", "top_k"])
    dtype = rng.choice(["float32", "float16", "bfloat16"])
    if kind == "add_relu":
        return {"kind": kind, "n": _log(rng, 8, 64), "c": _log(rng, 3, 256), "h": _log(rng, 14, 224),
                "w": _log(rng, 14, 224), "dtype": dtype}
    if kind == "row_ops":
        return {"kind": kind, "rows": _log(rng, 32, 16384), "cols": _log(rng, 64, 8192), "dtype": dtype}
    if kind == "matmul":
        batch = rng.choice([1, 1, _log(rng, 2, 64)])
        return {"kind": kind, "batch": batch, "m": _log(rng, 16, 4096), "n": _log(rng, 16, 4096),
                "k": _log(rng, 16, 4096), "ta": rng.random() < 0.25, "tb": rng.random() < 0.5, "dtype": dtype}
    if kind == "linear_train":
        return {"kind": kind, "tokens": _log(rng, 32, 16384), "inp": _log(rng, 64, 4096), "out": _log(rng, 64, 4096),
                "dtype": dtype}
    if kind == "conv_train":
        k = rng.choice([1, 3, 3, 5, 7])
        return {"kind": kind, "n": _log(rng, 1, 32), "c": rng.choice([3, _log(rng, 8, 512), 16 * _log(rng, 1, 32)]),
                "h": _log(rng, 7, 112), "w": _log(rng, 7, 112), "f": rng.choice([_log(rng, 8, 512), 16 * _log(rng, 1, 32)]),
                "k": k, "stride": rng.choice([1, 1, 2]), "pool": rng.random() < 0.3, "layout": rng.choice(["NCHW", "NHWC"]),
                "dtype": dtype}
    if kind == "resnet50":
        return {"kind": kind, "batch": _log(rng, 1, 32), "image": rng.choice([160, 192, 224]),
                "graph": rng.random() < 0.5, "dtype": rng.choice(["float32", "float16"])}
    if kind == "transformer":
        heads = rng.choice([8, 12, 16])
        decode = rng.random() < 0.5
        return {"kind": kind, "batch": _log(rng, 1, 16), "tokens": 1 if decode else _log(rng, 16, 768),
                "past": _log(rng, 31, 1023) if decode else 0, "hidden": heads * rng.choice([48, 64, 80]), "heads": heads,
                "graph": rng.random() < 0.5, "dtype": rng.choice(["float16", "float16", "bfloat16", "float32"])}
    return {"kind": kind, "rows": _log(rng, 1, 4096), "cols": _log(rng, 100, 8192), "k": rng.choice([1, 5, 10, 50]),
            "dtype": rng.choice(["float32", "float32", "float16"])}


def _affordable(case):
    """a pass is at least a few microseconds of work and no more than the listed cases ask for: multiply-adds, bytes,
    comparisons"""
    kind, w = case["kind"], work(case)
    if kind == "add_relu":
        return 1 << 21 <= case["n"] * case["c"] * case["h"] * case["w"] <= 1 << 25
    if kind == "row_ops":
        return 1 << 20 <= case["rows"] * case["cols"] <= 1 << 24
    if kind == "matmul":
        return w["flops"] <= 2 ** 37 * (1.0 if case["dtype"] != "float32" else 0.1) and w["bytes"] <= 1 << 28
    if kind == "linear_train":
        return w["flops"] <= 6e10 * (2.0 if case["dtype"] != "float32" else 0.5)
    if kind == "conv_train":
        # a filter gradient's cost is its multiply-adds; the window has to fit, pooling needs something to pool;
        # channels-last convolutions are defined for whole 16-byte groups of channels
        oh, ow = _conv_out(case)
        if case["layout"] == "NHWC" and case["c"] % 8 != 0:
            return False
        return min(case["h"], case["w"]) >= case["k"] and min(oh, ow) >= 4 and w["flops"] <= 2.3e10
    if kind == "transformer":
        return w["flops"] <= 1.3e11 * (1.0 if case["dtype"] != "float32" else 0.15)
    if kind == "top_k":
        return case["rows"] * case["cols"] ** 2 <= 2048 * 1000 ** 2 * 8
    return True


def draw(rng):
    while True:
        case = _pick_case(rng)
        if _affordable(case):
            return case


# ---- building programs -----------------------------------------------------------------------------------------------
def _type(dtype):
    return BFloat16() if dtype == "bfloat16" else Float(8 * _BYTES[dtype])


class _DeviceArray(object):
    """what torch needs to see a tensor of a compiled computation where it lies; torch keeps this object for as long as
    it looks at the memory, and this object keeps the computation, which owns the memory"""

    def __init__(self, owner, pointer, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (pointer, False), "shape": tuple(shape), "typestr": typestr,
                                         "strides": None, "version": 2}


def _view(comp, name):
    t = comp.get_tensor(name)
    dtype = str(t.type())
    typestr = {"float32": "<f4", "float16": "<f2", "bfloat16": "<i2", "int32": "<i4", "int64": "<i8"}[dtype]
    seen = torch.as_tensor(_DeviceArray(comp, t.device_ptr, t.shape(), typestr), device="cuda")
    return seen.view(_TORCH[dtype]) if dtype == "bfloat16" else seen


def _host(t):
    """a tensor as Tensor.from_numpy takes it (bfloat16 travels as bit patterns)"""
    if t.dtype == torch.bfloat16:
        return t.view(torch.int16).cpu().numpy().view(np.uint16)
    return t.cpu().numpy()


class _Feeder(object):
    """makes inputs on the GPU from one seed and remembers them until the program is compiled"""

    def __init__(self, builder, dtype, seed):
        self.b, self.dtype = builder, dtype
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(int(seed))
        self.data = {}

    def _put(self, name, value, dtype, const):
        var = self.b.create_input(_type(dtype), list(value.shape), name)
        if const:
            var.set_const(True)
        self.data[var.id] = value.to(_TORCH[dtype])
        return var

    def normal(self, name, shape, scale=1.0, mean=0.0, dtype=None, const=False):
        value = torch.randn(list(shape), generator=self.gen, device="cuda") * scale + mean
        return self._put(name, value, dtype or self.dtype, const)

    def uniform(self, name, shape, low, high, dtype=None, const=False):
        value = torch.rand(list(shape), generator=self.gen, device="cuda") * (high - low) + low
        return self._put(name, value, dtype or self.dtype, const)


_STREAM = []


def _stream():
    """the program's one stream; its computations follow one another on it"""
    if not _STREAM:
        _STREAM.append(runtime.Stream())
    return _STREAM[0]


def _conv_out(case):
    pad = case["k"] // 2
    return tuple((case[d] + 2 * pad - case["k"]) // case["stride"] + 1 for d in ("h", "w"))


def _pool_out(extent):
    return (extent + 2 - 3) // 2 + 1


def _add_relu(case, b, feed):
    shape = [case["n"], case["c"], case["h"], case["w"]]
    x, y = feed.normal("x", shape), feed.normal("y", shape)
    return [b.relu(b.scale(b.add(x, y), 0.5, 0.1))]


def _row_ops(case, b, feed):
    x = feed.normal("x", [case["rows"], case["cols"]])
    gamma, beta = feed.uniform("gamma", [case["cols"]], 0.5, 1.5), feed.normal("beta", [case["cols"]], 0.1)
    y, mean, var = b.paddle_layer_norm(x, gamma, beta)
    return [b.softmax(x, axes=[-1]), y, mean, var, b.reduce_sum(x, [1]), b.argmax(x, 1)]


def _matmul(case, b, feed):
    lead = [] if case["batch"] == 1 else [case["batch"]]
    m, n, k = case["m"], case["n"], case["k"]
    x = feed.normal("x", lead + ([k, m] if case["ta"] else [m, k]))
    y = feed.normal("y", lead + ([n, k] if case["tb"] else [k, n]), 1.0 / math.sqrt(k))
    return [b.matmul(x, y, case["ta"], case["tb"])]


def _linear_train(case, b, feed):
    t, i, o = case["tokens"], case["inp"], case["out"]
    x, w = feed.normal("x", [t, i]), feed.normal("w", [i, o], 1.0 / math.sqrt(i))
    bias, dy = feed.normal("bias", [o], 0.1), feed.normal("dy", [t, o], 0.1)
    return [b.add(b.matmul(x, w), bias), b.matmul(dy, w, False, True), b.matmul(x, dy, True, False),
            b.reduce_sum(dy, [0])]


def _conv_train(case, b, feed):
    n, c, h, w_, f, k, s = (case[q] for q in ("n", "c", "h", "w", "f", "k", "stride"))
    layout, pad = case["layout"], k // 2
    oh, ow = _conv_out(case)

    def image(channels, height, width):
        return [n, channels, height, width] if layout == "NCHW" else [n, height, width, channels]

    w_shape = [f, c, k, k] if layout == "NCHW" else [f, k, k, c]
    x = feed.normal("x", image(c, h, w_))
    w = feed.normal("w", w_shape, math.sqrt(2.0 / (c * k * k)))
    gamma, beta = feed.uniform("gamma", [f], 0.5, 1.5, "float32"), feed.normal("beta", [f], 0.1, dtype="float32")
    mean, var = feed.normal("mean", [f], 0.1, dtype="float32"), feed.uniform("var", [f], 0.8, 1.2, "float32")
    geometry = dict(strides=[s, s], paddings=[pad, pad], data_format=layout)
    z = b.conv(x, w, **geometry)
    norm, saved_mean, saved_var, new_mean, new_var = b.batchnorm(z, gamma, beta, mean, var, data_layout=layout,
                                                                 is_test=False)
    act = b.relu(norm)
    outs = [new_mean, new_var]
    if case["pool"]:
        args = ("max", [3, 3], [2, 2], [1, 1])
        y = b.pool2d(act, *args, data_format=layout)
        dy = feed.normal("dy", image(f, _pool_out(oh), _pool_out(ow)), 0.1)
        dact = b.pool2d_grad(act, y, dy, *args, data_format=layout)
    else:
        y = act
        dy = feed.normal("dy", image(f, oh, ow), 0.1)
        dact = dy
    dz, dgamma, dbeta = b.batch_norm_grad(b.relu_grad(dact, act), z, gamma, saved_mean, saved_var, data_layout=layout)
    dx = b.conv(w, dz, conv_type="backward_data", output_shape=image(c, h, w_), **geometry)
    dw = b.conv(x, dz, conv_type="backward_filter", output_shape=w_shape, **geometry)
    return [y, dx, dw, dgamma, dbeta] + outs


_STAGES = ((3, 64, 1), (4, 128, 2), (6, 256, 2), (3, 512, 2))  # blocks, bottleneck width, stride of the stage


def _resnet50(case, b, feed):
    def conv_bn(x, name, channels, k, stride, relu, last=False):
        cin = x.shape()[1]
        w = feed.normal(name + "_w", [channels, cin, k, k], math.sqrt(2.0 / (cin * k * k)), const=True)
        # the last batch norm of a block is scaled down: activations keep their size through the residual additions
        gamma = feed.uniform(name + "_g", [channels], *((0.2, 0.4) if last else (0.8, 1.2)), const=True)
        beta, mean = (feed.normal(name + e, [channels], 0.1, const=True) for e in ("_b", "_m"))
        var = feed.uniform(name + "_v", [channels], 0.8, 1.2, const=True)
        y = b.batchnorm(b.conv2d(x, w, strides=[stride, stride], paddings=[k // 2, k // 2]), gamma, beta, mean, var)[0]
        return b.relu(y) if relu else y

    x = feed.normal("image", [case["batch"], 3, case["image"], case["image"]])
    y = b.pool2d(conv_bn(x, "stem", 64, 7, 2, True), "max", [3, 3], [2, 2], [1, 1])
    for si, (blocks, mid, stride) in enumerate(_STAGES):
        for bi in range(blocks):
            name, s = "s%db%d" % (si, bi), stride if bi == 0 else 1
            short = conv_bn(y, name + "_s", 4 * mid, 1, s, False) if bi == 0 else y
            z = conv_bn(y, name + "_1", mid, 1, 1, True)
            z = conv_bn(z, name + "_2", mid, 3, s, True)
            z = conv_bn(z, name + "_3", 4 * mid, 1, 1, False, last=True)
            y = b.relu(b.add(z, short))
    y = b.reshape(b.pool2d(y, "avg", [7, 7], global_pooling=True), [case["batch"], 2048])
    w = feed.normal("fc_w", [2048, 1000], 1.0 / math.sqrt(2048), const=True)
    return [b.add(b.matmul(y, w), feed.normal("fc_b", [1000], 0.1, const=True))]


def _transformer(case, b, feed):
    n, t, past, hidden, heads = (case[q] for q in ("batch", "tokens", "past", "hidden", "heads"))
    d = hidden // heads

    def linear(x, name, inp, out):
        w = feed.normal(name + "_w", [inp, out], 1.0 / math.sqrt(inp), const=True)
        return b.add(b.matmul(x, w), feed.normal(name + "_b", [out], 0.02, const=True))

    def norm(x, name):
        gamma = feed.uniform(name + "_g", [hidden], 0.8, 1.2, const=True)
        return b.paddle_layer_norm(x, gamma, feed.normal(name + "_b", [hidden], 0.02, const=True))[0]

    def split(x):
        return b.transpose(b.reshape(x, [n, t, heads, d]), [0, 2, 1, 3])

    x = feed.normal("x", [n * t, hidden])
    z = norm(x, "ln1")
    q, k, v = (split(linear(z, e, hidden, hidden)) for e in ("q", "k", "v"))
    outs = []
    if past:
        outs = [k, v]  # what the caller appends to its cache
        k = b.concat([feed.normal("past_k", [n, heads, past, d]), k], axis=2)
        v = b.concat([feed.normal("past_v", [n, heads, past, d]), v], axis=2)
    p = b.softmax(b.matmul(q, k, False, True, 1.0 / math.sqrt(d)), axes=[-1])
    o = b.reshape(b.transpose(b.matmul(p, v), [0, 2, 1, 3]), [n * t, hidden])
    x = b.add(x, linear(o, "o", hidden, hidden))
    y = b.add(x, linear(b.gelu(linear(norm(x, "ln2"), "up", hidden, 4 * hidden)), "down", 4 * hidden, hidden))
    return [y] + outs


def _top_k(case, b, feed):
    return list(b.top_k(feed.normal("scores", [case["rows"], case["cols"]]), case["k"]))


_BUILD = {"add_relu": _add_relu, "row_ops": _row_ops, "matmul": _matmul, "linear_train": _linear_train,
          "conv_train": _conv_train, "resnet50": _resnet50, "transformer": _transformer, "top_k": _top_k}


def prepare(case, seed):
    """a compiled program with its weights and inputs on the GPU"""
    b = NetBuilder(case["kind"])
    feed = _Feeder(b, case["dtype"], seed)
    outs = _BUILD[case["kind"]](case, b, feed)
    comp = Computation.build_and_compile(DefaultAMDGPUTarget(), b, outputs=outs, stream=_stream())
    for name, value in feed.data.items():
        comp.get_tensor(name).from_numpy(_host(value))
    return {"comp": comp, "graph": bool(case.get("graph", False)), "outputs": [_view(comp, o.id) for o in outs]}


def run(state):
    if state["graph"]:
        state["comp"].execute_graph()
    else:
        state["comp"].execute()
    return state["outputs"]


# ---- what a pass cannot do without -----------------------------------------------------------------------------------
def _resnet50_work(case):
    n, e = case["batch"], _BYTES[case["dtype"]]
    size = (case["image"] + 2 * 3 - 7) // 2 + 1
    weights, flops = 64 * 3 * 49, 2.0 * n * 64 * 3 * 49 * size * size
    size, cin = _pool_out(size), 64
    for blocks, mid, stride in _STAGES:
        for bi in range(blocks):
            s = stride if bi == 0 else 1
            out = (size - 1) // s + 1
            layers = [(mid * cin, size), (9 * mid * mid, out), (4 * mid * mid, out)]
            layers += [(4 * mid * cin, out)] if bi == 0 else []
            weights += sum(w for w, _ in layers)
            flops += sum(2.0 * n * w * side * side for w, side in layers)
            size, cin = out, 4 * mid
    weights += 2048 * 1000
    flops += 2.0 * n * 2048 * 1000
    return {"bytes": e * (weights + n * (3 * case["image"] ** 2 + 1000)), "flops": flops}


def work(case):
    """bytes: every fed tensor read once and every fetched one written once; flops: the contractions (the operators
    themselves where there is no contraction)"""
    kind, e = case["kind"], _BYTES[case["dtype"]]
    if kind == "add_relu":
        count = case["n"] * case["c"] * case["h"] * case["w"]
        return {"bytes": 3 * e * count, "flops": 4 * count}
    if kind == "row_ops":
        rows, cols = case["rows"], case["cols"]
        return {"bytes": 3 * e * rows * cols + rows * (8 + e + 4) + 2 * e * cols, "flops": 15 * rows * cols}
    if kind == "matmul":
        n, m, o, k = case["batch"], case["m"], case["n"], case["k"]
        return {"bytes": n * e * (m * k + k * o + m * o), "flops": 2.0 * n * m * o * k}
    if kind == "linear_train":
        t, i, o = case["tokens"], case["inp"], case["out"]
        return {"bytes": e * (2 * t * i + 2 * t * o + 2 * i * o + 2 * o), "flops": 6.0 * t * i * o}
    if kind == "conv_train":
        n, c, f, k = case["n"], case["c"], case["f"], case["k"]
        oh, ow = _conv_out(case)
        image, conv = n * c * case["h"] * case["w"], n * f * oh * ow
        pooled = n * f * _pool_out(oh) * _pool_out(ow) if case["pool"] else conv
        # the convolution's result has to be complete before its statistics are known, and the sums of the gradient
        # before the gradient is: it is written once and read three times
        return {"bytes": e * (3 * image + 2 * pooled + 3 * f * c * k * k + 4 * conv) + 32 * f,
                "flops": 6.0 * conv * c * k * k}
    if kind == "resnet50":
        return _resnet50_work(case)
    if kind == "transformer":
        n, t, hidden = case["batch"], case["tokens"], case["hidden"]
        total = t + case["past"]
        moved = 2 * n * t * hidden + 12 * hidden * hidden + 13 * hidden
        if case["past"]:
            moved += 2 * n * total * hidden
        return {"bytes": e * moved, "flops": 24.0 * n * t * hidden * hidden + 4.0 * n * t * total * hidden}
    count = case["rows"] * case["cols"]
    return {"bytes": e * count + case["rows"] * case["k"] * (e + 8), "flops": count * math.log2(max(2, case["k"]))}


def tolerance(case):
    """Measured against the same programs in float64 (relative 2-norm), stated about four times as wide: products and
    blocks 2.1e-4 to 4.1e-4 in float16, 1.6e-3 to 2.4e-3 in bfloat16, 5.7e-7 in float32 at 1000 terms a sum (longer sums:
    growing with their root)."""
    kind, dtype = case["kind"], case["dtype"]
    if kind in ("add_relu", "top_k"):  # one rounding for each operator; values and indices that are only moved
        return "exact"
    if kind == "conv_train":
        # A relu whose input lies within one rounding of zero passes its gradient or not, and a pooling window whose two
        # largest values do gives it to the one or the other: whole elements of the gradient differ, not their last
        # digits.  Measured 4e-3 to 1e-2 in float16 (largest element 0.4 to 0.8 of the root mean square), 6e-3 to
        # 1.6e-2 in bfloat16, and without such an element 1e-6 in float32; one among the 3e5 to 6e6 values of a layer,
        # which float32 meets now and then, is 4e-4 to 2e-3.
        return {"float32": {"rel": 2e-3, "max": 0.3}, "float16": {"rel": 1.6e-2, "max": 0.9},
                "bfloat16": {"rel": 3e-2, "max": 0.99}}[dtype]
    return {"float32": {"rel": 1e-5, "max": 4e-4}, "float16": {"rel": 2e-3, "max": 2e-2},
            "bfloat16": {"rel": 1e-2, "max": 1e-1}}[dtype]
