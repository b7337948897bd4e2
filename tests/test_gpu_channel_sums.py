"""Training batch norm on channels-last tensors: the statistics and the gradient sums are one library call each
(cinn_call_hip_channel_statistics / cinn_call_hip_channel_gradient_sums), what they are applied to is one more each
(cinn_call_hip_channel_normalize / cinn_call_hip_channel_gradient), a relu and its mask go inside these, and a convolution's training step written in NCHW stays channels-last between its first convolution and its gradients."""
import numpy as np
import pytest
import torch

from cinn_amd.common import BFloat16, DefaultAMDGPUTarget, Float, bfloat16_bits_to_float32, float32_to_bfloat16_bits
from cinn_amd.frontend import Computation, NetBuilder

pytestmark = pytest.mark.gpu

# half a unit in the last place of the stored result
ROUNDING = {"float32": 2.0 ** -24, "float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}


def _type(dtype):
    return BFloat16() if dtype == "bfloat16" else Float(16 if dtype == "float16" else 32)


def _stored(a, dtype):
    """what Tensor.from_numpy takes, and the same values in float64"""
    if dtype == "bfloat16":
        raw = float32_to_bfloat16_bits(a.astype(np.float32))
        return raw, bfloat16_bits_to_float32(raw).astype(np.float64)
    raw = a.astype(dtype)
    return raw, raw.astype(np.float64)


def _run(b, outs, data):
    comp = Computation.build_and_compile(DefaultAMDGPUTarget(), b, outputs=outs)
    for var, raw in data:
        comp.get_tensor(var.id).from_numpy(raw)
    comp.execute()
    names = [comp.instruction_info(i)[0] for i in range(comp.num_instructions())]
    got = []
    for o in outs:
        a = comp.get_tensor(o.id).numpy()
        got.append(bfloat16_bits_to_float32(a).astype(np.float64) if str(o.type()) == "bfloat16" else a.astype(np.float64))
    return got, names


# channels: one, no whole chunk, one chunk, a power of two, several blocks of channels; pixels: one, fewer than a block's
# rows, ragged splits
@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (1, 1, 1, 8), (2, 3, 5, 7), (3, 17, 19, 64), (2, 9, 5, 200), (1, 5, 7, 1100),
                                   (4, 33, 31, 3), (8, 61, 67, 16)])
@pytest.mark.parametrize("masked", [False, True])
def test_statistics_and_gradient(gpu, shape, dtype, masked):
    rng = np.random.default_rng(sum(shape))
    raw = {n: _stored(rng.standard_normal(shape) + m, dtype) for n, m in (("x", 0.5), ("dy", 0.0), ("act", 0.0))}
    c, count = shape[3], float(np.prod(shape[:3]))
    vec = {n: rng.uniform(0.5, 1.5, c).astype(np.float32) for n in ("scale", "bias", "mean", "var")}
    b = NetBuilder("channel_sums")
    X, DY, A = (b.create_input(_type(dtype), list(shape), n) for n in ("x", "dy", "act"))
    V = {n: b.create_input(Float(32), [c], n) for n in vec}
    outs = list(b.batchnorm(X, V["scale"], V["bias"], V["mean"], V["var"], is_test=False, data_layout="NHWC"))
    if masked:
        outs[0] = b.relu(outs[0])
    grad = b.relu_grad(DY, A) if masked else DY
    outs += list(b.batch_norm_grad(grad, X, V["scale"], V["mean"], V["var"], data_layout="NHWC"))
    got, names = _run(b, outs, [(v, raw[n][0]) for v, n in ((X, "x"), (DY, "dy"), (A, "act")) if masked or n != "act"] +
                      [(V[n], vec[n]) for n in vec])
    for call in ("channel_statistics", "channel_normalize", "channel_gradient_sums", "channel_gradient"):
        assert sum("hip_" + call in n for n in names) == (2 if call == "channel_gradient" else 1)
    assert not any("reduce" in n or "relu" in n or "select" in n for n in names)
    x, dy, act = (raw[n][1] for n in ("x", "dy", "act"))
    dy = np.where(act > 0, dy, 0.0) if masked else dy
    v64 = {n: vec[n].astype(np.float64) for n in vec}
    axes = (0, 1, 2)
    # fp32 sums in chains of at most `count` terms, each rounded once, of the sizes that are added
    unit = 2.0 ** -23 * (4 + min(count, 300))

    def near(a, want, size):
        assert np.all(np.abs(a - want) <= unit * size + 1e-30), np.max(np.abs(a - want) / (unit * size + 1e-30))

    mean, square = x.mean(axes), (x * x).mean(axes)
    var = square - mean * mean
    near(got[1], mean, np.abs(x).mean(axes))
    near(got[2], var, 3 * square)
    near(got[3], 0.9 * v64["mean"] + 0.1 * mean, v64["mean"] + np.abs(x).mean(axes))
    near(got[4], 0.9 * v64["var"] + 0.1 * var, v64["var"] + 3 * square)
    inv = 1.0 / np.sqrt(var + 1e-5)
    y = (x - mean) * inv * v64["scale"] + v64["bias"]
    # y's share of the statistics' errors: of the mean by inv, of the variance by inv^2 / 2 of the normalised value
    size = inv * v64["scale"] * (np.abs(x) + np.abs(mean) + np.abs(x - mean) * 3 * square * inv * inv) + v64["bias"]
    y_err = np.abs(got[0] - (np.maximum(y, 0.0) if masked else y))
    assert np.all(y_err <= 2 * unit * size + ROUNDING[dtype] * np.abs(y) + 1e-7)
    centred = x - v64["mean"]
    sum_dy, sum_dyx = dy.sum(axes), (dy * centred).sum(axes)
    size_dy, size_dyx = np.abs(dy).sum(axes), np.abs(dy * centred).sum(axes)
    near(got[7], sum_dy, size_dy)
    inv = 1.0 / np.sqrt(v64["var"] + 1e-5)
    near(got[6], sum_dyx * inv, 2 * size_dyx * inv)
    want = v64["scale"] * inv / count * (count * dy - sum_dy - centred * sum_dyx * inv * inv)
    size = v64["scale"] * inv / count * (count * np.abs(dy) + size_dy + np.abs(centred) * size_dyx * inv * inv)
    assert np.all(np.abs(got[5] - want) <= 2 * unit * size + ROUNDING[dtype] * np.abs(want) + 1e-7)


# channels that are whole chunks and not, filters of 1x1 (reshaped, not transposed) and 3x3, strides, pooling
@pytest.mark.parametrize("c,f,k,stride,pool", [(8, 16, 3, 1, False), (3, 8, 3, 1, False), (16, 5, 1, 1, True), (12, 24, 3, 2, True)])
def test_nchw_training_step_matches_the_unconverted_one(gpu, c, f, k, stride, pool):
    """the same program with conv_layout_nhwc on and off: fp32 sums in another order, and no transposes of gradients in
    between.  A value near a relu's or a window's edge would move whole elements, so inputs keep clear of ties by being
    random in fp32; the bound is relative to the largest element of each result."""
    rng = np.random.default_rng(c + f)
    n, h, w = 3, 13, 11
    results = []
    for convert in (True, False):
        b = NetBuilder("step")
        rng = np.random.default_rng(c * 100 + f)
        data = []

        def put(name, shape, low=None):
            a = (rng.standard_normal(shape) if low is None else rng.uniform(low, low + 1.0, shape)).astype(np.float32)
            v = b.create_input(Float(32), list(shape), name)
            data.append((v, a))
            return v

        geometry = dict(strides=[stride, stride], paddings=[k // 2, k // 2], data_format="NCHW")
        x, wt = put("x", (n, c, h, w)), put("w", (f, c, k, k))
        vecs = [put("scale", (f,), 0.5), put("bias", (f,)), put("mean", (f,)), put("var", (f,), 0.5)]
        z = b.conv(x, wt, **geometry)
        norm, sm, sv, nm, nv = b.batchnorm(z, *vecs, is_test=False)
        act = b.relu(norm)
        y, outs = act, [nm, nv]
        if pool:
            y = b.pool2d(act, "max", [3, 3], [2, 2], [1, 1])
        dy = put("dy", tuple(y.shape()))
        dact = b.pool2d_grad(act, y, dy, "max", [3, 3], [2, 2], [1, 1]) if pool else dy
        dz, dg, db = b.batch_norm_grad(b.relu_grad(dact, act), z, vecs[0], sm, sv)
        dx = b.conv(wt, dz, conv_type="backward_data", output_shape=[n, c, h, w], **geometry)
        dw = b.conv(x, dz, conv_type="backward_filter", output_shape=[f, c, k, k], **geometry)
        outs = [y, dx, dw, dg, db] + outs
        comp = Computation.build_and_compile(DefaultAMDGPUTarget(), b, outputs=outs, conv_layout_nhwc=int(convert))
        for var, raw in data:
            comp.get_tensor(var.id).from_numpy(raw)
        comp.execute()
        results.append([comp.get_tensor(o.id).numpy().astype(np.float64) for o in outs])
    for a, want in zip(*results):
        assert a.shape == want.shape
        assert np.max(np.abs(a - want)) <= 2e-5 * max(1.0, np.max(np.abs(want)))
