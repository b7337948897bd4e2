"""Projections of one input that an attention reads are one product with joined weights, and a tensor added after a
product with a bias is that product's residual: against the same programs in float64."""
import numpy as np
import pytest

from cinn_amd.common import BFloat16, DefaultAMDGPUTarget, Float, bfloat16_bits_to_float32, float32_to_bfloat16_bits
from cinn_amd.frontend import Computation, NetBuilder

from helpers import run

pytestmark = pytest.mark.gpu

UNIT = {"float32": 2.0 ** -24, "float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}


class _Program(object):
    def __init__(self, dtype, seed):
        self.b, self.dtype, self.rng, self.data = NetBuilder("projections"), dtype, np.random.default_rng(seed), {}
        self.type = BFloat16() if dtype == "bfloat16" else Float(16 if dtype == "float16" else 32)

    def put(self, name, shape, scale=1.0, const=False):
        a = (self.rng.standard_normal(shape) * scale).astype(np.float32)
        raw = float32_to_bfloat16_bits(a) if self.dtype == "bfloat16" else a.astype(self.dtype)
        var = self.b.create_input(self.type, list(shape), name)
        if const:
            var.set_const(True)
        self.data[name] = raw
        return var, self.wide(raw)

    def wide(self, raw):
        return (bfloat16_bits_to_float32(raw) if self.dtype == "bfloat16" else raw).astype(np.float64)

    def run(self, outs, **options):
        comp = Computation.build_and_compile(DefaultAMDGPUTarget(), self.b, outputs=outs, **options)
        for name, raw in self.data.items():
            comp.get_tensor(name).from_numpy(raw)
        comp.execute()
        return [self.wide(comp.get_tensor(o.id).numpy()) for o in outs], [comp.instruction_info(i)[0] for i in range(comp.num_instructions())]


def _close(got, want, unit, factor):
    # roundings of the stored intermediates, relative to the result's size
    assert got.shape == want.shape
    assert np.max(np.abs(got - want)) <= factor * unit * max(1.0, np.max(np.abs(want)))


# one query, a few, several tiles; a cache or none; rows of one 16-byte chunk (16-bit) upwards, odd numbers of heads;
# rows of the product below, at and above 64
@pytest.mark.parametrize("dtype", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("n,t,past,heads,d", [(1, 1, 0, 1, 8), (2, 1, 7, 3, 16), (3, 5, 0, 2, 48), (2, 37, 20, 3, 64), (1, 150, 0, 5, 80)])
@pytest.mark.parametrize("fetched", [False, True])
def test_joined_projections(gpu, n, t, past, heads, d, dtype, fetched):
    p = _Program(dtype, n * 1000 + t + d)
    b, hidden = p.b, heads * d
    x, x64 = p.put("x", (n * t, hidden))
    outs, parts, parts64 = [], [], []
    for e in "qkv":
        w, w64 = p.put("w" + e, (hidden, hidden), hidden ** -0.5, True)
        c, c64 = p.put("c" + e, (hidden,), 0.5, True)
        parts.append(b.transpose(b.reshape(b.add(b.matmul(x, w), c), [n, t, heads, d]), [0, 2, 1, 3]))
        parts64.append((x64 @ w64 + c64).reshape(n, t, heads, d).transpose(0, 2, 1, 3))
    q, k, v = parts
    q64, k64, v64 = parts64
    fetch = [k, v] if fetched else []
    want = [k64, v64] if fetched else []
    if past:
        pk, pk64 = p.put("pk", (n, heads, past, d))
        pv, pv64 = p.put("pv", (n, heads, past, d))
        k, v = b.concat([pk, k], axis=2), b.concat([pv, v], axis=2)
        k64, v64 = np.concatenate([pk64, k64], 2), np.concatenate([pv64, v64], 2)
    s = b.softmax(b.matmul(q, k, False, True, d ** -0.5), axes=[-1])
    y = b.reshape(b.transpose(b.matmul(s, v), [0, 2, 1, 3]), [n * t, hidden])
    got, names = p.run([y] + fetch)
    s64 = np.exp((q64 @ k64.transpose(0, 1, 3, 2)) * d ** -0.5)
    s64 /= s64.sum(-1, keepdims=True)
    want = [(s64 @ v64).transpose(0, 2, 1, 3).reshape(n * t, hidden)] + want
    products = [m for m in names if "matmul" in m or "conv2d" in m]
    assert len(products) == 1 and sum("hip_attention" in m for m in names) == 1, names
    for a, w in zip(got, want):
        _close(a, w, UNIT[dtype], 40 if dtype != "float32" else 40 * 8)


def test_projections_that_differ_stay_apart(gpu):
    """another input for keys and values: three products, same results"""
    p = _Program("float16", 5)
    b, n, t, heads, d = p.b, 2, 9, 2, 32
    x, x64 = p.put("x", (n * t, 64))
    z, z64 = p.put("z", (n * t, 64))
    parts, parts64 = [], []
    for e, (src, src64) in zip("qkv", ((x, x64), (z, z64), (z, z64))):
        w, w64 = p.put("w" + e, (64, 64), 0.125, True)
        c, c64 = p.put("c" + e, (64,), 0.5, True)
        parts.append(b.transpose(b.reshape(b.add(b.matmul(src, w), c), [n, t, heads, d]), [0, 2, 1, 3]))
        parts64.append((src64 @ w64 + c64).reshape(n, t, heads, d).transpose(0, 2, 1, 3))
    y = b.matmul(b.softmax(b.matmul(parts[0], parts[1], False, True, d ** -0.5), axes=[-1]), parts[2])
    (got,), names = p.run([y])
    assert len([m for m in names if "conv2d" in m]) == 3
    s64 = np.exp((parts64[0] @ parts64[1].transpose(0, 1, 3, 2)) * d ** -0.5)
    _close(got, (s64 / s64.sum(-1, keepdims=True)) @ parts64[2], UNIT["float16"], 40)


# rows: the few-row kernel, its limit, the tiled kernels; k no multiple of a step
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("m,k,n", [(1, 256, 16), (64, 256, 40), (65, 72, 24), (130, 768, 768), (515, 192, 136)])
@pytest.mark.parametrize("first", [False, True])
def test_residual_after_a_bias(gpu, m, k, n, dtype, first):
    p = _Program(dtype, m + k + n)
    x, x64 = p.put("x", (m, k))
    w, w64 = p.put("w", (k, n), k ** -0.5, True)
    c, c64 = p.put("c", (n,), 0.5, True)
    r, r64 = p.put("r", (m, n))
    linear = p.b.add(p.b.matmul(x, w), c)
    (got,), names = p.run([p.b.add(r, linear) if first else p.b.add(linear, r)])
    assert len(names) == 1, names
    want = x64 @ w64 + c64 + r64
    # fp32 sums of k terms and one rounding
    bound = UNIT[dtype] * np.abs(want) + k * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64) + np.abs(c64) + np.abs(r64))
    assert np.all(np.abs(got - want) <= 1.01 * bound + 1e-7)


# a layer in training: weights in either order that are no constants; k with and without whole chunks, few and many columns
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("m,k,n", [(2048, 64, 1024), (2051, 768, 1030), (16400, 72, 128), (131, 200, 16384), (262144, 8, 8), (64, 256, 32768)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_bias_of_a_layer_in_training(gpu, m, k, n, dtype, trans_b):
    p = _Program(dtype, m + k + n)
    x, x64 = p.put("x", (m, k))
    w, w64 = p.put("w", (n, k) if trans_b else (k, n), k ** -0.5)
    c, c64 = p.put("c", (n,), 0.5)
    (got,), names = p.run([p.b.add(p.b.matmul(x, w, False, trans_b), c)])
    assert sum("matmul_bias" in e for e in names) == 1 and not any("add" in e for e in names), names
    w64 = w64.T if trans_b else w64
    want = x64 @ w64 + c64
    bound = UNIT[dtype] * np.abs(want) + k * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64) + np.abs(c64))
    assert np.all(np.abs(got - want) <= 1.01 * bound + 1e-7)


# the kernels for one step of K and for 256x256 tiles, which read the 16-bit bias themselves
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("m,k,n", [(16384, 64, 128), (16400, 64, 256), (4096, 192, 3072), (4090, 192, 3080)])
def test_narrow_bias_in_every_epilogue(gpu, m, k, n, dtype):
    test_bias_of_a_layer_in_training(gpu, m, k, n, dtype, False)


# the same with small results and ragged extents, in fp32 too, where K is split and where it is not; the bias has the
# operands' type or fp32
@pytest.mark.parametrize("dtype", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (5, 40, 9), (33, 64, 8), (64, 128, 40), (200, 90, 147), (130, 4100, 136), (256, 512, 512)])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("wide_bias", [False, True])
def test_bias_of_a_small_layer_in_training(gpu, m, k, n, dtype, trans_b, wide_bias):
    import ctypes
    from cinn_amd import _lib, runtime
    from test_gpu_backward import from_dev, round_to, to_dev
    rng = np.random.default_rng(m + k + n)
    x, w = round_to(rng.standard_normal((m, k)), dtype), round_to(rng.standard_normal((n, k) if trans_b else (k, n)) * k ** -0.5, dtype)
    c = round_to(rng.standard_normal(n), "float32" if wide_bias else dtype)
    X, W, C, Y = to_dev(x, dtype), to_dev(w, dtype), to_dev(c, "float32" if wide_bias else dtype), to_dev(np.full((m, n), np.nan), dtype)
    fn = _lib.load().cinn_call_hip_matmul_bias
    fn.argtypes, fn.restype = [ctypes.c_void_p] + [ctypes.c_int] * 5 + [ctypes.c_void_p], None
    fn(runtime.pod_args([X, W, C, Y]), 4, int(trans_b), m, n, k, None)
    runtime.synchronize()
    x64, w64 = x.astype(np.float64), (w.T if trans_b else w).astype(np.float64)
    want  = x64 @ w64 + c
    bound = UNIT[dtype] * np.abs(want) + k * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64) + np.abs(c))
    assert np.all(np.abs(from_dev(Y, dtype) - want) <= 1.01 * bound + 1e-7)


@pytest.mark.parametrize("read_again", [False, True])
def test_bias_of_an_fp32_layer(gpu, read_again):
    """a sum that is a result only comes out of the product; one that is read in the program stays an addition"""
    rng = np.random.default_rng(1)
    b = NetBuilder("fc")
    x, w, c = (b.create_input(Float(32), s, e) for e, s in (("x", [70, 90]), ("w", [90, 50]), ("c", [50])))
    y = b.add(b.matmul(x, w), c)
    out = b.relu(y) if read_again else y
    data = {v: rng.standard_normal(v.shape()).astype(np.float32) for v in (x, w, c)}
    (got,), comp = run(b, data, [out])
    names = [comp.instruction_info(i)[0] for i in range(comp.num_instructions())]
    assert any("matmul_bias" in e for e in names) == (not read_again) and len(names) == 1 + read_again
    want = data[x].astype(np.float64) @ data[w] + data[c]
    np.testing.assert_allclose(got, np.maximum(want, 0) if read_again else want, rtol=1e-4, atol=1e-4)
