"""Linear layers of few rows with the layer norm before them, the gelu behind them or their result in parts as one call
(FuseRowProducts, gemm_rows.hip): rows up to one below, at and above a tile of 16 and at 64; K of one block, of fewer blocks
than wavefronts, of uneven shares and the longest that is normalised; columns that are no multiple of a tile.

Bounds: norm in fp32, rounded once to the type (u = 2^-11 or 2^-8 of a value), a product of k terms with fp32 sums and one
rounding of the result.  |gelu'| < 1.13."""
import ctypes
import math

import numpy as np
import pytest
from scipy.special import erf

from cinn_amd import _lib, runtime

from test_gpu_projections import UNIT, _Program

pytestmark = pytest.mark.gpu


def norm64(x, g, b, eps=1e-5):
    mean, var = x.mean(1, keepdims=True), x.var(1, keepdims=True)
    return (x - mean) / np.sqrt(var + eps) * g + b


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("m,k,n", [(1, 32, 1), (3, 96, 40), (15, 384, 576), (16, 768, 100), (17, 960, 1000), (64, 1280, 50), (8, 576, 2304)])
@pytest.mark.parametrize("norm,gelu,residual", [(True, False, False), (True, True, False), (False, True, False), (True, False, True)])
def test_one_layer(gpu, m, k, n, norm, gelu, residual, dtype):
    p = _Program(dtype, m + k + n)
    b, u = p.b, UNIT[dtype]
    x, x64 = p.put("x", (m, k), 2.0)
    w, w64 = p.put("w", (k, n), k ** -0.5, True)
    c, c64 = p.put("c", (n,), 0.5, True)
    slack = np.zeros((m, k))
    if norm:
        g, g64 = p.put("g", (k,), 1.0, True)
        s, s64 = p.put("s", (k,), 0.1, True)
        x = b.paddle_layer_norm(x, g, s)[0]
        x64 = norm64(x64, g64, s64)
        # E(x^2) - mean^2 in fp32 loses 2^-20 of the variance or so, the value is rounded once
        slack = (u + 2.0 ** -18) * (np.abs(x64) + np.abs(s64))
    y, want = b.add(b.matmul(x, w), c), x64 @ w64 + c64
    bound = slack @ np.abs(w64) + k * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64)) + 2.0 ** -24 * np.abs(c64)
    if gelu:
        y, want, bound = b.gelu(y), want * 0.5 * (1 + erf(want / math.sqrt(2))), 1.13 * bound + 2.0 ** -22 * np.abs(want)
    if residual:
        r, r64 = p.put("r", (m, n))
        y, want = b.add(r, y), want + r64
    (got,), names = p.run([y])
    assert len([e for e in names if "matmul_rows" in e]) == 1 and len(names) == 1, names
    assert np.all(np.abs(got - want) <= 1.01 * (bound + u * np.abs(want)) + 1e-7)


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("fetched", [False, True])
@pytest.mark.parametrize("n,t,past,heads,d", [(2, 1, 7, 8, 48), (1, 1, 100, 12, 64), (3, 5, 0, 4, 64)])
def test_block_of_one_token(gpu, n, t, past, heads, d, fetched, dtype):
    """norm, projections into parts, attention, output layer with its residual, norm, gelu: five calls, against the separate
    operators in float64"""
    p = _Program(dtype, n + past + d)
    b, hidden, u = p.b, heads * d, UNIT[dtype]
    x, x64 = p.put("x", (n * t, hidden))

    def linear(v, v64, name, inp, out):
        w, w64 = p.put(name + "w", (inp, out), inp ** -0.5, True)
        c, c64 = p.put(name + "c", (out,), 0.1, True)
        return b.add(b.matmul(v, w), c), v64 @ w64 + c64

    def norm(v, v64, name):
        g, g64 = p.put(name + "g", (hidden,), 1.0, True)
        s, s64 = p.put(name + "s", (hidden,), 0.1, True)
        return b.paddle_layer_norm(v, g, s)[0], norm64(v64, g64, s64)

    z, z64 = norm(x, x64, "n1")
    parts = []
    for e in "qkv":
        v, v64 = linear(z, z64, e, hidden, hidden)
        parts.append((b.transpose(b.reshape(v, [n, t, heads, d]), [0, 2, 1, 3]), v64.reshape(n, t, heads, d).transpose(0, 2, 1, 3)))
    (q, q64), (k, k64), (v, v64) = parts
    fetch, want = ([k, v], [k64, v64]) if fetched else ([], [])
    if past:
        pk, pk64 = p.put("pk", (n, heads, past, d))
        pv, pv64 = p.put("pv", (n, heads, past, d))
        k, v = b.concat([pk, k], axis=2), b.concat([pv, v], axis=2)
        k64, v64 = np.concatenate([pk64, k64], 2), np.concatenate([pv64, v64], 2)
    o = b.reshape(b.transpose(b.matmul(b.softmax(b.matmul(q, k, False, True, d ** -0.5), axes=[-1]), v), [0, 2, 1, 3]), [n * t, hidden])
    s64 = np.exp((q64 @ k64.transpose(0, 1, 3, 2)) * d ** -0.5)
    o64 = ((s64 / s64.sum(-1, keepdims=True)) @ v64).transpose(0, 2, 1, 3).reshape(n * t, hidden)
    y, y64 = linear(o, o64, "o", hidden, hidden)
    x, x64 = b.add(x, y), x64 + y64
    y, y64 = norm(x, x64, "n2")
    y, y64 = linear(y, y64, "up", hidden, 2 * hidden)
    y, y64 = b.gelu(y), y64 * 0.5 * (1 + erf(y64 / math.sqrt(2)))
    y, y64 = linear(y, y64, "down", 2 * hidden, hidden)
    got, names = p.run([b.add(x, y)] + fetch)
    copies = 2 if fetched and t > 1 else 0  # heads of several tokens are moved
    assert sum("matmul_rows" in e for e in names) == 4 and sum("hip_attention" in e for e in names) == 1, names
    assert len(names) == 5 + (1 if copies else 0), names
    # every intermediate is rounded a handful of times; errors of independent roundings add up in squares
    for g, w in zip(got, [x64 + y64] + want):
        assert np.linalg.norm(g - w) <= 4 * u * np.linalg.norm(w)


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("offset", [0, 2, 8, 14])
def test_operands_at_any_address(gpu, offset, norm):
    """the call takes what the 1x1 convolution it stands for takes: operands that start anywhere in an allocation"""
    m, k, n, rng, u = 9, 96, 40, np.random.default_rng(offset), UNIT["float16"]
    data = [rng.standard_normal(s).astype(np.float16) for s in ((m, k), (n, k), (k,), (k,))]

    def view(a):
        room = runtime.DeviceBuffer((a.size + 8,), "float16")
        room.copy_from(np.r_[np.zeros(offset // 2, np.float16), a.ravel(), np.zeros(8 - offset // 2, np.float16)])
        room.buffer.memory = room.ptr.value + offset
        return room

    x, w, g, s = (view(a) for a in data)
    scale, shift = (runtime.DeviceBuffer.from_numpy(a.astype(np.float32)) for a in (np.ones(n), np.arange(n)))
    out = view(np.zeros((m, n), np.float16))
    inputs = [x, w, scale, shift] + ([g, s] if norm else [])
    operands = 0x3210 | 15 << 16 | (5 << 24 | 4 << 20 if norm else 255 << 20)
    fn = _lib.load().cinn_call_hip_matmul_rows
    fn.restype, fn.argtypes = None, [ctypes.c_void_p] + [ctypes.c_int] * 6 + [ctypes.c_float, ctypes.c_int, ctypes.c_void_p]
    fn(runtime.pod_args(inputs + [out]), len(inputs) + 1, m, n, k, operands, 1, 1e-5, 0, None)
    runtime.synchronize()
    got = out.numpy()[offset // 2:][:m * n].reshape(m, n).astype(np.float64)
    x64, w64, g64, s64 = (a.astype(np.float64) for a in data)
    if norm:
        x64 = norm64(x64, g64, s64)
    want = x64 @ w64.T + np.arange(n)
    bound = k * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T) + u * np.abs(want) + 2.0 ** -24 * n
    if norm:
        bound += (u + 2.0 ** -18) * (np.abs(x64) + np.abs(s64)) @ np.abs(w64).T
    assert np.all(np.abs(got - want) <= 1.01 * bound + 1e-7)
