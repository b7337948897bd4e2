"""Channels-last convolutions of few output tiles (conv_few_mfma.hip) through cinn_call_hip_conv2d_bn_relu: each of the kernel's
tiles at its edges - one pixel, one below and above a tile of 16, channels that are no multiple of a tile -, K of one step, of
fewer steps than wavefronts and of uneven shares, windows that reach beyond the image, strides and dilations.

Bound: products of k terms with fp32 sums (k 2^-24 of the sum of magnitudes; two more roundings for scale, shift and residual),
and one rounding of the result to its type."""
import ctypes

import numpy as np
import pytest
import torch

from cinn_amd import _lib, runtime
from cinn_amd.common import bfloat16_bits_to_float32, float32_to_bfloat16_bits

pytestmark = pytest.mark.gpu

UNIT = {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8, "float32": 2.0 ** -24}


def _put(a, dtype):
    """the array on the device and its values in float64"""
    a = np.ascontiguousarray(a, np.float32)
    if dtype == "bfloat16":
        bits = float32_to_bfloat16_bits(a)
        return runtime.DeviceBuffer.from_numpy(bits, dtype), bfloat16_bits_to_float32(bits).astype(np.float64)
    a = a.astype(dtype)
    return runtime.DeviceBuffer.from_numpy(a, dtype), a.astype(np.float64)


def _conv64(x, w, stride, pad, dil):
    y = torch.nn.functional.conv2d(torch.from_numpy(x).permute(0, 3, 1, 2), torch.from_numpy(w).permute(0, 3, 1, 2), None, stride, pad, dil)
    return y.permute(0, 2, 3, 1).numpy()


@pytest.mark.parametrize("dtype", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("n,h,w,c,oc,k,stride,pad,dil,residual,relu", [
    (1, 1, 1, 128, 4, 1, 1, 0, 1, False, False),     # one pixel
    (1, 3, 5, 128, 20, 1, 1, 0, 1, True, True),      # 15 pixels, more wavefronts than steps
    (1, 1, 17, 64, 16, 1, 1, 0, 1, False, True),     # one K step (two in fp32)
    (1, 4, 4, 192, 100, 3, 1, 1, 1, False, True),    # every pixel's window reaches beyond the image; 27 steps
    (1, 17, 1, 128, 36, 3, 2, 1, 1, True, False),    # one column
    (2, 7, 7, 512, 260, 3, 1, 1, 1, True, True),     # a long K
    (1, 14, 13, 320, 132, 1, 1, 0, 1, False, False), # eleven and a half tile rows of 16
    (1, 28, 28, 128, 132, 3, 1, 1, 1, False, True),
    (3, 9, 11, 64, 68, 3, 1, 2, 2, False, True),     # dilated, images within a tile
    (2, 15, 15, 64, 72, 5, 3, 2, 1, True, False),
    (1, 56, 56, 64, 64, 1, 1, 0, 1, True, True),     # several blocks on a CU
    (5, 28, 28, 64, 100, 3, 1, 1, 1, True, True),    # 62 x 2 tiles of 64 x 64
    (1, 10, 12, 64, 512, 2, 2, 0, 1, False, False),  # windows that lie inside everywhere
])
def test_layer(gpu, n, h, w, c, oc, k, stride, pad, dil, residual, relu, dtype):
    rng = np.random.default_rng(h * w + c + oc)
    oh, ow = ((e + 2 * pad - ((k - 1) * dil + 1)) // stride + 1 for e in (h, w))
    X, x64 = _put(rng.standard_normal((n, h, w, c)), dtype)
    W, w64 = _put(rng.standard_normal((oc, k, k, c)) * (c * k * k) ** -0.5, dtype)
    S, s64 = _put(rng.uniform(0.5, 1.5, oc), "float32")
    T, t64 = _put(rng.standard_normal(oc), "float32")
    bufs = [X, W, S, T]
    want = _conv64(x64, w64, stride, pad, dil) * s64 + t64
    size = _conv64(np.abs(x64), np.abs(w64), stride, pad, dil) * s64 + np.abs(t64)
    if residual:
        R, r64 = _put(rng.standard_normal((n, oh, ow, oc)), dtype)
        bufs.append(R)
        want, size = want + r64, size + np.abs(r64)
    Y = runtime.DeviceBuffer((n, oh, ow, oc), dtype)
    bufs.append(Y)
    fn = _lib.load().cinn_call_hip_conv2d_bn_relu
    fn.argtypes, fn.restype = [ctypes.c_void_p] + [ctypes.c_int] * 22 + [ctypes.c_void_p], None
    fn(runtime.pod_args(bufs), len(bufs), 1, int(relu), n, c, h, w, oc, c, k, k, pad, pad, stride, stride, dil, dil, 1, n, oc, oh, ow, None)
    runtime.synchronize()
    got = bfloat16_bits_to_float32(Y.numpy()) if dtype == "bfloat16" else Y.numpy()
    want = np.maximum(want, 0) if relu else want
    bound = (c * k * k + 2) * 2.0 ** -24 * size + UNIT[dtype] * np.abs(want) + 2.0 ** -25
    assert np.all(np.abs(got.astype(np.float64) - want) <= 1.01 * bound)


# more than 128 tiles of 64x64 whose columns are mostly padding: one group of four channels, one below and above a tile of 16 and
# of 64, a split that the tiled kernels would have, a K of one step
@pytest.mark.parametrize("dtype", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("n,h,w,c,oc,k,stride,pad,dil,residual,relu", [
    (9, 31, 37, 128, 4, 3, 1, 1, 1, False, False),
    (3, 57, 56, 64, 12, 5, 1, 2, 1, True, True),
    (5, 91, 97, 64, 20, 1, 1, 0, 1, False, True),
    (2, 70, 71, 192, 68, 3, 1, 1, 1, True, False),
    (1, 129, 127, 64, 16, 7, 2, 3, 1, False, True),
    (7, 40, 41, 320, 60, 3, 1, 1, 1, False, False),
])
def test_narrow_layer(gpu, n, h, w, c, oc, k, stride, pad, dil, residual, relu, dtype):
    test_layer(gpu, n, h, w, c, oc, k, stride, pad, dil, residual, relu, dtype)


@pytest.mark.parametrize("shape,oc,k", [((1, 1, 1, 32), 4, 1), ((2, 13, 11, 96), 36, 3), ((8, 35, 41, 96), 200, 3), ((4, 33, 31, 160), 12, 5)])
def test_fp32_without_a_scale(gpu, shape, oc, k):
    from cinn_amd.common import DefaultAMDGPUTarget, Float
    from cinn_amd.frontend import Computation, NetBuilder
    rng = np.random.default_rng(oc)
    x = rng.standard_normal(shape).astype(np.float32)
    w = (rng.standard_normal((oc, k, k, shape[3])) * 0.05).astype(np.float32)
    b = NetBuilder("plain")
    X, W = b.create_input(Float(32), list(x.shape), "x"), b.create_input(Float(32), list(w.shape), "w")
    y = b.conv2d(X, W, [2, 2], [k // 2] * 2, data_format="NHWC")
    comp = Computation.build_and_compile(DefaultAMDGPUTarget(), b, outputs=[y])
    comp.get_tensor("x").from_numpy(x)
    comp.get_tensor("w").from_numpy(w)
    comp.execute()
    got = comp.get_tensor(y.id).numpy().astype(np.float64)
    x, w = x.astype(np.float64), w.astype(np.float64)
    want, size = _conv64(x, w, 2, k // 2, 1), _conv64(np.abs(x), np.abs(w), 2, k // 2, 1)
    assert np.all(np.abs(got - want) <= (shape[3] * k * k + 2) * 2.0 ** -24 * size + 2.0 ** -25)
