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
