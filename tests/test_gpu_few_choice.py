"""Which convolutions run on the small tiles whose wavefronts share K (conv_few_mfma.hip), and on which of its tiles: the counters of
launches, not values, which the tiled kernels would give as well.  The values of these layers are checked in
test_gpu_conv_few."""
import ctypes

import numpy as np
import pytest

from cinn_amd import _lib, runtime

from launch_counts import FEW, launches
from test_gpu_conv_few import _conv64, test_layer as check_layer
from test_gpu_few_products import check as check_product
from test_gpu_gemm import call_cublas

pytestmark = pytest.mark.gpu


def convolve(lib, shape, oc, k, stride, dtype, scale):
    """x, w and y of a convolution with or without a layer's scale and shift, channels last"""
    n, h, w, c = shape
    pad = k // 2
    oh, ow = ((e + 2 * pad - k) // stride + 1 for e in (h, w))
    rng = np.random.default_rng(c + oc)
    x, wt = rng.standard_normal(shape).astype(dtype), (rng.standard_normal((oc, k, k, c)) * (c * k * k) ** -0.5).astype(dtype)
    Y = runtime.DeviceBuffer((n, oh, ow, oc), dtype)
    bufs = [runtime.DeviceBuffer.from_numpy(a, d) for a, d in ((x, dtype), (wt, dtype))]
    if scale:
        bufs += [runtime.DeviceBuffer.from_numpy(np.full(oc, v, np.float32)) for v in (1.0, 0.0)] + [Y]
        fn = lib.cinn_call_hip_conv2d_bn_relu
        fn.argtypes, fn.restype = [ctypes.c_void_p] + [ctypes.c_int] * 22 + [ctypes.c_void_p], None
        fn(runtime.pod_args(bufs), 5, 1, 0, n, c, h, w, oc, c, k, k, pad, pad, stride, stride, 1, 1, 1, n, oc, oh, ow, None)
    else:
        bufs += [Y]
        fn = lib.cinn_call_cudnn_conv2d_forward
        fn.argtypes, fn.restype = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_float, ctypes.c_float] + [ctypes.c_int] * 19 + [ctypes.c_void_p], None
        fn(runtime.pod_args(bufs), 3, 1, 1.0, 0.0, n, c, h, w, oc, c, k, k, pad, pad, stride, stride, 1, 1, 1, n, oc, oh, ow, None)
    runtime.synchronize()
    return x, wt, Y.numpy()


# measured on both kernels; a layer's scale and whole tiles of 64 filters have no part in the choice of fp32
@pytest.mark.parametrize("shape,oc,k,stride,dtype,few", [
    ((1, 56, 56, 64), 64, 3, 1, "float32", True), ((1, 14, 14, 256), 256, 3, 1, "float32", True), ((1, 7, 7, 512), 512, 3, 1, "float32", True),
    ((1, 14, 14, 1024), 256, 1, 1, "float32", True), ((8, 28, 28, 128), 256, 3, 2, "float32", True),
    ((5, 42, 44, 480), 64, 1, 1, "float32", True),     # 145 tiles
    ((1, 57, 57, 384), 64, 7, 1, "float32", False),    # 588 steps
    ((8, 12, 22, 416), 192, 3, 1, "float32", False),   # 99 tiles, 117 steps
    ((2, 43, 30, 32), 384, 1, 1, "float32", False),    # 246 tiles of one step
    ((2, 43, 30, 32), 288, 1, 1, "float32", False),
    ((16, 56, 56, 64), 64, 3, 1, "float32", False),    # 784 tiles
    ((1, 56, 56, 64), 64, 3, 1, "float16", True), ((1, 26, 29, 320), 512, 5, 1, "float16", True),
    ((1, 39, 49, 512), 144, 7, 1, "float16", False),   # 392 steps
    ((2, 56, 56, 256), 128, 1, 1, "float16", False),   # 196 tiles
])
@pytest.mark.parametrize("scale", [False, True])
def test_kernel(gpu, shape, oc, k, stride, dtype, few, scale):
    with launches() as count:
        x, w, y = convolve(_lib.load(), shape, oc, k, stride, dtype, scale)
        assert count(*FEW) == few
    # a few pixels of the last image, whose windows reach beyond it or not: as in test_gpu_conv_few
    x, w, rows = x[-1:].astype(np.float64), w.astype(np.float64), slice(0, 3)
    x = x[:, :3 * stride + k]
    want, size = (_conv64(a, b, stride, k // 2, 1)[:, rows] for a, b in ((x, w), (np.abs(x), np.abs(w))))
    unit = 2.0 ** -11 if dtype == "float16" else 2.0 ** -24
    assert np.all(np.abs(y[-1:, rows].astype(np.float64) - want) <= 1.01 * ((w[0].size + 2) * 2.0 ** -24 * size + unit * np.abs(want) + 2.0 ** -25))


# fp32 products with both operands in runs of K; whole tiles of 128 as well
@pytest.mark.parametrize("m,n,k,few", [
    (7, 1792, 1152, True), (92, 576, 3168, True), (1, 1208, 192, True), (64, 60, 2048, True), (1912, 3520, 64, False), (466, 576, 3520, False),
    (128, 128, 128, True), (128, 128, 4096, True), (512, 512, 512, True), (4096, 128, 512, True), (256, 128, 64, True), (768, 768, 768, True),
    (128, 128, 32, False), (256, 3072, 768, False), (1024, 1024, 1024, False)])
def test_product(gpu, m, n, k, few):
    rng = np.random.default_rng(m + n + k)
    a, b = (rng.standard_normal(s).astype(np.float32) for s in ((m, k), (n, k)))
    with launches() as count:
        got = call_cublas(a, b, (m, n), "float32", False, True)
        assert count(*FEW) == few
    check_product(got, a.astype(np.float64), b.astype(np.float64), 1.0, 0.0, k)


def test_every_tile_is_reached(gpu):
    """by the layers whose values are checked; two of them in fp16 and three in fp32 are left to the tiled kernels"""
    layers = [m.args[1] for t in ("test_layer", "test_narrow_layer") for m in getattr(__import__("test_gpu_conv_few"), t).pytestmark
              if m.name == "parametrize" and "," in m.args[0]]
    by_tile, none = {dtype: [0] * len(FEW) for dtype in ("float16", "float32")}, []
    for dtype in by_tile:
        for case in sum(layers, []):
            with launches() as count:
                check_layer(gpu, *case, dtype)
                counts = [count(tile) for tile in FEW]
            assert sum(counts) <= 1
            if not sum(counts):
                none.append((dtype,) + case[:5])
            by_tile[dtype] = [a + b for a, b in zip(by_tile[dtype], counts)]
    assert len(none) == 5, none
    assert all(n > 0 for counts in by_tile.values() for n in counts), by_tile
