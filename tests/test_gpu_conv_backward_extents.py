"""Convolution gradients at extents that the matrix-core kernels leave to the gather kernels: an empty batch, a window that
fits nowhere (no output pixel), and negative paddings, which cut the image's border off.  Results against the gradients'
definition in float64; bound as in test_gpu_conv_backward_mfma.py."""
import numpy as np
import pytest

from oracle import backward as ob
from cinn_amd import _lib, runtime

from test_gpu_backward import CONV_ARGTYPES, from_dev, layout, round_to, to_dev, unlayout
from test_gpu_conv_backward_mfma import bound

pytestmark = pytest.mark.gpu


def call(name, fmt, beta, dims, *tensors):
    fn = getattr(_lib.load(), name)
    fn.argtypes = CONV_ARGTYPES
    fn(runtime.pod_args(tensors), 3, fmt, 1.0, beta, *dims, None)
    runtime.synchronize()


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("dtype", ["float32", "float16"])
def test_an_empty_sum_is_zero(gpu, dtype, fmt):
    rng = np.random.default_rng(0)
    w0 = round_to(rng.standard_normal((16, 8, 5, 5)), dtype)
    some = to_dev(np.zeros((1, 16, 4, 4)), dtype)  # an empty tensor's memory: nothing is read of it
    for beta in (0.0, 0.5):
        # no image
        DW = to_dev(layout(w0 if beta else np.full_like(w0, np.nan), fmt), dtype)
        call("cinn_call_cudnn_conv2d_backward_filter", fmt, beta, (0, 8, 9, 9, 16, 8, 5, 5, 2, 2, 1, 1, 1, 1, 1, 0, 16, 9, 9), some, some, DW)
        assert np.array_equal(unlayout(from_dev(DW, dtype), fmt), round_to(beta * w0, dtype))
        # a 5x5 window on 4x4 pixels without padding: no output pixel
        dims = (3, 8, 4, 4, 16, 8, 5, 5, 0, 0, 1, 1, 1, 1, 1, 3, 16, 0, 0)
        x0 = round_to(rng.standard_normal((3, 8, 4, 4)), dtype)
        X, W = to_dev(layout(x0, fmt), dtype), to_dev(layout(w0, fmt), dtype)
        DX, DW = (to_dev(layout(t if beta else np.full_like(t, np.nan), fmt), dtype) for t in (x0, w0))
        call("cinn_call_cudnn_conv2d_backward_filter", fmt, beta, dims, X, some, DW)
        call("cinn_call_cudnn_conv2d_backward_data", fmt, beta, dims, W, some, DX)
        assert np.array_equal(unlayout(from_dev(DW, dtype), fmt), round_to(beta * w0, dtype))
        assert np.array_equal(unlayout(from_dev(DX, dtype), fmt), round_to(beta * x0, dtype))


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("dtype", ["float32", "float16"])
@pytest.mark.parametrize("stride", [1, 2, 3])
@pytest.mark.parametrize("ph,pw", [(-1, 0), (0, -2), (-1, -1), (1, -1)])
def test_negative_padding(gpu, ph, pw, stride, dtype, fmt):
    n, c, h, w_, f, k = 2, 8, 13, 12, 16, 3
    rng = np.random.default_rng(stride)
    oh, ow = (h + 2 * ph - k) // stride + 1, (w_ + 2 * pw - k) // stride + 1
    x = round_to(rng.standard_normal((n, c, h, w_)), dtype)
    w = round_to(rng.standard_normal((f, c, k, k)), dtype)
    dy = round_to(rng.standard_normal((n, f, oh, ow)), dtype)
    X, W, DY = (to_dev(layout(t, fmt), dtype) for t in (x, w, dy))
    DX, DW = to_dev(layout(np.full_like(x, np.nan), fmt), dtype), to_dev(layout(np.full_like(w, np.nan), fmt), dtype)
    dims = (n, c, h, w_, f, c, k, k, ph, pw, stride, stride, 1, 1, 1, n, f, oh, ow)
    call("cinn_call_cudnn_conv2d_backward_data", fmt, 0.0, dims, W, DY, DX)
    call("cinn_call_cudnn_conv2d_backward_filter", fmt, 0.0, dims, X, DY, DW)
    cut = (slice(None), slice(None), slice(max(0, -ph), h - max(0, -ph)), slice(max(0, -pw), w_ - max(0, -pw)))
    geometry = ((stride, stride), (max(0, ph), max(0, pw)), (1, 1), 1)
    for out, other, shape, terms, fn, got in ((dy, w, x[cut].shape, f * k * k, ob.conv2d_backward_data, DX),
                                              (dy, x[cut], w.shape, dy.size / f, ob.conv2d_backward_filter, DW)):
        pair = (other, out)
        want, scale = (fn(*(g(t) for t in pair), shape, *geometry) for g in (lambda t: t, np.abs))
        result = unlayout(from_dev(got, dtype), fmt)
        if got is DX:  # what is cut off has no gradient
            kept = result[cut].copy()
            result[cut] = 0.0
            assert not result.any()
            result = kept
        assert np.all(np.abs(result - want) <= bound(want, scale, terms, dtype))
