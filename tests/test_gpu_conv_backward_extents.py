"""Convolution gradients at extents that the matrix-core kernels leave to the gather kernels: an empty batch, and a window that
fits nowhere (no output pixel)."""
import numpy as np
import pytest

from cinn_amd import _lib, runtime

from test_gpu_backward import CONV_ARGTYPES, from_dev, layout, round_to, to_dev, unlayout

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
