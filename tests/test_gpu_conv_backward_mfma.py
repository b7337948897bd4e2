"""Convolution gradients on the matrix cores (conv_backward_mfma.hip) at the edges of their tiles, K steps, chunks and
remainder classes, in both tensor formats, against the numpy oracle.

Bound: operands are exact in the type and sums are fp32 (2^-24 of the sum of magnitudes per rounding, far fewer roundings
in a row than terms: 2^-24 sqrt(terms) + 2^-22 covers them); a 16-bit result is rounded once (half an ulp of itself), also
where beta times what was there is added and where it is copied back to NCHW."""
import ctypes

import numpy as np
import pytest

from oracle import backward as ob
from cinn_amd import _lib, runtime

from test_gpu_backward import CONV_ARGTYPES, conv_dims, conv_problem, from_dev, layout, round_to, to_dev, unlayout

pytestmark = pytest.mark.gpu

CASES = [
    # n, c, h, w, f, k, stride, pad, dilation, groups
    (1, 1, 1, 1, 1, 1, 1, 0, 1, 1),
    (1, 3, 5, 70, 7, 3, 1, 1, 1, 1),     # an image's channels, one odd filter count
    (2, 64, 9, 8, 64, 3, 1, 1, 1, 1),    # whole chunks: no copies in NHWC
    (2, 65, 7, 9, 129, 3, 1, 1, 1, 1),   # one above the tiles
    (1, 40, 11, 13, 24, 5, 1, 2, 2, 1),  # dilation
    (1, 16, 6, 6, 8, 1, 1, 2, 1, 1),     # more padding than the window covers: the class kernel at stride 1
    (3, 24, 13, 10, 40, 3, 2, 1, 1, 1),  # four classes of different extents
    (2, 8, 9, 9, 136, 1, 2, 0, 1, 1),    # three classes without a tap
    (1, 9, 17, 16, 12, 7, 3, 3, 1, 1),
    (1, 16, 2, 2, 16, 3, 2, 1, 1, 1),    # one output pixel
    (1, 16, 19, 22, 24, 3, 5, 1, 1, 1),  # sixteen classes without a tap among those that have one
    (40, 72, 10, 11, 200, 3, 1, 1, 1, 1),  # many K steps, split
]


def bound(want, scale, terms, dtype):
    ulp = {"float32": 2.0 ** -24, "float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}[dtype]
    return (2.0 ** -24 * np.sqrt(terms) + 2.0 ** -22) * scale + ulp * np.abs(want) + 2.0 ** -24


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("case", CASES)
def test_gradients(gpu, case, dtype, fmt):
    n, c, h, w_, f, k, s, p, d, g = case
    x, w, dy = conv_problem(case, dtype)
    lib = _lib.load()
    lib.cinn_call_cudnn_conv2d_backward_data.argtypes = CONV_ARGTYPES
    lib.cinn_call_cudnn_conv2d_backward_filter.argtypes = CONV_ARGTYPES
    X, W, DY = (to_dev(layout(t, fmt), dtype) for t in (x, w, dy))
    nan_x, nan_w = np.full_like(x, np.nan), np.full_like(w, np.nan)  # beta = 0 does not read what was there
    DX, DW = to_dev(layout(nan_x, fmt), dtype), to_dev(layout(nan_w, fmt), dtype)
    dims = conv_dims(case, x, w, dy)
    lib.cinn_call_cudnn_conv2d_backward_data(runtime.pod_args([W, DY, DX]), 3, fmt, 1.0, 0.0, *dims, None)
    lib.cinn_call_cudnn_conv2d_backward_filter(runtime.pod_args([X, DY, DW]), 3, fmt, 1.0, 0.0, *dims, None)
    runtime.synchronize()
    geometry = ((s, s), (p, p), (d, d), g)
    want, scale = (ob.conv2d_backward_data(q, r, x.shape, *geometry) for q, r in ((w, dy), (np.abs(w), np.abs(dy))))
    assert np.all(np.abs(unlayout(from_dev(DX, dtype), fmt) - want) <= bound(want, scale, f * k * k, dtype))
    want, scale = (ob.conv2d_backward_filter(q, r, w.shape, *geometry) for q, r in ((x, dy), (np.abs(x), np.abs(dy))))
    assert np.all(np.abs(unlayout(from_dev(DW, dtype), fmt) - want) <= bound(want, scale, dy.size / f, dtype))


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("dtype", ["float32", "float16"])
@pytest.mark.parametrize("case", [CASES[2], CASES[3], CASES[6], CASES[7]])
def test_alpha_beta(gpu, case, dtype, fmt):
    n, c, h, w_, f, k, s, p, d, g = case
    x, w, dy = conv_problem(case, dtype)
    rng = np.random.default_rng(3)
    dx0, dw0 = (round_to(rng.standard_normal(t.shape), dtype) for t in (x, w))
    lib = _lib.load()
    X, W, DY, DX, DW = (to_dev(layout(t, fmt), dtype) for t in (x, w, dy, dx0, dw0))
    dims = conv_dims(case, x, w, dy)
    lib.cinn_call_cudnn_conv2d_backward_data.argtypes = CONV_ARGTYPES
    lib.cinn_call_cudnn_conv2d_backward_filter.argtypes = CONV_ARGTYPES
    lib.cinn_call_cudnn_conv2d_backward_data(runtime.pod_args([W, DY, DX]), 3, fmt, 0.5, 2.0, *dims, None)
    lib.cinn_call_cudnn_conv2d_backward_filter(runtime.pod_args([X, DY, DW]), 3, fmt, -1.5, 0.25, *dims, None)
    runtime.synchronize()
    geometry = ((s, s), (p, p), (d, d), g)
    grad, scale = (ob.conv2d_backward_data(q, r, x.shape, *geometry) for q, r in ((w, dy), (np.abs(w), np.abs(dy))))
    want = 0.5 * grad + 2.0 * dx0
    err  = np.abs(unlayout(from_dev(DX, dtype), fmt) - want)
    assert np.all(err <= bound(want, 0.5 * scale + 2.0 * np.abs(dx0), f * k * k, dtype))
    grad, scale = (ob.conv2d_backward_filter(q, r, w.shape, *geometry) for q, r in ((x, dy), (np.abs(x), np.abs(dy))))
    want = -1.5 * grad + 0.25 * dw0
    err  = np.abs(unlayout(from_dev(DW, dtype), fmt) - want)
    assert np.all(err <= bound(want, 1.5 * scale + 0.25 * np.abs(dw0), dy.size / f, dtype))


@pytest.mark.parametrize("fmt", [0, 1])
def test_scratch_of_a_large_stride(gpu, fmt):
    """a data gradient keeps the filter once, not once for every remainder class"""
    case = (1, 64, 33, 30, 128, 1, 16, 0, 1, 1)
    x, w, dy = conv_problem(case, "float16")
    lib, stream = _lib.load(), runtime.Stream()
    lib.cinn_call_cudnn_conv2d_backward_data.argtypes = CONV_ARGTYPES
    lib.cinn_hip_scratch_release_stream.argtypes = [ctypes.c_void_p]
    assert lib.cinn_hip_scratch_release_stream(stream.handle) == 0
    W, DY, DX = (to_dev(layout(t, fmt), "float16") for t in (w, dy, np.full_like(x, np.nan)))
    lib.cinn_call_cudnn_conv2d_backward_data(runtime.pod_args([W, DY, DX]), 3, fmt, 1.0, 0.0, *conv_dims(case, x, w, dy), stream.handle)
    stream.synchronize()
    capacity = ctypes.c_size_t(0)
    assert lib.cinn_hip_scratch_info(stream.handle, None, ctypes.byref(capacity), None) == 0
    copies = 2 * (dy.size + x.size) if fmt == 0 else 0
    assert capacity.value <= copies + 2 * w.size + 3 * 256
    want, scale = (ob.conv2d_backward_data(q, r, x.shape, (16, 16), (0, 0), (1, 1), 1) for q, r in ((w, dy), (np.abs(w), np.abs(dy))))
    assert np.all(np.abs(unlayout(from_dev(DX, "float16"), fmt) - want) <= bound(want, scale, 128, "float16"))


@pytest.mark.parametrize("case,limit", [((1, 64, 28, 28, 64, 3, 1, 1, 1, 1), 1.3e-7), ((16, 64, 28, 28, 64, 3, 1, 1, 1, 1), 1.8e-7),
                                        ((2, 128, 14, 14, 96, 3, 1, 1, 1, 1), 1.3e-7)])
def test_rounding_of_the_fp32_filter_gradient(gpu, case, limit):
    """fp32 sums over 392 to 12544 pixels, relative 2-norm of the error.  A chain of n terms of random sign is off by about
    2^-24 * 0.3 * sqrt(n): 0.7e-7 for the sixteen of a part, and as much for up to sixteen steps and planes on top of it;
    1.3e-7 is a third above that, as one chain the sums are off by more than 2.2e-7.  12544 pixels have longer chains of
    steps."""
    n, c, h, w_, f, k, s, p, d, g = case
    x, w, dy = conv_problem(case, "float32")
    lib = _lib.load()
    lib.cinn_call_cudnn_conv2d_backward_filter.argtypes = CONV_ARGTYPES
    X, DY, DW = (to_dev(layout(t, 1), "float32") for t in (x, dy, w))
    lib.cinn_call_cudnn_conv2d_backward_filter(runtime.pod_args([X, DY, DW]), 3, 1, 1.0, 0.0, *conv_dims(case, x, w, dy), None)
    runtime.synchronize()
    want = ob.conv2d_backward_filter(x, dy, w.shape, (s, s), (p, p), (d, d), g)
    got = unlayout(from_dev(DW, "float32"), 1).astype(np.float64)
    assert np.linalg.norm(got - want) <= limit * np.linalg.norm(want)
