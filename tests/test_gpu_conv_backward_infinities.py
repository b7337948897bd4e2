"""Infinite and NaN operands of the convolution gradients.  A tap outside the image is no term of the filter gradient's sum,
so an infinite output gradient does not meet a zero there, and results are inf or NaN exactly where the definition (terms
left out, float64) says so.  The data gradient does so for every output gradient; an infinite or NaN filter value counts
as multiplied by zero where its tap lies outside dy, as it does in the forward convolution: those pixels, near the border,
are NaN."""
import numpy as np
import pytest

from cinn_amd import _lib, runtime

from test_gpu_backward import CONV_ARGTYPES, conv_dims, conv_problem, from_dev, layout, round_to, to_dev, unlayout
from test_gpu_conv_backward_mfma import bound

pytestmark = pytest.mark.gpu

CASES = [
    # n, c, h, w, f, k, stride, pad, dilation, groups
    (2, 16, 9, 8, 24, 3, 1, 1, 1, 1),
    (2, 13, 9, 8, 21, 3, 1, 1, 1, 1),    # copies in either format
    (1, 64, 12, 12, 72, 5, 1, 4, 2, 1),  # dilation
    (2, 24, 13, 10, 40, 3, 2, 1, 1, 1),  # remainder classes
    (2, 8, 12, 11, 16, 1, 2, 0, 1, 1),   # classes without a tap
    (1, 16, 6, 6, 8, 1, 1, 2, 1, 1),     # output pixels that see no pixel of the image
    (12, 64, 14, 14, 64, 3, 1, 1, 1, 1),
]


def gradients(x, w, dy, s, p, d):
    """dx and dw with the terms outside the image left out"""
    k, (oh, ow), (h, w_) = w.shape[2], dy.shape[2:], x.shape[2:]
    dx, dw = np.zeros(x.shape), np.zeros(w.shape)

    def inside(tap, out, size):
        o = np.arange(out)
        i = o * s - p + tap * d
        keep = (i >= 0) & (i < size)
        return o[keep], i[keep]
    for ky in range(k):
        for kx in range(k):
            (oy, iy), (ox, ix) = inside(ky, oh, h), inside(kx, ow, w_)
            if len(oy) == 0 or len(ox) == 0:
                continue
            g = dy[:, :, oy][:, :, :, ox]
            # term by term: a product over all filters (pixels) at once may reorder infinities, but their sum is the same
            dx[np.ix_(range(x.shape[0]), range(x.shape[1]), iy, ix)] += np.einsum("nfyx,fc->ncyx", g, w[:, :, ky, kx])
            dw[:, :, ky, kx] = np.einsum("ncyx,nfyx->fc", x[:, :, iy][:, :, :, ix], g)
    return dx, dw


def check(got, want, scale, terms, dtype):
    got = got.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    finite = np.isfinite(want)
    assert np.array_equal(got[~finite & ~np.isnan(want)], want[~finite & ~np.isnan(want)])
    assert np.all(np.abs(got[finite] - want[finite]) <= bound(want[finite], scale[finite], terms, dtype))


def run(name, fmt, alpha, beta, dims, *tensors):
    fn = getattr(_lib.load(), name)
    fn.argtypes = CONV_ARGTYPES
    fn(runtime.pod_args(tensors), 3, fmt, alpha, beta, *dims, None)
    runtime.synchronize()


@pytest.mark.parametrize("beta", [0.0, 0.5])
@pytest.mark.parametrize("value", [-np.inf, np.nan])
@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("case", CASES)
def test_filter_gradient(gpu, case, dtype, fmt, value, beta):
    n, c, h, w_, f, k, s, p, d, g = case
    x, w, dy = conv_problem(case, dtype)
    dy[0, 1, 0, 0] = value                    # at a corner: outside the image for some taps
    dy[-1, 3, -1, dy.shape[3] // 2] = value   # at the lower edge
    x[0, 2, 0, 0] = value                     # a value of the image itself is a term of every sum it is in
    dw0 = round_to(np.random.default_rng(1).standard_normal(w.shape), dtype)
    X, DY, DW = (to_dev(layout(t, fmt), dtype) for t in (x, dy, dw0))
    run("cinn_call_cudnn_conv2d_backward_filter", fmt, 1.0, beta, conv_dims(case, x, w, dy), X, DY, DW)
    with np.errstate(invalid="ignore"):
        want = gradients(x.astype(np.float64), w, dy.astype(np.float64), s, p, d)[1] + beta * dw0
        scale = gradients(np.abs(x).astype(np.float64), w, np.abs(dy).astype(np.float64), s, p, d)[1] + np.abs(beta * dw0)
    check(unlayout(from_dev(DW, dtype), fmt), want, scale, dy.size / f, dtype)


@pytest.mark.parametrize("beta", [0.0, 0.5])
@pytest.mark.parametrize("value", [-np.inf, np.nan])
@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("filter_too", [False, True])
@pytest.mark.parametrize("case", CASES)
def test_data_gradient(gpu, case, filter_too, dtype, fmt, value, beta):
    n, c, h, w_, f, k, s, p, d, g = case
    x, w, dy = conv_problem(case, dtype)
    dy[0, 2, 0, 0] = dy[-1, 3, -1, dy.shape[3] // 2] = value
    if filter_too:
        w[1, 2, 0, 0] = w[3, 4, -1, k // 2] = value
    dx0 = round_to(np.random.default_rng(1).standard_normal(x.shape), dtype)
    W, DY, DX = (to_dev(layout(t, fmt), dtype) for t in (w, dy, dx0))
    run("cinn_call_cudnn_conv2d_backward_data", fmt, 1.0, beta, conv_dims(case, x, w, dy), W, DY, DX)
    with np.errstate(invalid="ignore"):
        want = gradients(x, w.astype(np.float64), dy.astype(np.float64), s, p, d)[0] + beta * dx0
        scale = gradients(x, np.abs(w).astype(np.float64), np.abs(dy).astype(np.float64), s, p, d)[0] + np.abs(beta * dx0)
    got = unlayout(from_dev(DX, dtype), fmt).copy()
    if filter_too:
        # pixels all of whose taps lie inside: the last tap not above the first output row, the first not below the last
        oh, ow = dy.shape[2:]
        inner = np.zeros(x.shape, bool)
        inner[:, :, max(0, (k - 1) * d - p):max(0, oh * s - p), max(0, (k - 1) * d - p):max(0, ow * s - p)] = True
        assert np.all(np.isin(np.nonzero(np.isnan(got) & ~np.isnan(want) & ~inner)[1], [2, 4]))  # the channels of those values
        got[~inner] = want[~inner]
    check(got, want, scale, f * k * k, dtype)


# Neighbouring taps share what is read (fp16 / bf16, stride 1): positions behind an output row and the last two of every K step have
# a zero in place of dy, and x of a pixel inside the image.  Here a step is a row: its last two positions read the next row's first pixels,
# for the centre tap too, which reaches no padding.
@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_filter_gradient_of_a_pixel_that_meets_no_dy(gpu, dtype, fmt, value):
    case = (8, 64, 4, 60, 8, 3, 1, 1, 1, 1)
    n, c, h, w_, f, k, s, p, d, g = case
    x, w, dy = conv_problem(case, dtype)
    dy[np.abs(dy) < 0.01] = 0.01  # nothing that an infinity would turn to NaN
    dy = round_to(dy, dtype)
    x[1, 5, 2, 0] = x[3, 9, 1, 1] = x[4, 11, 0, w_ - 1] = value
    X, DY, DW = (to_dev(layout(t, fmt), dtype) for t in (x, dy, np.zeros_like(w)))
    run("cinn_call_cudnn_conv2d_backward_filter", fmt, 1.0, 0.0, conv_dims(case, x, w, dy), X, DY, DW)
    with np.errstate(invalid="ignore"):
        want = gradients(x.astype(np.float64), w, dy.astype(np.float64), s, p, d)[1]
        scale = gradients(np.abs(x).astype(np.float64), w, np.abs(dy).astype(np.float64), s, p, d)[1]
    if np.isinf(value):
        assert not np.isnan(want).any() and np.isinf(want[:, 5, 1, 1]).all()
    check(unlayout(from_dev(DW, dtype), fmt), want, scale, dy.size / f, dtype)


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_filter_gradient_without_padding(gpu, dtype):
    """an infinity of x where no padding is: inf or NaN exactly where it is a term"""
    case = (32, 64, 12, 90, 24, 3, 1, 0, 1, 1)
    n, c, h, w_, f, k, s, p, d, g = case
    x, w, dy = conv_problem(case, dtype)
    x[2, 7, 5, w_ - 1] = x[1, 3, 0, 0] = np.inf
    X, DY, DW = (to_dev(layout(t, 1), dtype) for t in (x, dy, np.zeros_like(w)))
    run("cinn_call_cudnn_conv2d_backward_filter", 1, 1.0, 0.0, conv_dims(case, x, w, dy), X, DY, DW)
    with np.errstate(invalid="ignore"):
        want = gradients(x.astype(np.float64), w, dy.astype(np.float64), s, p, d)[1]
        scale = gradients(np.abs(x).astype(np.float64), w, np.abs(dy).astype(np.float64), s, p, d)[1]
    check(unlayout(from_dev(DW, dtype), 1), want, scale, dy.size / f, dtype)
