"""Filter gradients whose neighbouring taps share what is read (conv_filter_taps_kernel) where positions, steps and tiles end:
output rows as long as a K step's own positions and one more or less, a single column, rows shorter than the taps, channel
and filter counts beside a tile's, windows that are no multiple of three taps, and one to many splits of K; against the numpy
oracle with the bound of test_gpu_conv_backward_mfma.py."""
import numpy as np
import pytest

from oracle import backward as ob
from cinn_amd import _lib, runtime

from test_gpu_backward import CONV_ARGTYPES, conv_dims, conv_problem, from_dev, layout, to_dev, unlayout
from test_gpu_conv_backward_mfma import bound

pytestmark = pytest.mark.gpu

CASES = [
    # n, c, h, w, f, k, stride, pad, dilation, groups
    (1, 64, 3, 59, 64, 3, 1, 1, 1, 1),
    (2, 64, 3, 60, 64, 3, 1, 1, 1, 1),   # an output row and the positions behind it are one step
    (2, 64, 5, 61, 63, 3, 1, 1, 1, 1),
    (3, 64, 4, 124, 8, 3, 1, 1, 1, 1),
    (3, 64, 9, 3, 64, 3, 1, 0, 1, 1),    # one output column
    (5, 64, 1, 2, 64, 3, 1, 2, 1, 1),    # padding on more sides than pixels
    (2, 72, 11, 17, 65, 3, 1, 1, 1, 1),
    (2, 128, 8, 23, 136, 5, 1, 2, 1, 1),
    (1, 64, 13, 20, 40, 7, 1, 3, 1, 1),
    (1, 64, 7, 9, 64, 4, 1, 1, 1, 1),
    (16, 64, 28, 29, 64, 3, 1, 1, 1, 1),
]
# The above are the shapes where both kernels' ends meet; by the estimate most of them run on conv_filter_kernel.  These run on
# conv_filter_taps_kernel:
TAKEN = [
    (8, 56, 4, 59, 8, 3, 1, 1, 1, 1),
    (8, 64, 4, 60, 8, 3, 1, 1, 1, 1),     # an output row and the positions behind it are one step
    (1, 64, 7, 61, 8, 3, 1, 1, 1, 1),
    (1, 64, 3, 124, 136, 3, 1, 1, 1, 1),
    (1, 56, 3, 1, 136, 3, 1, 1, 1, 1),    # one output column
    (1, 56, 3, 1, 136, 3, 1, 2, 1, 1),    # padding on more sides than pixels
    (1, 65, 3, 17, 136, 3, 1, 1, 1, 1),
    (5, 61, 5, 16, 13, 3, 1, 1, 1, 1),
    (2, 128, 8, 23, 136, 5, 1, 2, 1, 1),
    (1, 64, 4, 17, 129, 7, 1, 3, 1, 1),
    (1, 64, 7, 12, 129, 4, 1, 2, 1, 1),
    (32, 72, 28, 17, 40, 3, 1, 1, 1, 1),  # 40 splits
]


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("case", CASES + TAKEN)
def test_filter_gradient(gpu, case, dtype, fmt):
    n, c, h, w_, f, k, s, p, d, g = case
    x, w, dy = conv_problem(case, dtype)
    lib = _lib.load()
    lib.cinn_call_cudnn_conv2d_backward_filter.argtypes = CONV_ARGTYPES
    X, DY = (to_dev(layout(t, fmt), dtype) for t in (x, dy))
    DW = to_dev(layout(np.full_like(w, np.nan), fmt), dtype)
    lib.cinn_call_cudnn_conv2d_backward_filter(runtime.pod_args([X, DY, DW]), 3, fmt, 1.0, 0.0, *conv_dims(case, x, w, dy), None)
    runtime.synchronize()
    want, scale = (ob.conv2d_backward_filter(q, r, w.shape, (s, s), (p, p), (d, d), g) for q, r in ((x, dy), (np.abs(x), np.abs(dy))))
    assert np.all(np.abs(unlayout(from_dev(DW, dtype), fmt) - want) <= bound(want, scale, dy.size / f, dtype))


def test_row_longer_than_24_bits(gpu):
    """one row of more than 2^23 pixels (fp16, channels last, 1x3), which the neighbouring taps would read less of: its last pixels
    and a few of its first, the others zero"""
    n, c, f, w_ = 1, 48, 8, (1 << 23) + 9
    rng = np.random.default_rng(0)
    x, dy = np.zeros((w_, c), np.float16), np.zeros((w_, f), np.float16)
    at = np.r_[0:8, w_ - 24:w_]
    for t in (x, dy):
        t[at] = rng.standard_normal((len(at), t.shape[1]))
    dims = (n, c, 1, w_, f, c, 1, 3, 0, 1, 1, 1, 1, 1, 1, n, f, 1, w_)
    lib = _lib.load()
    lib.cinn_call_cudnn_conv2d_backward_filter.argtypes = CONV_ARGTYPES
    X, DY = (to_dev(t.reshape(n, 1, w_, -1), "float16") for t in (x, dy))
    DW = to_dev(np.full((f, 1, 3, c), np.nan, np.float16), "float16")
    lib.cinn_call_cudnn_conv2d_backward_filter(runtime.pod_args([X, DY, DW]), 3, 1, 1.0, 0.0, *dims, None)
    runtime.synchronize()
    got = from_dev(DW, "float16")
    for tap in range(3):
        rows = at[(at + tap - 1 >= 0) & (at + tap - 1 < w_)]
        a, b = dy[rows].astype(np.float64), x[rows + tap - 1].astype(np.float64)
        assert np.all(np.abs(got[:, 0, tap] - a.T @ b) <= bound(a.T @ b, np.abs(a).T @ np.abs(b), len(at), "float16"))
