"""Gradient of max pooling in 3x3 windows two apart (its own kernel, 16 bytes of channels per thread where a channels-last
tensor has whole chunks) against the oracle.  Inputs are small whole numbers, so windows are full of ties and every sum is
exact: the results are equal."""
import numpy as np
import pytest

from cinn_amd.common import DefaultAMDGPUTarget, Float
from cinn_amd.frontend import Computation, NetBuilder
from oracle import backward as ob

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float16", "float32", "float64"])
@pytest.mark.parametrize("padding", [0, 1, 2])
@pytest.mark.parametrize("n,c,h,w", [(1, 1, 3, 3), (2, 8, 4, 7), (3, 5, 9, 8), (1, 24, 13, 16), (2, 4, 3, 31)])
@pytest.mark.parametrize("fmt", ["NCHW", "NHWC"])
def test_ties_and_edges(gpu, fmt, n, c, h, w, padding, dtype):
    rng = np.random.default_rng(n * c + h * w + padding)
    x = rng.integers(0, 3, (n, c, h, w)).astype(dtype)
    to = (lambda v: np.ascontiguousarray(v.transpose(0, 2, 3, 1))) if fmt == "NHWC" else (lambda v: v)
    back = (lambda v: v.transpose(0, 3, 1, 2)) if fmt == "NHWC" else (lambda v: v)
    t = Float({"float16": 16, "float32": 32, "float64": 64}[dtype])
    b = NetBuilder("pool")
    X = b.create_input(t, list(to(x).shape), "x")
    args = ("max", [3, 3], [2, 2], [padding, padding])
    y = b.pool2d(X, *args, data_format=fmt)
    oh, ow = back(np.empty(y.shape())).shape[2:]
    dy = rng.integers(-4, 5, (n, c, oh, ow)).astype(dtype)
    DY = b.create_input(t, y.shape(), "dy")
    dx = b.pool2d_grad(X, y, DY, *args, data_format=fmt)
    comp = Computation.build_and_compile(DefaultAMDGPUTarget(), b, outputs=[dx])
    comp.get_tensor("x").from_numpy(to(x))
    comp.get_tensor("dy").from_numpy(to(dy))
    comp.execute()
    want = ob.pool2d_backward(x, dy, (3, 3), (2, 2), (padding, padding), "max", True)
    assert np.array_equal(back(comp.get_tensor(dx.id).numpy()).astype(np.float64), np.asarray(want, np.float64))
