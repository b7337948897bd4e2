"""The first call of a convolution gradient, or of a ragged product, may be made while its stream is being captured and
without scratch reserved for it: a gradient then runs in gather form (which needs none), a product keeps its K whole.
Some scratch (room for the copies, none for a split): the data gradient's convolution stays whole.  Every replay is
checked against the oracle, with eager work between the replays.

Bounds as in test_gpu_conv_backward_mfma.py and test_gpu_gemm_flex.py."""
import ctypes

import numpy as np
import pytest

from oracle import backward as ob
from cinn_amd import _lib, runtime

from test_gpu_backward import CONV_ARGTYPES, conv_dims, conv_problem, from_dev, layout, to_dev, unlayout
from test_gpu_conv_backward_mfma import bound

pytestmark = pytest.mark.gpu


def fresh_stream(lib, copies_bytes):
    """a stream whose handle has no scratch of an earlier owner, with the page of zeros and room for copies"""
    stream = runtime.Stream()
    lib.cinn_hip_scratch_release_stream.argtypes = [ctypes.c_void_p]
    lib.cinn_hip_scratch_reserve.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_size_t]
    assert lib.cinn_hip_scratch_release_stream(stream.handle) == 0
    if copies_bytes:
        assert lib.cinn_hip_scratch_reserve(stream.handle, 0, copies_bytes) == 0
    return stream


def replays(stream, call, out, clear):
    """what three replays of a captured call give, with `out` overwritten before each"""
    hip = ctypes.CDLL("libamdhip64.so")
    graph, graph_exec = ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamBeginCapture(stream.handle, 1) == 0  # hipStreamCaptureModeThreadLocal
    call()
    assert hip.hipStreamEndCapture(stream.handle, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(graph_exec), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(3):
        out.copy_from(clear)
        runtime.synchronize()
        assert hip.hipGraphLaunch(graph_exec, stream.handle) == 0
        stream.synchronize()
        yield out
    hip.hipGraphExecDestroy(graph_exec)
    hip.hipGraphDestroy(graph)


@pytest.mark.parametrize("copies_bytes", [0, 1 << 22])
@pytest.mark.parametrize("dtype", ["float32", "float16"])
@pytest.mark.parametrize("case", [(2, 64, 9, 8, 128, 3, 1, 1, 1, 1), (1, 128, 12, 12, 1024, 1, 1, 0, 1, 1),
                                  (3, 24, 13, 10, 40, 3, 2, 1, 1, 1)])
def test_gradients_are_captured_without_an_eager_run(gpu, case, dtype, copies_bytes):
    n, c, h, w_, f, k, s, p, d, g = case
    fmt = 0
    x, w, dy = conv_problem(case, dtype)
    lib = _lib.load()
    stream = fresh_stream(lib, copies_bytes)
    X, W, DY, DX, DW = (to_dev(layout(t, fmt), dtype) for t in (x, w, dy, np.zeros_like(x), np.zeros_like(w)))
    dims, geometry = conv_dims(case, x, w, dy), ((s, s), (p, p), (d, d), g)
    for name, args, out, shape, oracle, a, b, terms in (
            ("cinn_call_cudnn_conv2d_backward_data", [W, DY, DX], DX, x.shape, ob.conv2d_backward_data, w, dy, f * k * k),
            ("cinn_call_cudnn_conv2d_backward_filter", [X, DY, DW], DW, w.shape, ob.conv2d_backward_filter, x, dy, dy.size / f)):
        call = getattr(lib, name)
        call.argtypes = CONV_ARGTYPES
        pods = runtime.pod_args(args)
        want, scale = oracle(a, b, shape, *geometry), oracle(np.abs(a), np.abs(b), shape, *geometry)
        clear = layout(np.zeros(shape, dtype), fmt)
        for got in replays(stream, lambda: call(pods, 3, fmt, 1.0, 0.0, *dims, stream.handle), out, clear):
            assert np.all(np.abs(unlayout(from_dev(got, dtype), fmt) - want) <= bound(want, scale, terms, dtype))


@pytest.mark.parametrize("dtype", ["float32", "float16"])
def test_a_ragged_product_is_captured_without_an_eager_run(gpu, dtype):
    m, n, k = 70, 90, 3001  # eager: K split
    rng = np.random.default_rng(9)
    a, b = rng.standard_normal((m, k)).astype(dtype), rng.standard_normal((k, n)).astype(dtype)
    lib = _lib.load()
    stream = fresh_stream(lib, 0)
    lib.cinn_call_cublas.argtypes = ([ctypes.c_void_p, ctypes.c_int] + [ctypes.c_bool] * 3 + [ctypes.c_float] * 2 +
                                     [ctypes.c_int] * 8 + [ctypes.c_void_p])
    A, B, C = to_dev(a, dtype), to_dev(b, dtype), to_dev(np.zeros((m, n), dtype), dtype)
    pods = runtime.pod_args([A, B, C])
    want, scale = a.astype(np.float64) @ b.astype(np.float64), np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    for got in replays(stream, lambda: lib.cinn_call_cublas(pods, 3, False, False, False, 1.0, 0.0, 1, 1, m, k, 1, 1, k, n, stream.handle),
                       C, np.zeros((m, n), dtype)):
        assert np.all(np.abs(from_dev(got, dtype) - want) <= bound(want, scale, k, dtype))
