"""The channel sums of a training batch norm (cinn_call_hip_channel_statistics, cinn_call_hip_channel_gradient_sums) may be
called first while their stream is captured and without scratch reserved: they then need no partial sums.  Every replay is
checked against float64, with eager work between the replays; a whole training batch norm is captured the same way.

Bound: fp32 sums in rows, splits and their total, far fewer roundings in a row than pixels: 2^-24 sqrt(pixels) + 2^-22 of
the sum of magnitudes; each of the two further steps of a variance rounds once."""
import ctypes

import numpy as np
import pytest

from cinn_amd import _lib, runtime
from cinn_amd.common import Float
from cinn_amd.frontend import NetBuilder

from helpers import compile_only
from test_gpu_backward import from_dev, round_to, to_dev
from test_gpu_gradient_capture import fresh_stream, replays

pytestmark = pytest.mark.gpu

ARGS = [ctypes.c_void_p] + [ctypes.c_int] * 3


# one pixel; channels that are no whole chunk; more chunks than one block's lanes; many splits
@pytest.mark.parametrize("pixels,channels", [(1, 8), (77, 3), (1000, 64), (515, 1100), (30000, 16)])
@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
def test_sums_are_captured_without_an_eager_run(gpu, pixels, channels, dtype):
    rng = np.random.default_rng(pixels)
    x, dy, out = (round_to(rng.standard_normal((pixels, channels)) + m, dtype) for m in (0.5, 0.0, 0.2))
    mean = rng.standard_normal(channels).astype(np.float32)
    lib, clear = _lib.load(), np.full(channels, 7.0, np.float32)
    lib.cinn_call_hip_channel_statistics.argtypes = ARGS + [ctypes.c_void_p]
    lib.cinn_call_hip_channel_gradient_sums.argtypes = ARGS + [ctypes.c_int] * 2 + [ctypes.c_void_p]
    X, DY, OUT = (to_dev(t, dtype) for t in (x, dy, out))
    M, S, T = (runtime.DeviceBuffer.from_numpy(t) for t in (mean, clear, clear))
    x, dy, out = (t.astype(np.float64) for t in (x, dy, out))
    rel = 2.0 ** -24 * np.sqrt(pixels) + 2.0 ** -22

    stream = fresh_stream(lib, 0)
    pods = runtime.pod_args([X, S, T])
    for got in replays(stream, lambda: lib.cinn_call_hip_channel_statistics(pods, 3, pixels, channels, stream.handle), S, clear):
        assert np.all(np.abs(got.numpy() - x.mean(0)) <= 2 * rel * np.abs(x).mean(0))
        assert np.all(np.abs(T.numpy() - x.var(0)) <= 4 * rel * (x * x).mean(0))
        T.copy_from(clear)

    for masked in (0, 1):
        stream = fresh_stream(lib, 0)
        d = np.where(out > 0, dy, 0.0) if masked else dy
        pods, n = runtime.pod_args([DY, X, M] + ([OUT] if masked else []) + [S, T]), 5 + masked
        for got in replays(stream, lambda: lib.cinn_call_hip_channel_gradient_sums(pods, n, pixels, channels, 0x3210, masked, stream.handle),
                           S, clear):
            assert np.all(np.abs(got.numpy() - d.sum(0)) <= 2 * rel * np.abs(d).sum(0))
            assert np.all(np.abs(T.numpy() - (d * (x - mean)).sum(0)) <= 2 * rel * (np.abs(d) * (np.abs(x) + np.abs(mean))).sum(0))
            T.copy_from(clear)


def test_a_training_batch_norm_is_captured_without_an_eager_run(gpu):
    shape, c = [4, 13, 11, 24], 24
    rng = np.random.default_rng(4)
    stream = fresh_stream(_lib.load(), 0)
    b = NetBuilder("batch_norm")
    X, DY = (b.create_input(Float(32), shape, n) for n in ("x", "dy"))
    V = [b.create_input(Float(32), [c], n) for n in ("scale", "bias", "mean", "var")]
    y, mean, var = b.batchnorm(X, *V, is_test=False, data_layout="NHWC")[:3]
    dx = b.batch_norm_grad(DY, X, V[0], mean, var, data_layout="NHWC")[0]
    feeds = {n: rng.standard_normal(shape).astype(np.float32) for n in ("x", "dy")}
    feeds.update({n: rng.uniform(0.5, 1.5, c).astype(np.float32) for n in ("scale", "bias", "mean", "var")})

    def program(stream):
        comp = compile_only(b, [y, dx], stream=stream)
        for n, t in feeds.items():
            comp.get_tensor(n).from_numpy(t)
        return comp
    eager = program(runtime.Stream())
    eager.execute()
    runtime.synchronize()
    want = [eager.get_tensor(o.id).numpy() for o in (y, dx)]
    comp = program(stream)

    class Result(object):  # what `replays` overwrites
        def copy_from(self, t):
            for o in (y, dx):
                comp.get_tensor(o.id).from_numpy(t)
    for _ in replays(stream, comp.execute, Result(), np.zeros(shape, np.float32)):
        for o, w in zip((y, dx), want):
            # sums in another order: a few times 2^-24 of values below 8
            np.testing.assert_allclose(comp.get_tensor(o.id).numpy(), w, rtol=0, atol=1e-5)
