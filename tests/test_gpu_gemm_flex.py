"""Products that run on the register-staged MFMA kernel (gemm_flex.hip), at the edges of its tiles, K steps and chunks:
one row, one column, one k; extents one below and above 64 and 128; operands whose rows are no multiple of a 16-byte
chunk; enough tiles for the 128x128 forms; few tiles and a long K for the split reduction.

Bounds: the inputs are exact in the type, sums are fp32: every rounding of a sum of k products is at most 2^-24 of the
sum of their magnitudes, and a blocked sum has far fewer of them in a row than k, so 2^-24 * sqrt(k) + 2^-22 of that
magnitude covers it; a 16-bit result adds half an ulp of itself (2^-11 fp16, 2^-8 bf16)."""
import ctypes

import numpy as np
import pytest

from cinn_amd import _lib, runtime
from cinn_amd.common import bfloat16_bits_to_float32, float32_to_bfloat16_bits

from test_gpu_gemm import call_cublas

pytestmark = pytest.mark.gpu

SHAPES = [
    (1, 1, 1, 1), (1, 1, 7, 3), (1, 3, 1, 65), (1, 63, 65, 64), (1, 65, 63, 129), (1, 129, 127, 127), (5, 1, 215, 48),
    (3, 48, 1, 215), (1, 17, 300, 172), (2, 1500, 1300, 33), (1, 1290, 1540, 700),  # many 64x64 tiles
    (1, 2050, 2000, 200),   # 16 bits: 128x128 tiles of one group
    (1, 1290, 1540, 1410),  # 16 bits: 128x128 tiles of two groups
    (1, 70, 90, 3001),      # K split
]


def rounded(rng, shape, kind):
    v = rng.standard_normal(shape).astype(np.float32)
    if kind == "bfloat16":
        bits = float32_to_bfloat16_bits(v)
        return bits, bfloat16_bits_to_float32(bits).astype(np.float64)
    v = v.astype(kind)
    return v, v.astype(np.float64)


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("kind", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("batch,m,n,k", SHAPES)
def test_edges(gpu, batch, m, n, k, kind, ta, tb):
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    a, af = rounded(rng, (batch, k, m) if ta else (batch, m, k), kind)
    b, bf = rounded(rng, (batch, n, k) if tb else (batch, k, n), kind)
    c0, cf = rounded(rng, (batch, m, n), kind)
    got = call_cublas(a, b, (batch, m, n), kind, ta, tb, alpha=0.5, beta=-1.0, c_init=c0)
    got = (bfloat16_bits_to_float32(got) if kind == "bfloat16" else got).astype(np.float64)
    am, bm = (np.swapaxes(af, 1, 2) if ta else af), (np.swapaxes(bf, 1, 2) if tb else bf)
    want  = 0.5 * (am @ bm) - cf
    scale = 0.5 * (np.abs(am) @ np.abs(bm)) + np.abs(cf)
    ulp   = {"float32": 2.0 ** -24, "float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}[kind]
    assert np.all(np.abs(got - want) <= (2.0 ** -24 * np.sqrt(k) + 2.0 ** -22) * scale + ulp * np.abs(want) + 2.0 ** -25)


@pytest.mark.parametrize("kind", ["float32", "float16"])
@pytest.mark.parametrize("ta,tb", [(False, True), (True, False)])
def test_what_lies_beyond_k_is_not_multiplied(gpu, kind, ta, tb):
    """k = 65: the chunk that reaches beyond a row's k holds the next row's first values, which are infinite here; and
    rows beyond a [k][row] operand's last full chunk neighbour the next k row"""
    m, n, k = 67, 70, 65
    rng = np.random.default_rng(5)
    a, b = rng.standard_normal((m, k)).astype(kind), rng.standard_normal((n, k)).astype(kind)
    a[1:, :] = np.inf
    got = call_cublas(np.ascontiguousarray(a.T) if ta else a, b if tb else np.ascontiguousarray(b.T), (m, n), kind, ta, tb)
    want = a[0].astype(np.float64) @ b.astype(np.float64).T
    assert np.all(np.isfinite(got[0].astype(np.float64)))
    np.testing.assert_allclose(got[0].astype(np.float64), want, rtol=2.0 ** -10, atol=2.0 ** -10)


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False)])
@pytest.mark.parametrize("batch,m,n,k,split", [(1, 128, 128, 4096, True), (1, 256, 128, 2048, True), (3, 128, 256, 1024, True),
                                               (1, 512, 1024, 1024, True), (1, 1024, 1024, 96, False), (2, 128, 128, 32, False),
                                               (1, 896, 1152, 1024, False)])
def test_whole_fp32_tiles_that_leave_cus_idle_split_k(tiled_kernels, batch, m, n, k, split, ta, tb):
    """extents that are whole 128x128 tiles: a K that is worth splitting over the CUs left idle uses partial sums (the stream
    has no scratch before), others do not"""
    rng = np.random.default_rng(k)
    a, af = rounded(rng, (batch, k, m) if ta else (batch, m, k), "float32")
    b, bf = rounded(rng, (batch, n, k) if tb else (batch, k, n), "float32")
    lib, stream = _lib.load(), runtime.Stream()
    lib.cinn_hip_scratch_release_stream.argtypes = [ctypes.c_void_p]
    assert lib.cinn_hip_scratch_release_stream(stream.handle) == 0
    lib.cinn_call_cublas.argtypes = ([ctypes.c_void_p, ctypes.c_int] + [ctypes.c_bool] * 3 + [ctypes.c_float] * 2 +
                                     [ctypes.c_int] * 8 + [ctypes.c_void_p])
    A, B, C = (runtime.DeviceBuffer.from_numpy(t) for t in (a, b, np.zeros((batch, m, n), np.float32)))
    lib.cinn_call_cublas(runtime.pod_args([A, B, C]), 3, ta, tb, False, 1.0, 0.0, 1, *a.shape, 1, *b.shape, stream.handle)
    stream.synchronize()
    capacity = ctypes.c_size_t(0)
    assert lib.cinn_hip_scratch_info(stream.handle, ctypes.byref(capacity), None, None) == 0
    assert (capacity.value >= 2 * batch * m * n * 4) == split
    am, bm = (np.swapaxes(af, 1, 2) if ta else af), (np.swapaxes(bf, 1, 2) if tb else bf)
    want, scale = am @ bm, np.abs(am) @ np.abs(bm)
    assert np.all(np.abs(C.numpy() - want) <= (2.0 ** -24 * np.sqrt(k) + 2.0 ** -22) * scale + 2.0 ** -24 * np.abs(want))
