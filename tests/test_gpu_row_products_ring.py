"""Layers of few rows in whole K steps of 64 (gemm_rows_ring_kernel) through cinn_call_hip_matmul_rows: every tile of the kernel, K
of fewer steps than wavefronts and of uneven shares, each length that a normalised row may have in a wavefront, one and two
fragments of columns in a normalising block, rows and columns that are no multiple of a tile, one to three results.

Bounds as in test_gpu_row_products: norm in fp32, rounded once to the type, a product of k terms with fp32 sums and one rounding of
the result; |gelu'| < 1.13."""
import ctypes
import math

import numpy as np
import pytest
from scipy.special import erf

from cinn_amd import _lib, runtime
from cinn_amd.common import bfloat16_bits_to_float32, float32_to_bfloat16_bits

from test_gpu_projections import UNIT
from test_gpu_row_products import norm64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("m,k,n,outputs,norm", [
    (1, 64, 4, 1, False), (16, 192, 36, 3, False), (17, 4096, 100, 1, False), (3, 320, 8200, 1, False), (33, 640, 1204, 1, False),
    (64, 512, 4100, 1, False), (50, 128, 16388, 1, False), (9, 2048, 68, 1, False), (31, 960, 2004, 3, False),
    (1, 64, 20, 1, True), (16, 512, 300, 3, True), (15, 704, 100, 1, True), (8, 1024, 36, 1, True), (17, 1280, 68, 1, True),
    (5, 128, 6148, 1, True), (40, 384, 2004, 3, True), (33, 640, 1700, 1, True), (20, 896, 2500, 1, True), (16, 1216, 4500, 1, True),
])
@pytest.mark.parametrize("gelu,residual", [(False, False), (True, False), (False, True)])
def test_rows(gpu, m, k, n, outputs, norm, gelu, residual, dtype):
    if residual and outputs > 1:
        pytest.skip("a residual goes to one result")
    rng = np.random.default_rng(m + k + n)

    def put(values, kind=dtype):
        values = np.ascontiguousarray(values, np.float32)
        if kind == "bfloat16":
            bits = float32_to_bfloat16_bits(values)
            return runtime.DeviceBuffer.from_numpy(bits, kind), bfloat16_bits_to_float32(bits).astype(np.float64)
        return runtime.DeviceBuffer.from_numpy(values.astype(kind), kind), values.astype(kind).astype(np.float64)

    X, x64 = put(rng.standard_normal((m, k)) * 2.0 + 0.3)
    W, w64 = put(rng.standard_normal((n, k)) * k ** -0.5)
    S, s64 = put(rng.uniform(0.5, 1.5, n), "float32")
    C, c64 = put(rng.standard_normal(n), "float32")
    bufs, slots, u = [X, W, S, C], 0x3210, UNIT[dtype]
    slack = np.zeros((m, k))
    where = {4: 15, 5: 15, 6: 15}
    if residual:
        R, r64 = put(rng.standard_normal((m, n)))
        where[4] = len(bufs)
        bufs.append(R)
    if norm:
        G, g64 = put(rng.uniform(0.5, 1.5, k))
        B, b64 = put(rng.standard_normal(k) * 0.1)
        where[5], where[6] = len(bufs), len(bufs) + 1
        bufs += [G, B]
        x64 = norm64(x64, g64, b64)
        slack = (u + 2.0 ** -18) * (np.abs(x64) + np.abs(b64))
    for slot, at in where.items():
        slots |= at << (4 * slot)
    outs = [runtime.DeviceBuffer((m, n // outputs), dtype) for _ in range(outputs)]
    bufs += outs
    fn = _lib.load().cinn_call_hip_matmul_rows
    fn.argtypes = [ctypes.c_void_p] + [ctypes.c_int] * 6 + [ctypes.c_float, ctypes.c_int, ctypes.c_void_p]
    fn.restype = None
    fn(runtime.pod_args(bufs), len(bufs), m, n, k, slots, outputs, 1e-5, int(gelu), None)
    runtime.synchronize()
    got = np.concatenate([bfloat16_bits_to_float32(o.numpy()) if dtype == "bfloat16" else o.numpy() for o in outs], axis=1).astype(np.float64)
    want = (x64 @ w64.T) * s64 + c64
    bound = (slack @ np.abs(w64.T) + (k + 2) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64.T))) * s64 + 2.0 ** -24 * np.abs(c64)
    if residual:
        want = want + r64
        bound = bound + 2.0 ** -24 * np.abs(r64)
    if gelu:
        want, bound = want * 0.5 * (1 + erf(want / math.sqrt(2))), 1.13 * bound + 2.0 ** -22 * np.abs(want)
    assert np.all(np.abs(got - want) <= 1.01 * (bound + u * np.abs(want)) + 1e-7)
