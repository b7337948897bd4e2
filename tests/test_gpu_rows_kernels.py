"""Which of gemm_rows.hip's two kernels runs a product of few rows, and the instances of gemm_rows_kernel that keep two to four row
tiles in a block (256 blocks of columns and more; K that is no whole step of 64, results in other than aligned groups of four)."""
import ctypes

import numpy as np
import pytest

from cinn_amd import _lib, runtime

from launch_counts import ROWS, ROWS_RING, launches
from test_gpu_row_products_ring import test_rows as check_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("m,k,n,outputs", [(17, 96, 4112, 1), (32, 64, 4098, 1), (33, 160, 4100, 1), (48, 256, 8196, 2), (49, 544, 4096, 1), (64, 1120, 4090, 1),
                                           (64, 32, 12294, 3)])
@pytest.mark.parametrize("residual", [False, True])
def test_row_tiles_of_a_block(gpu, m, k, n, outputs, residual, dtype):
    with launches() as count:
        check_rows(gpu, m, k, n, outputs, False, False, residual, dtype)
    assert count(ROWS) == 1 and count(ROWS_RING) == 0


@pytest.mark.parametrize("m,k,n,outputs,norm,gelu,ring", [
    (1, 64, 1024, 1, False, False, False), (1, 1024, 4096, 1, False, False, False), (1, 768, 2304, 3, False, False, True), (1, 1024, 4100, 1, False, False, True),
    (1, 1280, 3840, 3, False, False, True), (2, 1024, 4096, 1, False, False, True), (1, 384, 1536, 1, False, True, False), (1, 1024, 1024, 1, False, True, False),
    (1, 1280, 1280, 1, False, True, True), (2, 384, 1536, 1, False, True, True), (1, 768, 3072, 1, True, True, True), (1, 1024, 3072, 1, True, True, True), (1, 1024, 1024, 1, False, False, True),
    (1, 1280, 2560, 1, True, True, False), (1, 1280, 2560, 1, True, False, True),
])
def test_one_row(gpu, m, k, n, outputs, norm, gelu, ring):
    with launches() as count:
        check_rows(gpu, m, k, n, outputs, norm, gelu, False, "float16")
    assert (count(ROWS_RING), count(ROWS)) == ((1, 0) if ring else (0, 1))


# normalising blocks beyond 512, and of a grid of many rounds
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("m,k,n,outputs", [(64, 384, 6276, 1), (50, 128, 16388, 1), (33, 320, 12300, 3)])
@pytest.mark.parametrize("gelu", [False, True])
def test_norm_in_many_blocks(gpu, m, k, n, outputs, gelu, dtype):
    with launches() as count:
        check_rows(gpu, m, k, n, outputs, True, gelu, False, dtype)
    assert count(ROWS_RING) == 1 and count(ROWS) == 0


@pytest.mark.parametrize("m,k,n,outputs,ring", [(8, 768, 768, 1, True), (40, 512, 4104, 3, True), (40, 512, 4100, 2, False), (12, 576, 12, 2, False), (8, 96, 768, 1, False)])
def test_kernel(gpu, m, k, n, outputs, ring):
    with launches() as count:
        check_rows(gpu, m, k, n, outputs, False, False, False, "float16")
    assert (count(ROWS_RING), count(ROWS)) == ((1, 0) if ring else (0, 1))


# a result (offset in elements) in other than aligned groups of four goes by the rule of the kernel that would run it: the ring's
# rule sends 64 x 64 -> 4096 to gemm_rows.hip, the other kernel's (1024 blocks of one row tile's work) does not
@pytest.mark.parametrize("offset,ring,rows", [(0, 1, 0), (4, 1, 0), (2, 0, 0), (1, 0, 0)])
def test_result_at_any_address(gpu, offset, ring, rows):
    m, n, k, rng = 64, 4096, 64, np.random.default_rng(offset)
    a, b = (rng.standard_normal(s).astype(np.float16) for s in ((m, k), (n, k)))
    A, B, C = runtime.DeviceBuffer.from_numpy(a), runtime.DeviceBuffer.from_numpy(b), runtime.DeviceBuffer((m * n + 8,), "float16")
    C.copy_from(np.zeros(m * n + 8, np.float16))
    C.buffer.memory = C.ptr.value + 2 * offset
    fn = _lib.load().cinn_call_cublas
    fn.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_bool, ctypes.c_bool, ctypes.c_bool, ctypes.c_float, ctypes.c_float] + [ctypes.c_int] * 8 + [ctypes.c_void_p]
    with launches() as count:
        fn(runtime.pod_args([A, B, C]), 3, False, True, False, 1.0, 0.0, 1, 1, m, k, 1, 1, n, k, None)
        runtime.synchronize()
        assert (count(ROWS_RING), count(ROWS)) == (ring, rows)
    C.buffer.memory = C.ptr.value
    got = C.numpy()
    want = a.astype(np.float64) @ b.T.astype(np.float64)
    bound = k * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b.T).astype(np.float64)) + 2.0 ** -11 * np.abs(want)
    assert np.all(np.abs(got[offset:offset + m * n].reshape(m, n) - want) <= 1.01 * bound)
    assert not got[:offset].any() and not got[offset + m * n:].any()
