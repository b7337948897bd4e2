"""Threads of 4 instead of 16 bytes of channels, for tensors that would leave CUs without a block (channel_sums_kernel,
channel_apply_kernel, max_pool3s2_backward_kernel): one chunk and odd numbers of chunks, and the last size that has them next to the
first that has not."""
import numpy as np
import pytest

from test_gpu_backward import test_pool2d_backward as check_pool_backward
from test_gpu_channel_sums import test_statistics_and_gradient as check_batch_norm

pytestmark = pytest.mark.gpu


# 256 CUs * 512 pixels are 2^17 chunks: of 8 channels 16383 and 16384 pixels, of 4 channels half as many
@pytest.mark.parametrize("dtype,shape", [
    ("float16", (1, 1, 1, 24)), ("bfloat16", (1, 1, 2, 8)), ("float32", (2, 1, 2, 12)), ("float16", (2, 9, 5, 1032)), ("bfloat16", (3, 31, 37, 40)),
    ("float16", (1, 129, 127, 64)), ("float16", (1, 128, 128, 64)), ("bfloat16", (1, 129, 127, 64)), ("bfloat16", (1, 128, 128, 64)),
    ("float32", (1, 8191, 1, 64)), ("float32", (1, 64, 128, 64)),
])
@pytest.mark.parametrize("masked", [False, True])
def test_batch_norm(gpu, shape, dtype, masked):
    check_batch_norm(gpu, shape, dtype, masked)


# 2^16 threads of 16 bytes: 524288 elements of 16 bits, 262144 of 32
@pytest.mark.parametrize("dtype,tol", [("float16", 2.0 ** -10), ("bfloat16", 2.0 ** -7), ("float32", 2.0 ** -22)])
@pytest.mark.parametrize("shape", [(1, 8, 1, 1), (2, 24, 12, 11), (1, 16, 7, 2), (2, 64, 64, 63), (2, 64, 64, 64), (2, 64, 32, 63), (2, 64, 32, 64)])
def test_max_pool_gradient(gpu, shape, dtype, tol):
    check_pool_backward(gpu, shape + (3, 2, 1), 0, dtype, tol, 1)
