"""Which kernel a channels-last convolution runs on: a switch that asks for one of the kernels for larger grids, or for a tile or a
split of theirs, wins over the automatic choice for layers of few tiles (conv_few_mfma.hip).  And what those kernels are tested
for at layers of few tiles, on those kernels."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

from cinn_amd import _lib

from launch_counts import FEW, PATCH, launches
from test_gpu_c_abi import test_channels_last_convolution_is_captured_after_reserving_its_scratch as check_capture
from test_gpu_conv_pool import PATCH_CASES, PATCH_CHUNK_CASES, call_conv_nhwc
from test_gpu_conv_pool import test_fused_relu_of_nan_and_infinite_sums as check_relu_of_nan

pytestmark = pytest.mark.gpu


@pytest.fixture
def modes():
    """sets a switch for the length of a test"""
    lib, before = _lib.load(), []

    def put(switch, value):
        fn = getattr(lib, switch)
        fn.argtypes, fn.restype = [ctypes.c_int], ctypes.c_int
        before.append((fn, fn(value)))

    yield put
    for fn, value in reversed(before):
        fn(value)


def run(case):
    n, ic, h, w, oc = case
    rng = np.random.default_rng(1)
    call_conv_nhwc(rng.standard_normal((n, ic, h, w)), rng.standard_normal((oc, ic, 3, 3)) * 0.05, 1, 1, 1, "float16")


@pytest.mark.parametrize("case", PATCH_CASES + PATCH_CHUNK_CASES)
def test_kernel_that_keeps_the_input_patch(gpu, modes, case):
    """forced, switched off (an implicit GEMM), and by the automatic choice"""
    # (not: blocks that would be half empty, and a row whose patch is beyond LDS)
    qualifies = case not in ((3, 64, 14, 14, 192), (1, 64, 1, 400, 64))
    for mode, patch, few in ((2, qualifies, False), (0, False, False), (1, False, True)):
        modes("cinn_hip_conv_patch_mode", mode)
        with launches() as count:
            run(case)
        assert (count(PATCH) == 1) == patch and (count(*FEW) == 1) == few, mode


@pytest.mark.parametrize("switch,value,case", [("cinn_hip_conv_patch_tiles", 2, (2, 128, 28, 28, 128)), ("cinn_hip_conv_patch_tiles", 4, (2, 256, 14, 14, 256)),
                                               ("cinn_hip_conv_patch_stream", 0, (2, 64, 56, 56, 64)), ("cinn_hip_conv_few_mode", 0, (2, 64, 56, 56, 64))])
def test_its_other_switches(gpu, modes, switch, value, case):
    modes(switch, value)
    with launches() as count:
        run(case)
    assert count(*FEW) == 0


CHILD = """
import sys
import numpy as np
sys.path.insert(0, {tests!r})
from launch_counts import FEW, launches
from test_gpu_conv_pool import call_conv_nhwc
rng = np.random.default_rng(1)
for shape, k, dtype in (((1, 256, 14, 14), 1, "float16"), ((1, 128, 14, 14), 3, "float16"), ((1, 128, 14, 14), 3, "float32")):
    x, w = rng.standard_normal(shape), rng.standard_normal((132, shape[1], k, k)) * 0.05
    with launches() as count:
        call_conv_nhwc(x, w, 1, k // 2, 1, dtype)
    print("few", count(*FEW))
"""


@pytest.mark.parametrize("flag,value,few", [("gemm_tile", "128", (0, 0, 1)), ("gemm_split_k", "2", (0, 0, 1)), ("gemm_split_k", "0", (1, 1, 1)), ("conv_pointwise_gemm", "2", (0, 1, 1)),
                                            ("conv_tile", "2", (0, 0, 0)), ("conv_splits", "3", (0, 0, 0)), ("conv_few", "0", (0, 0, 0)),
                                            ("conv_few", "1", (1, 1, 1))])
def test_switches_that_are_read_once(gpu, flag, value, few):
    here = os.path.dirname(os.path.abspath(__file__))
    code = CHILD.format(tests=here)
    out = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, **{"FLAGS_cinn_hip_" + flag: value}), cwd=os.path.dirname(here),
                         stdout=subprocess.PIPE, check=True, timeout=100, text=True).stdout
    assert tuple(int(line.split()[1]) for line in out.splitlines() if line.startswith("few")) == few


@pytest.mark.parametrize("dtype", ["float16", "float32"])
@pytest.mark.parametrize("shape", [(2, 64, 56, 56, 64, 3, 1), (2, 128, 28, 28, 128, 3, 1), (4, 256, 14, 14, 512, 1, 0)])
def test_fused_relu_of_nan_and_infinite_sums(gpu, modes, shape, dtype):
    modes("cinn_hip_conv_few_mode", 0)
    check_relu_of_nan(gpu, shape, dtype)


def test_capture_of_the_patch_by_channel_chunks(gpu, modes):
    modes("cinn_hip_conv_patch_mode", 2)
    with launches() as count:
        check_capture(gpu, "float16", (3, 128, 28, 28, 128), 1e-2)
    assert count(PATCH) == 2  # recorded, and the eager call
