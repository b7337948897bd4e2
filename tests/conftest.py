import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu on the GPU box)")


@pytest.fixture(scope="session")
def gpu():
    """The GPU tests must run the HIP path: no device (or no native library) is a failure, not a skip."""
    from cinn_amd import runtime
    n = runtime.device_count()
    assert n > 0, "a test marked gpu ran without a visible GPU"
    return n


@pytest.fixture
def tiled_kernels(gpu):
    """for the length of a test, layers and products of few tiles stay with the kernels that split their K over blocks and add the
    parts through scratch memory"""
    import ctypes
    from cinn_amd import _lib
    mode = _lib.load().cinn_hip_conv_few_mode
    mode.argtypes, mode.restype = [ctypes.c_int], ctypes.c_int
    before = mode(0)
    yield
    mode(before)


@pytest.fixture
def rng():
    return np.random.default_rng(1234)
