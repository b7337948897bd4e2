"""Counters of kernel launches (cinn_amd/csrc/kernels/launch_count.h)."""
import contextlib
import ctypes

from cinn_amd import _lib

FEW, PATCH, ROWS_RING, ROWS, GROUP = range(5), 5, 6, 7, 8


def _counts():
    fn = _lib.load().cinn_hip_launches
    fn.argtypes, fn.restype = [ctypes.c_int], ctypes.c_longlong
    return [fn(i) for i in range(GROUP + 1)]


@contextlib.contextmanager
def launches():
    """count(counter, ...): launches since the block was entered"""
    before = _counts()

    def count(*which):
        now = _counts()
        return sum(now[i] - before[i] for i in which)

    yield count
