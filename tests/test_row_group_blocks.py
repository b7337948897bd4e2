"""Threads that a group of several row reductions gives a row: blocks of 512 where a wavefront would have walked it, and of as
many as keep a longer row in registers (1024 threads of up to 64 elements) however many reductions read it."""
import re

import numpy as np
import pytest

from cinn_amd.common import Float
from cinn_amd.frontend import NetBuilder

from helpers import compile_only, run


def program(rows, cols):
    b = NetBuilder("rows")
    x = b.create_input(Float(32), [rows, cols], "x")
    return b, x, [b.softmax(x, axes=[-1]), b.reduce_sum(x, [1]), b.argmax(x, 1)]


@pytest.mark.parametrize("rows", [4, 600])
@pytest.mark.parametrize("cols,threads", [(2600, (256, 512)), (4096, (256, 512)), (8193, (1024,)), (16384, (1024,)), (32769, (1024,)), (50257, (1024,))])
def test_threads_of_a_row(rows, cols, threads):
    b, _, outs = program(rows, cols)
    bounds = re.findall(r"__launch_bounds__\((\d+)", compile_only(b, outs, split_reductions=False).source_code())
    assert len(bounds) == 1 and int(bounds[0]) in threads


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 65])
@pytest.mark.parametrize("cols", [8193, 32769, 50257])
def test_long_rows(gpu, rows, cols):
    x = np.random.default_rng(cols).standard_normal((rows, cols)).astype(np.float32)
    b, v, outs = program(rows, cols)
    (soft, total, index), _ = run(b, {v: x}, outs)
    x64 = x.astype(np.float64)
    e = np.exp(x64)
    want = e / e.sum(1, keepdims=True)
    # sums of `cols` terms in chains far shorter than that; exp of up to 2 |x| of fp32 error, eight roundings
    unit = 2.0 ** -24
    assert np.all(np.abs(soft - want) <= unit * (16 + np.sqrt(cols)) * want)
    assert np.all(np.abs(total.reshape(-1) - x64.sum(1)) <= unit * np.sqrt(cols) * np.abs(x64).sum(1))
    assert np.array_equal(index.reshape(-1), x.argmax(1))
