"""Sorting networks and selection of rows (sort.hip) at the sizes where one form ends and the next begins, against the
oracle's restatement of the reference's loop nests: indices, positions and values are exact, ties, signed zeros and NaNs
included.  Long rows, where the O(size^2) oracle is slow, are checked against numpy's stable argsort."""
import ctypes

import numpy as np
import pytest

from cinn_amd import _lib, runtime
from cinn_amd.common import Float, Int
from cinn_amd.frontend import NetBuilder

import oracle
from helpers import run

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 63, 64, 65, 256, 257, 1000, 1024, 1025, 4096, 4097, 16384]


def values(rng, shape, kind):
    if kind == "int32":
        x = rng.integers(-50, 50, shape).astype(np.int32)
        x.flat[0], x.flat[-1] = np.iinfo(np.int32).max, np.iinfo(np.int32).min
        return x
    x = (rng.integers(-40, 40, shape) / 8).astype(kind)  # ties
    x[rng.random(shape) < 0.05] = -0.0
    return x


def order(x, ascend):
    """stable order along the last axis with the reference's positions"""
    if x.shape[-1] <= 1100:
        return oracle.argsort(x, x.ndim - 1, ascend)
    key = x.astype(np.float64) if ascend else -x.astype(np.float64)
    index = np.argsort(key, axis=-1, kind="stable").astype(np.int32)
    ranked = np.take_along_axis(key, index, -1)
    first = np.stack([np.searchsorted(r, r, side="left") for r in ranked.reshape(-1, x.shape[-1])]).reshape(x.shape)
    positions = np.empty_like(index)
    np.put_along_axis(positions, index, first.astype(np.int32), -1)
    return index, positions, np.take_along_axis(x, index, -1)


@pytest.mark.parametrize("ascend", [True, False])
@pytest.mark.parametrize("kind", ["float32", "float16", "int32"])
@pytest.mark.parametrize("size", SIZES)
def test_rows(gpu, size, kind, ascend):
    rng = np.random.default_rng(size)
    x = values(rng, (3, size), kind)
    b = NetBuilder("rows")
    v = b.create_input(Int(32) if kind == "int32" else Float(16 if kind == "float16" else 32), list(x.shape), "x")
    index, positions = b.argsort(v, 1, ascend)
    got, _ = run(b, {v: x}, [index, positions, b.sort(v, 1, ascend)])
    for g, w in zip(got, order(x, ascend)):
        assert np.array_equal(g, w) and g.dtype == w.dtype


@pytest.mark.parametrize("size,inner", [(255, 3), (256, 3), (1000, 17)])
def test_columns(gpu, size, inner):
    """the other axes behind the sorted one: below 256 elements the tile scan, from there on the network"""
    rng = np.random.default_rng(size)
    x = values(rng, (2, size, inner), "float32")
    b = NetBuilder("columns")
    v = b.create_input(Float(32), list(x.shape), "x")
    index, positions = b.argsort(v, 1, False)
    got, _ = run(b, {v: x}, [index, positions, b.sort(v, 1, False)])
    for g, w in zip(got, oracle.argsort(x, 1, False)):
        assert np.array_equal(g, w)


@pytest.mark.parametrize("ascend", [True, False])
@pytest.mark.parametrize("size", [5, 64, 300, 1000])
def test_rows_with_nans(gpu, size, ascend):
    rng = np.random.default_rng(size)
    x = values(rng, (4, size), "float32")
    x[:3][rng.random((3, size)) < 0.2] = np.nan  # the last row has none
    x[1] = np.nan
    b = NetBuilder("nans")
    v = b.create_input(Float(32), list(x.shape), "x")
    index, positions = b.argsort(v, 1, ascend)
    got, _ = run(b, {v: x}, [index, positions, b.sort(v, 1, ascend)])
    for g, w in zip(got, oracle.argsort(x, 1, ascend)):
        assert np.array_equal(g, w, equal_nan=g.dtype == np.float32)


@pytest.mark.parametrize("k", [1, 5, 16, 17, 50])
@pytest.mark.parametrize("kind", ["float32", "float16", "int32"])
@pytest.mark.parametrize("size", [50, 256, 257, 1024, 1025, 5000, 16384])
def test_top_k(gpu, size, kind, k):
    rng = np.random.default_rng(size + k)
    x = values(rng, (3, size), kind)
    if kind != "int32" and size < 1000:
        x[1][rng.random(size) < 0.3] = np.nan
    b = NetBuilder("top")
    v = b.create_input(Int(32) if kind == "int32" else Float(16 if kind == "float16" else 32), list(x.shape), "x")
    best, where = b.top_k(v, k, 1)
    (got_values, got_index), comp = run(b, {v: x}, [best, where])
    assert comp.num_instructions() == 1 and "hip_top_k" in comp.instruction_info(0)[0]
    index, _, ranked = order(x, False)
    assert got_index.dtype == np.int64 and np.array_equal(got_index, index[:, :k])
    assert np.array_equal(got_values, ranked[:, :k], equal_nan=kind != "int32")


@pytest.mark.parametrize("equal", [1, 59, 60, 61, 300])
@pytest.mark.parametrize("k", [1, 16, 17, 50, 64])
@pytest.mark.parametrize("size", [64, 65, 1000, 1025, 4097])
def test_top_k_of_distinct_scores_and_equal_ones(gpu, size, k, equal):
    """the words up to the bound are ranked against each other, more than 64 or 128 of them are taken one by one: distinct
    scores, scores of which the k-th largest is shared, and a row whose largest ones a few lanes hold.  (For k of 50 and up to 1024
    elements these few rows are sorted by the network; test_top_k_of_many_rows has the selection.)"""
    rng = np.random.default_rng(size + k)
    x = rng.permuted(np.tile(np.arange(size, dtype=np.float32) - size // 2, (5, 1)), axis=1)
    x[4, rng.permutation(size)] = np.where(np.arange(size) % 64 < 3, size, 0) + x[4]
    for row in x[2:]:
        row[np.argsort(-row, kind="stable")[k - 1:k - 1 + equal]] = size
    b = NetBuilder("top")
    v = b.create_input(Float(32), list(x.shape), "x")
    (values, where), _ = run(b, {v: x}, list(b.top_k(v, k, 1)))
    index = np.argsort(-x, axis=1, kind="stable")[:, :k]
    assert np.array_equal(where, index) and np.array_equal(values, np.take_along_axis(x, index, 1))


# rows of up to 1024 elements go to the selection or to the network by their number, for k from 21 to 50
@pytest.mark.parametrize("equal", ["distinct", "few values", "one value"])
@pytest.mark.parametrize("rows,k", [(256, 20), (256, 24), (257, 25), (512, 32), (513, 33), (1024, 40), (1281, 41), (1792, 50), (1793, 50), (1793, 51), (600, 1)])
@pytest.mark.parametrize("size", [257, 1000])
def test_top_k_of_many_rows(gpu, size, rows, k, equal):
    rng = np.random.default_rng(size + rows + k)
    if equal == "distinct":
        x = rng.permuted(np.tile(np.arange(size, dtype=np.float32), (rows, 1)), axis=1)
    else:
        x = rng.integers(0, 9 if equal == "few values" else 1, (rows, size)).astype(np.float32)
    b = NetBuilder("top")
    v = b.create_input(Float(32), list(x.shape), "x")
    (values, where), _ = run(b, {v: x}, list(b.top_k(v, k, 1)))
    index = np.argsort(-x, axis=1, kind="stable")[:, :k]
    assert np.array_equal(where, index) and np.array_equal(values, np.take_along_axis(x, index, 1))


def test_top_k_of_one_output_or_shared_results(gpu):
    """only the values or only the indices are wanted; a full sort that something else reads stays"""
    rng = np.random.default_rng(1)
    x = values(rng, (6, 70, 2), "float32")
    index, positions, ranked = oracle.argsort(x, 1, False)
    b = NetBuilder("one")
    v = b.create_input(Float(32), list(x.shape), "x")
    (got,), comp = run(b, {v: x}, [b.top_k(v, 3, 1)[1]])
    assert np.array_equal(got, index[:, :3])
    b = NetBuilder("shared")
    v = b.create_input(Float(32), list(x.shape), "x")
    full = b.sort(v, 1, False)
    got, comp = run(b, {v: x}, [full, b.slice(full, [1], [0], [3])])
    assert np.array_equal(got[0], ranked) and np.array_equal(got[1], ranked[:, :3])


def test_top_k_ascending_through_the_c_abi(gpu):
    rng = np.random.default_rng(2)
    x = rng.standard_normal((2, 90, 3)).astype(np.float32)
    X = runtime.DeviceBuffer.from_numpy(x)
    V, I = runtime.DeviceBuffer((2, 4, 3), "float32"), runtime.DeviceBuffer((2, 4, 3), "int64")
    lib = _lib.load()
    lib.cinn_call_hip_top_k.argtypes = [ctypes.c_void_p, ctypes.c_int] + [ctypes.c_int] * 6 + [ctypes.c_void_p]
    lib.cinn_call_hip_top_k.restype = None
    lib.cinn_call_hip_top_k(runtime.pod_args([X, V, I]), 3, 2, 90, 3, 1, 4, 3, None)
    runtime.synchronize()
    index = np.argsort(x, axis=1, kind="stable")
    assert np.array_equal(I.numpy(), index[:, :4]) and np.array_equal(V.numpy(), np.sort(x, axis=1)[:, :4])


# the scan up to 64 elements of which at least (size - 16) / 4 are wanted, the selection and the network elsewhere
@pytest.mark.parametrize("kind", ["float32", "float16", "int32"])
@pytest.mark.parametrize("size,inner,k", [(1, 3, 1), (16, 1000, 1), (16, 33, 16), (21, 17, 1), (20, 17, 1), (64, 5, 12), (64, 5, 11), (63, 40, 50),
                                          (65, 9, 20), (300, 4, 5)])
def test_top_k_of_columns(gpu, size, inner, k, kind):
    rng = np.random.default_rng(size + inner + k)
    x = values(rng, (3, size, inner), kind)
    if kind != "int32":
        x[1][rng.random((size, inner)) < 0.2] = np.nan
    b = NetBuilder("top")
    v = b.create_input(Int(32) if kind == "int32" else Float(16 if kind == "float16" else 32), list(x.shape), "x")
    (got_values, got_index), comp = run(b, {v: x}, list(b.top_k(v, k, 1)))
    assert comp.num_instructions() == 1
    index, _, ranked = oracle.argsort(x, 1, False)
    assert np.array_equal(got_index, index[:, :k])
    assert np.array_equal(got_values, ranked[:, :k], equal_nan=kind != "int32")
