"""Attention as one call (attention.hip, frontend/attention_pass.cc) at the edges of its tiles - 32 queries per wavefront,
32 to 128 per block, 64 keys per stage, four queries for the row kernel, rows between the instantiated lengths -
against float64, and in every layout the pass reads in place against the calls it replaces.

Bounds: a score is an fp32 sum of d products (2^-24 sqrt(d) + 2^-22 of the products' magnitudes); the relative error of a
probability is twice that and what exp adds (its argument's rounding, 2^-24 of up to 32, and its own 2^-21).  16-bit
operands of the second product are rounded probabilities (half an ulp, subnormal ones 2^-25); the result rounds once."""
import math

import numpy as np
import pytest

from cinn_amd.common import BFloat16, Float, bfloat16_bits_to_float32, float32_to_bfloat16_bits
from cinn_amd.frontend import NetBuilder

from helpers import run

pytestmark = pytest.mark.gpu

ULP = {"float32": 2.0 ** -24, "float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}
TYPES = sorted(ULP)


def inputs(rng, shape, kind, scale=1.0):
    v = (rng.standard_normal(shape) * scale).astype(np.float32)
    if kind == "bfloat16":
        bits = float32_to_bfloat16_bits(v)
        return bits, bfloat16_bits_to_float32(bits).astype(np.float64)
    v = v.astype(kind)
    return v, v.astype(np.float64)


def as_float64(x, kind):
    return (bfloat16_bits_to_float32(x) if kind == "bfloat16" else x).astype(np.float64)


def dtype(kind):
    return BFloat16() if kind == "bfloat16" else Float(32 if kind == "float32" else 16)


def reference(q, k, v, alpha, kind):
    """float64 result and the bound on its error"""
    kt = np.swapaxes(k, -1, -2)
    s = alpha * (q @ kt)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    score = (2.0 ** -24 * math.sqrt(q.shape[-1]) + 2.0 ** -22) * abs(alpha) * (np.abs(q) @ np.abs(kt)).max(-1, keepdims=True)
    u = ULP[kind]
    bound = (2 * score + 2.0 ** -18 + 2 * u) * (p @ np.abs(v)) + u * np.abs(p @ v)
    if kind == "float16":
        bound += (k.shape[-2] * 2.0 ** -25) * np.abs(v).max() + 2.0 ** -24
    return p @ v, bound


@pytest.mark.parametrize("kind", TYPES)
@pytest.mark.parametrize("bh,tq,tk,d", [
    (1, 1, 1, 8), (2, 1, 31, 64), (3, 1, 1024, 80), (1, 4, 65, 48), (2, 3, 257, 128), (1, 2, 1500, 32), (1, 1, 70, 120),
    (1, 5, 1, 8), (2, 31, 33, 64), (1, 32, 64, 48), (3, 33, 65, 80), (1, 64, 63, 16), (2, 100, 129, 96), (1, 40, 200, 128),
    (1, 37, 50, 72), (130, 129, 40, 64), (130, 256, 64, 32), (86, 300, 97, 80), (128, 257, 33, 128), (1, 700, 700, 40)])
def test_edges(gpu, bh, tq, tk, d, kind):
    rng = np.random.default_rng(tq * 1000 + tk + d)
    q, qf = inputs(rng, (bh, tq, d), kind)
    k, kf = inputs(rng, (bh, tk, d), kind)
    v, vf = inputs(rng, (bh, tk, d), kind)
    alpha = 1.0 / math.sqrt(d)
    b = NetBuilder("attention")
    Q, K, V = (b.create_input(dtype(kind), list(x.shape), n) for x, n in ((q, "q"), (k, "k"), (v, "v")))
    o = b.matmul(b.softmax(b.matmul(Q, K, False, True, alpha), axes=[2]), V)
    (got,), _ = run(b, {Q: q, K: k, V: v}, [o])
    want, bound = reference(qf, kf, vf, alpha, kind)
    assert np.all(np.abs(as_float64(got, kind) - want) <= bound)


@pytest.mark.parametrize("kind", TYPES)
@pytest.mark.parametrize("tq,past,new", [(1, 37, 1), (6, 0, 6), (40, 70, 9), (3, 5, 200)])
@pytest.mark.parametrize("split_cache,fetch", [(False, False), (True, False), (True, True)])
def test_layouts(gpu, kind, tq, past, new, split_cache, fetch):
    """heads split from and merged into [b][t][h][d], keys and values joined from a cache and new rows (the cache split
    from [b][t][h][d] too, or not), the new rows fetched or not: against the same program as separate calls"""
    n, heads, d = 2, 3, 64
    rng = np.random.default_rng(tq)

    def build():
        rng_in = np.random.default_rng(tq)
        feeds = {}
        b = NetBuilder("layouts")

        def given(name, shape):
            x, _ = inputs(rng_in, shape, kind)
            var = b.create_input(dtype(kind), list(shape), name)
            feeds[name] = x
            return var

        def split(x):
            return b.transpose(x, [0, 2, 1, 3])
        q = split(given("q", (n, tq, heads, d)))
        k, v = split(given("k", (n, new, heads, d))), split(given("v", (n, new, heads, d)))
        outs = [k, v] if fetch else []
        if past:
            shape = (n, past, heads, d) if split_cache else (n, heads, past, d)
            pk, pv = given("pk", shape), given("pv", shape)
            k = b.concat([split(pk) if split_cache else pk, k], axis=2)
            v = b.concat([split(pv) if split_cache else pv, v], axis=2)
        o = b.matmul(b.softmax(b.matmul(q, k, False, True, 0.125), axes=[-1]), v)
        return b, feeds, outs + [b.transpose(o, [0, 2, 1, 3])]

    results = []
    for fused in (1, 0):
        b, feeds, outs = build()
        got, _ = run(b, feeds, outs, fuse_attention=fused)
        results.append([as_float64(g, kind) for g in got])
    for g, w in zip(results[0][:-1], results[1][:-1]):
        assert np.array_equal(g, w)
    # the separate calls round scores (|s| < 8) and probabilities to the type
    np.testing.assert_allclose(results[0][-1], results[1][-1], rtol=0, atol=24 * ULP[kind] * 4 if kind != "float32" else 2e-5)


@pytest.mark.parametrize("tq", [2, 40])
def test_one_tensor_as_several_operands_and_fetched_probabilities(gpu, tq):
    rng = np.random.default_rng(3)
    x, xf = inputs(rng, (2, tq, 32), "float32")
    b = NetBuilder("shared")
    X = b.create_input(Float(32), [2, tq, 32], "x")
    o = b.matmul(b.softmax(b.matmul(X, X, False, True, -0.2), axes=[-1]), X)
    p = b.softmax(b.matmul(X, X, False, True, 0.3), axes=[-1])
    (got, probs, got2), _ = run(b, {X: x}, [o, p, b.matmul(p, X)])
    for alpha, g in ((-0.2, got), (0.3, got2)):
        want, bound = reference(xf, xf, xf, alpha, "float32")
        assert np.all(np.abs(g - want) <= 2 * bound)
    np.testing.assert_allclose(probs.sum(-1), 1.0, rtol=1e-5)


@pytest.mark.parametrize("kind", ["float32", "float16"])
@pytest.mark.parametrize("tq", [1, 40])
def test_infinities_and_nan(gpu, tq, kind):
    """keys whose scores are -inf count nothing (also where they fill the first tiles); +inf or NaN makes its row NaN;
    a row of -inf only has no probabilities"""
    tk, d = 200, 16
    q = np.ones((1, tq, d), kind)
    k = np.zeros((3, tk, d), kind)
    k[0, :150, 0] = -np.inf
    k[1, 70, 0] = np.inf
    k[2, :, 0] = -np.inf
    rng = np.random.default_rng(1)
    v, vf = inputs(rng, (3, tk, d), kind)
    b = NetBuilder("inf")
    Q, K, V = b.create_input(dtype(kind), [3, tq, d], "q"), b.create_input(dtype(kind), [3, tk, d], "k"), b.create_input(
        dtype(kind), [3, tk, d], "v")
    (got,), _ = run(b, {Q: np.repeat(q, 3, 0), K: k, V: v}, [b.matmul(b.softmax(b.matmul(Q, K, False, True), axes=[2]), V)])
    got = got.astype(np.float64)
    np.testing.assert_allclose(got[0], np.broadcast_to(vf[0, 150:].mean(0), (tq, d)), rtol=0, atol=4 * ULP[kind] + 1e-6)
    assert np.isnan(got[1:]).all()
