"""Attention with a scale of 0, or none that is finite: a program keeps its separate operators (0 times a score that
overflows is no number there), and cinn_call_hip_attention called by itself gives every key the same weight."""
import ctypes

import numpy as np
import pytest

from cinn_amd import _lib, runtime
from cinn_amd.common import Float
from cinn_amd.frontend import NetBuilder

from helpers import compile_only, run

ULP = {"float32": 2.0 ** -24, "float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}


def program(alpha, const):
    b = NetBuilder("scale")
    if const:  # the projections of one input, which one product computes where an attention reads them
        x = b.create_input(Float(32), [6, 32], "x")

        def heads(e):
            w, bias = b.create_input(Float(32), [32, 32], "w" + e), b.create_input(Float(32), [32], "b" + e)
            w.set_const(True), bias.set_const(True)
            return b.transpose(b.reshape(b.add(b.matmul(x, w), bias), [2, 3, 2, 16]), [0, 2, 1, 3])
        q, k, v = (heads(e) for e in "qkv")
    else:
        q, k, v = (b.create_input(Float(32), [2, 2, 3, 16], e) for e in "qkv")
    return b, b.matmul(b.softmax(b.matmul(q, k, False, True, alpha), axes=[-1]), v)


@pytest.mark.parametrize("const", [False, True])
@pytest.mark.parametrize("alpha,fused", [(0.0, False), (-0.0, False), (0.25, True), (-3.0, True)])
def test_programs_with_scale_zero_keep_their_operators(alpha, fused, const):
    b, o = program(alpha, const)
    comp = compile_only(b, [o])
    names = [comp.instruction_info(i)[0] for i in range(comp.num_instructions())]
    assert any("hip_attention" in n for n in names) == fused
    # three projections become one product only together with the attention that reads its parts
    products = sum("matmul" in n for n in names)
    assert products == {(True, True): 1, (True, False): 0, (False, True): 5, (False, False): 2}[fused, const], names


@pytest.mark.gpu
def test_program(gpu):
    rng = np.random.default_rng(2)
    feeds = {e: rng.standard_normal((2, 2, 3, 16)).astype(np.float32) for e in "qkv"}
    feeds["q"][1, 1, 2, 0] = np.inf  # 0 * inf: that row has no result
    b, o = program(0.0, False)
    (got,), _ = run(b, feeds, [o])
    want = np.broadcast_to(feeds["v"].astype(np.float64).mean(2, keepdims=True), got.shape).copy()
    assert np.isnan(got[1, 1, 2]).all()
    got[1, 1, 2] = want[1, 1, 2] = 0.0
    np.testing.assert_allclose(got, want, rtol=0, atol=2e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [0.0, -0.0])
@pytest.mark.parametrize("kind", sorted(ULP))
@pytest.mark.parametrize("tq,keys,appended", [(1, 1, 0), (1, 70, 0), (4, 65, 9), (40, 33, 0), (40, 64, 0), (33, 50, 47), (5, 1, 0)])
def test_call(gpu, tq, keys, appended, kind, scale):
    from test_gpu_backward import from_dev, round_to, to_dev
    bh, d = 3, 48
    rng = np.random.default_rng(tq * 100 + keys)
    q, k, v, k2, v2 = (round_to(rng.standard_normal((bh, 1, rows, d)), kind) for rows in (tq, keys, keys, max(1, appended), max(1, appended)))
    bufs = [to_dev(t, kind) for t in (q, k, k2, v, v2, np.zeros_like(q))]
    lib = _lib.load()
    lib.cinn_call_hip_attention.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_float] + [ctypes.c_int] * 9 + [ctypes.c_void_p]
    lib.cinn_call_hip_attention(runtime.pod_args(bufs), 6, scale, bh, 1, tq, keys, appended, d, 0x43210, 0, 1, None)
    runtime.synchronize()
    rows = np.concatenate([v, v2[:, :, :appended]], 2).astype(np.float64)
    want = np.broadcast_to(rows.mean(2, keepdims=True), q.shape)
    # every weight is exactly 1 before the division: an fp32 sum, and half an ulp of the result
    bound = (keys + appended) * 2.0 ** -24 * np.abs(rows).mean(2, keepdims=True) + ULP[kind] * np.abs(want) + 2.0 ** -25
    assert np.all(np.abs(from_dev(bufs[5], kind) - want) <= bound)
