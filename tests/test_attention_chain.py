"""Programs in which one attention reads what another one computes (frontend/attention_pass.cc): the transpose behind the
first is taken along by its call, and the second finds it as its query, keys, values or a piece of them (attention along
one axis of an image and then along the other has this form).  Every program compiles - compilation refuses one that reads
a value nothing defines - and on the GPU gives what the separate operators give."""
import itertools

import numpy as np
import pytest

from cinn_amd.common import Float
from cinn_amd.frontend import NetBuilder

from helpers import compile_only, run

B, H, T, D = 2, 5, 6, 16  # the transposed [B, T, H, D] is read as T heads of H rows

ROLES = ["q", "k", "v", "qkv", "k_piece", "v_piece", "kv_pieces", "kv_first", "q_and_reshape"]


def chain(role):
    rng = np.random.default_rng(len(role))
    b = NetBuilder("chain")
    feeds = {}

    def given(name, shape):
        feeds[name] = rng.standard_normal(shape).astype(np.float32)
        return b.create_input(Float(32), list(shape), name)

    def attention(q, k, v):
        return b.matmul(b.softmax(b.matmul(q, k, False, True, 0.25), axes=[-1]), v)

    q, k, v = (given(n, (B, H, T, D)) for n in "qkv")
    m = b.transpose(attention(q, k, v), [0, 2, 1, 3])  # [B, T, H, D]
    q2, k2, v2 = (given(n + "2", (B, T, H, D)) for n in "qkv")
    if role in ("q", "qkv", "q_and_reshape"):
        q2 = m
    if role in ("k", "qkv"):
        k2 = m
    if role in ("v", "qkv"):
        v2 = m
    if role in ("k_piece", "kv_pieces"):
        k2 = b.concat([k2, m], axis=2)
        v2 = b.concat([v2, m if role == "kv_pieces" else given("v3", (B, T, H, D))], axis=2)
    if role == "v_piece":
        k2, v2 = b.concat([k2, given("k3", (B, T, H, D))], axis=2), b.concat([v2, m], axis=2)
    if role == "kv_first":
        k2, v2 = b.concat([m, k2], axis=2), b.concat([m, v2], axis=2)
    outs = [b.transpose(attention(q2, k2, v2), [0, 2, 1, 3])]
    if role == "q_and_reshape":
        outs.append(b.relu(b.reshape(m, [B * T, H * D])))
    # a third one reads the second's result the same way
    outs.append(attention(q, k, outs[0]))
    return b, feeds, outs


@pytest.mark.parametrize("role", ROLES)
def test_compiles(role):
    b, _, outs = chain(role)
    compile_only(b, outs)
    compile_only(b, outs[1:])  # the second result not fetched: its transpose may be taken along too


@pytest.mark.gpu
@pytest.mark.parametrize("fetch_all,role", itertools.product([True, False], ROLES))
def test_equals_separate_operators(gpu, role, fetch_all):
    results = []
    for fused in (1, 0):
        b, feeds, outs = chain(role)
        results.append(run(b, feeds, outs if fetch_all else outs[1:], fuse_attention=fused)[0])
    for got, want in zip(*results):
        # fp32 sums of 16 to 32 terms of magnitude below 4, three attentions in a row
        np.testing.assert_allclose(got, want, rtol=0, atol=2e-5)
