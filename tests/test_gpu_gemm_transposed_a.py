"""Products with A stored [K][M] in whole 16-byte chunks, which run on the direct-to-LDS kernel (gemm_mfma.hip) where that is
faster: 128x128 tiles (K of any length when B is row-major: the k-rows beyond it come from a page of zeros) and 256x256
tiles, with last tiles of eight rows or columns, K of one step, of a step more or less than the stages, and a last step of
one k-row; batches; a beta term.

Bounds as in test_gpu_gemm_flex.py."""
import numpy as np
import pytest

from cinn_amd.common import bfloat16_bits_to_float32

from test_gpu_gemm import call_cublas
from test_gpu_gemm_flex import rounded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["float16", "bfloat16"])
@pytest.mark.parametrize("batch,m,n,k,tb", [
    (1, 1672, 1928, 1000, False), (1, 1800, 1672, 257, False), (1, 1608, 1608, 193, False),  # 128x128 tiles
    (1, 2056, 2048, 64, False), (2, 1288, 1544, 255, False),
    (1, 1672, 1928, 960, True), (1, 1800, 1672, 256, True), (1, 2056, 2048, 64, True),
    (1, 2824, 3080, 192, False), (1, 2824, 3080, 192, True), (2, 2056, 2056, 320, False),    # 256x256 tiles
])
def test_transposed_a(gpu, batch, m, n, k, tb, kind):
    rng = np.random.default_rng(m + n + k)
    a, af = rounded(rng, (batch, k, m), kind)
    b, bf = rounded(rng, (batch, n, k) if tb else (batch, k, n), kind)
    c0, cf = rounded(rng, (batch, m, n), kind)
    got = call_cublas(a, b, (batch, m, n), kind, True, tb, alpha=0.5, beta=-1.0, c_init=c0)
    got = (bfloat16_bits_to_float32(got) if kind == "bfloat16" else got).astype(np.float64)
    am, bm = np.swapaxes(af, 1, 2), (np.swapaxes(bf, 1, 2) if tb else bf)
    want  = 0.5 * (am @ bm) - cf
    scale = 0.5 * (np.abs(am) @ np.abs(bm)) + np.abs(cf)
    ulp   = {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}[kind]
    assert np.all(np.abs(got - want) <= (2.0 ** -24 * np.sqrt(k) + 2.0 ** -22) * scale + ulp * np.abs(want) + 2.0 ** -25)


def test_k_rows_beyond_the_last_are_zeros(gpu):
    """an infinite last k-row of B reaches the elements it belongs to and no others"""
    m, n, k = 1672, 1928, 1001
    rng = np.random.default_rng(3)
    a, b = rng.standard_normal((k, m)).astype(np.float16), rng.standard_normal((k, n)).astype(np.float16)
    b[-1, 5] = np.inf
    got = call_cublas(a[None], b[None], (1, m, n), "float16", True, False)[0]
    assert np.array_equal(np.isinf(got[:, 5]), a[-1] != 0) and np.all(np.isfinite(np.delete(got, 5, axis=1)))
