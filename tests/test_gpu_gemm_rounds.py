"""16-bit products where the choice of tile and split changes: 64x64 tiles with K whole and split (few tiles, a const weight
stored [N][K]), one round of 128x128 tiles or of 256x256 tiles instead of two of smaller ones; against float64 with one
rounding of the result and fp32 sums."""
import numpy as np
import pytest

from test_gpu_projections import UNIT, _Program

pytestmark = pytest.mark.gpu


def check(p, out, want, scale, k, dtype):
    (got,), names = p.run([out])
    assert len(names) == 1, names
    bound = UNIT[dtype] * np.abs(want) + k * 2.0 ** -24 * scale
    assert np.all(np.abs(got - want) <= 1.01 * bound + 1e-7)


# m, n, k: split eight, four, two ways and not at all; ragged rows and columns; around 256 tiles of 64x64
@pytest.mark.parametrize("m,n,k", [(65, 64, 4096), (96, 768, 3072), (200, 136, 2112), (130, 1280, 2048), (413, 384, 1536), (800, 384, 1536),
                                   (1024, 1024, 1024), (1025, 1032, 832), (1040, 1024, 768), (1500, 1536, 384), (800, 3072, 768)])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("residual", [False, True])
def test_const_weight(gpu, m, n, k, dtype, residual):
    p = _Program(dtype, m + n + k)
    x, x64 = p.put("x", (m, k))
    w, w64 = p.put("w", (k, n), k ** -0.5, True)
    c, c64 = p.put("c", (n,), 0.5, True)
    out, want, scale = p.b.add(p.b.matmul(x, w), c), x64 @ w64 + c64, np.abs(x64) @ np.abs(w64) + np.abs(c64)
    if residual:
        r, r64 = p.put("r", (m, n))
        out, want, scale = p.b.add(out, r), want + r64, scale + np.abs(r64)
    check(p, out, want, scale, k, dtype)


@pytest.mark.parametrize("m,n,k", [(800, 1280, 1280), (809, 1288, 768), (640, 1600, 3136), (2300, 3840, 128), (2300, 3840, 192), (4104, 2312, 256)])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_product(gpu, m, n, k, trans_b, dtype):
    p = _Program(dtype, m + n + k)
    x, x64 = p.put("x", (m, k))
    w, w64 = p.put("w", (n, k) if trans_b else (k, n), k ** -0.5)
    w64 = w64.T if trans_b else w64
    check(p, p.b.matmul(x, w, False, trans_b), x64 @ w64, np.abs(x64) @ np.abs(w64), k, dtype)
