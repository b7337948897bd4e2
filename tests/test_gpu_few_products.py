"""fp32 products with both operands in runs of K on the kernel whose wavefronts share K (TryFewProduct): one row, rows and columns
at the edges of its tiles of 16 to 64, K of one step and of uneven shares, alpha, beta and a bias, and the sizes next to them that other
kernels run: columns that are no multiple of four, K that is no whole step, whole tiles of 128.

Bounds: as in test_gpu_gemm_flex (sums of k products in fp32, one rounding of the result)."""
import numpy as np
import pytest

from cinn_amd.common import DefaultAMDGPUTarget, Float
from cinn_amd.frontend import Computation, NetBuilder

from test_gpu_gemm import call_cublas

pytestmark = pytest.mark.gpu

SHAPES = [(1, 4, 32), (1, 1208, 192), (7, 3840, 1280), (15, 20, 4096), (16, 16, 64), (17, 36, 96), (33, 68, 352), (63, 100, 32), (64, 60, 2048),
          (129, 132, 736), (250, 260, 512), (1097, 16, 32), (700, 64, 96), (340, 3328, 64), (10, 66, 64), (10, 64, 65), (10, 64, 16), (128, 128, 32)]


def check(got, a, b, scale, rest, k):
    want = scale * (a @ b.T) + rest
    size = scale * (np.abs(a) @ np.abs(b.T)) + np.abs(rest)
    assert np.all(np.abs(got.astype(np.float64) - want) <= (2.0 ** -24 * np.sqrt(k) + 2.0 ** -22) * size + 2.0 ** -24 * np.abs(want) + 2.0 ** -25)


@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (0.5, -1.0)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_product(gpu, m, n, k, alpha, beta):
    rng = np.random.default_rng(m + n + k)
    a, b, c = (rng.standard_normal(s).astype(np.float32) for s in ((m, k), (n, k), (m, n)))
    got = call_cublas(a, b, (m, n), "float32", False, True, alpha=alpha, beta=beta, c_init=c)
    check(got, a.astype(np.float64), b.astype(np.float64), alpha, beta * c.astype(np.float64), k)


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_with_a_bias_and_next_to_another_product(gpu, m, n, k):
    rng = np.random.default_rng(m + n + k)
    feeds = {"x": rng.standard_normal((m, k)), "w": rng.standard_normal((n, k)), "v": rng.standard_normal((n, k)), "c": rng.standard_normal(n)}
    feeds = {name: v.astype(np.float32) for name, v in feeds.items()}
    b = NetBuilder("layer")
    x, w, v, c = (b.create_input(Float(32), list(feeds[name].shape), name) for name in ("x", "w", "v", "c"))
    outs = [b.add(b.matmul(x, w, False, True), c), b.matmul(x, v, False, True)]
    comp = Computation.build_and_compile(DefaultAMDGPUTarget(), b, outputs=outs)
    for name, value in feeds.items():
        comp.get_tensor(name).from_numpy(value)
    for _ in range(2):
        comp.execute()
    x, w, v, c = (feeds[name].astype(np.float64) for name in ("x", "w", "v", "c"))
    check(comp.get_tensor(outs[0].id).numpy(), x, w, 1.0, c, k)
    check(comp.get_tensor(outs[1].id).numpy(), x, v, 1.0, 0.0, k)
