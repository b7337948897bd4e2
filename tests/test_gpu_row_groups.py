"""Softmax, layer norm, sum and argmax of one tensor, one kernel of five reductions, where a row goes from a wavefront to a
block (more than 32 elements per lane; 16-bit types only with at most as many rows as CUs) and where its columns are no
multiple of a 16-byte vector; against float64."""
import numpy as np
import pytest

from cinn_amd.common import Float
from cinn_amd.frontend import NetBuilder

from helpers import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "float16"])
@pytest.mark.parametrize("rows", [1, 256, 257])
@pytest.mark.parametrize("cols", [2048, 2049, 2050, 2600, 4095, 4096])
def test_row_operators(gpu, rows, cols, dtype):
    rng = np.random.default_rng(rows + cols)
    x, gamma, beta = rng.standard_normal((rows, cols)), rng.uniform(0.5, 1.5, cols), rng.standard_normal(cols)
    b = NetBuilder("rows")
    bits = 32 if dtype == "float32" else 16
    X, G, B = (b.create_input(Float(bits), s, e) for e, s in (("x", [rows, cols]), ("g", [cols]), ("b", [cols])))
    y, mean, var = b.paddle_layer_norm(X, G, B)
    outs = [b.softmax(X, axes=[-1]), y, mean, var, b.reduce_sum(X, [1]), b.argmax(X, 1)]
    feeds = {v: a.astype(dtype) for v, a in ((X, x), (G, gamma), (B, beta))}
    got, _ = run(b, feeds, outs)
    x, gamma, beta = (feeds[v].astype(np.float64) for v in (X, G, B))
    e = np.exp(x)
    m, v = x.mean(1), x.var(1)
    want = [e / e.sum(1, keepdims=True), (x - m[:, None]) / np.sqrt(v[:, None] + 1e-5) * gamma + beta, m, v, x.sum(1)]
    # fp32 sums of `cols` terms in chains far shorter than that: 2^-24 sqrt(cols) of the sum of magnitudes; every operator rounds
    # to the type, at most eight in a row
    unit   = 2.0 ** -24 if bits == 32 else 2.0 ** -11
    scaled = np.abs((x - m[:, None]) / np.sqrt(v[:, None] + 1e-5) * gamma) + np.abs(beta)
    sizes  = (np.abs(want[0]), 1.0 + scaled, np.full(rows, 1.0), 1.0 + v, np.abs(x).sum(1))
    for g, w, size, rounded in zip(got, want, sizes, (want[0], scaled, np.abs(x).mean(1), 1.0 + v, np.abs(want[4]))):
        tolerance = 8 * unit * rounded + 2.0 ** -24 * (4 + np.sqrt(cols)) * size + (2.0 ** -24 if bits == 16 else 0)
        assert np.all(np.abs(g.reshape(w.shape).astype(np.float64) - w) <= tolerance)
    assert np.array_equal(got[5].reshape(-1), x.argmax(1))
