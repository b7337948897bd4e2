"""Which layers FuseRowProducts takes: names of the calls of compiled programs (no GPU needed), and values."""
import numpy as np
import pytest

from cinn_amd.common import Float
from cinn_amd.frontend import NetBuilder

from helpers import compile_only, run

M, K, N = 8, 64, 32


def names(comp):
    return [comp.instruction_info(i)[0] for i in range(comp.num_instructions())]


def pointwise_layer(geometry, pixels=1):
    """a folded 1x1 convolution and batch norm on images of one pixel, seen as a matrix before and behind it, and gelu"""
    b, rng, data = NetBuilder("pointwise"), np.random.default_rng(3), {}

    def put(name, shape, low=-1.0, const=True):
        data[name] = rng.uniform(low, 1.0, shape).astype(np.float16)
        v = b.create_input(Float(16), list(shape), name)
        v.set_const(const)
        return v

    x, w = put("x", (M, K), const=False), put("w", (N, K))
    z = b.conv2d(b.reshape(x, [M, 1, 1, K]), b.reshape(w, [N, 1, 1, K]), data_format="NHWC", **geometry)
    norm = b.batchnorm(z, put("g", (N,)), put("b", (N,)), put("m", (N,)), put("v", (N,), 0.5), data_layout="NHWC")[0]
    return b, b.gelu(b.reshape(norm, [M, N])), data


GEOMETRIES = [dict(), dict(strides=[3, 3], paddings=[1, 1])]  # the latter's one output pixel sees padding alone


@pytest.mark.parametrize("geometry", GEOMETRIES)
def test_pointwise_layer_is_a_product_only_where_it_sees_its_pixel(geometry):
    b, y, _ = pointwise_layer(geometry)
    assert any("matmul_rows" in e for e in names(compile_only(b, [y]))) == (geometry == {})


@pytest.mark.gpu
@pytest.mark.parametrize("geometry", GEOMETRIES)
def test_pointwise_layer_values(gpu, geometry):
    from scipy.special import erf
    b, y, data = pointwise_layer(geometry)
    (got,), _ = run(b, data, [y])
    d = {e: v.astype(np.float64) for e, v in data.items()}
    product = d["x"] @ d["w"].T if geometry == {} else np.zeros((M, N))
    scale = d["g"] / np.sqrt(d["v"] + 1e-5)
    want = product * scale + d["b"] - d["m"] * scale
    want = want * 0.5 * (1 + erf(want / np.sqrt(2)))
    # 64 terms in fp32, results rounded to fp16 once behind the product and once behind gelu (|gelu'| < 1.13)
    size = np.abs(product * scale) + np.abs(d["b"]) + np.abs(d["m"] * scale)
    assert np.all(np.abs(got - want) <= 2.2 * 2.0 ** -11 * size + 2.0 ** -24)


def linear_layer(m, k, n, norm, gelu):
    b = NetBuilder("linear")

    def put(name, shape, const=True):
        v = b.create_input(Float(16), list(shape), name)
        v.set_const(const)
        return v

    x = put("x", (m, k), False)
    if norm:
        x = b.paddle_layer_norm(x, put("g", (k,)), put("s", (k,)))[0]
    y = b.add(b.matmul(x, put("w", (k, n))), put("c", (n,)))
    return b, b.gelu(y) if gelu else y


# gelu goes inside, the norm up to 512 blocks (32 columns x 16 rows) and with a short K (measured: ChooseRowFusion); without whole
# K steps of 64 one round of blocks (16 columns) takes everything along, several only what is faster inside
@pytest.mark.parametrize("m,k,n,norm,gelu,calls", [
    (8, 768, 3072, True, True, 1), (16, 384, 4096, True, False, 1), (64, 320, 1024, True, True, 1),
    (48, 384, 6272, True, False, 1),
    (64, 768, 8192, True, True, 2),    # the norm is a kernel of its own
    (16, 128, 8192, True, True, 1),
    (16, 960, 8192, True, False, 1),
    (48, 1280, 4096, True, True, 1),
    (64, 960, 8192, False, True, 1),
    (64, 1280, 4096, True, False, 1), (64, 1024, 4096, True, False, 2), (32, 1024, 4096, True, False, 1), (64, 1280, 4128, True, False, 2), (64, 448, 4128, True, False, 2),
    (48, 416, 6272, True, False, 2), (64, 800, 8192, True, True, 3), (16, 160, 8192, True, True, 2), (8, 800, 3072, True, True, 1),
])
def test_what_a_product_of_few_rows_takes_along(m, k, n, norm, gelu, calls):
    b, y = linear_layer(m, k, n, norm, gelu)
    got = names(compile_only(b, [y]))
    assert len(got) == calls, got


# results in other than whole groups of four columns run on the kernel without rings, and go by its rule
@pytest.mark.parametrize("width,calls", [(2050, 2), (2052, 1)])
def test_what_a_product_of_several_results_takes_along(width, calls):
    b, y = linear_layer(32, 384, 2 * width, True, False)
    got = names(compile_only(b, [b.slice(y, [1], [0], [width]), b.slice(y, [1], [width], [2 * width])]))
    assert len(got) == calls and any("matmul_rows" in e for e in got), got


@pytest.mark.parametrize("flag,taken", [("0", False), ("1", True)])
def test_switch_of_the_kernel(monkeypatch, flag, taken):
    monkeypatch.setenv("FLAGS_cinn_hip_gemm_skinny", flag)
    b, y = linear_layer(8, 256, 512, True, True)
    assert any("matmul_rows" in e for e in names(compile_only(b, [y]))) == taken


def norm_and_layers(fetch, readers=1, epsilon=1e-5):
    """a layer norm, `readers` linear layers of its result; `fetch`: which of its other results the program returns"""
    b, rng, data = NetBuilder("norm"), np.random.default_rng(5), {}

    def put(name, shape, const=True):
        data[name] = (rng.standard_normal(shape) + (1.0 if name == "g" else 0.0)).astype(np.float16)
        v = b.create_input(Float(16), list(shape), name)
        v.set_const(const)
        return v

    outs = b.paddle_layer_norm(put("x", (M, K), False), put("g", (K,)), put("s", (K,)), epsilon)
    results = [b.add(b.matmul(outs[0], put("w%d" % i, (K, N))), put("c%d" % i, (N,))) for i in range(readers)]
    return b, results + [outs[i] for i in fetch], data


# what keeps the norm a kernel of its own: its mean, variance or result is wanted, or two products that are not joined read it
@pytest.mark.parametrize("fetch,readers,inside", [([], 1, True), ([1], 1, False), ([2], 1, False), ([0], 1, False), ([], 2, False)])
def test_norms_that_are_read_by_others(fetch, readers, inside):
    b, outs, _ = norm_and_layers(fetch, readers)
    got = names(compile_only(b, outs))
    assert (len(got) == 1 and "matmul_rows" in got[0]) == inside, got


@pytest.mark.gpu
@pytest.mark.parametrize("fetch,readers,epsilon", [([], 1, 0.3), ([1], 1, 1e-5), ([2], 1, 1e-5), ([0], 1, 0.3), ([], 2, 1e-5), ([0, 1, 2], 2, 1e-5)])
def test_norm_values(gpu, fetch, readers, epsilon):
    b, outs, data = norm_and_layers(fetch, readers, epsilon)
    got, _ = run(b, data, outs)
    d = {e: v.astype(np.float64) for e, v in data.items()}
    mean, var = d["x"].mean(1), d["x"].var(1)
    norm = (d["x"] - mean[:, None]) / np.sqrt(var[:, None] + epsilon) * d["g"] + d["s"]
    u = 2.0 ** -11
    # the normalised value is rounded once (its fp32 variance loses 2^-18 or so), the sum once
    slack = (u + 2.0 ** -18) * (np.abs(norm) + np.abs(d["s"]))
    for i in range(readers):
        want = norm @ d["w%d" % i] + d["c%d" % i]
        assert np.all(np.abs(got[i] - want) <= 1.01 * (slack @ np.abs(d["w%d" % i]) + 2 * u * np.abs(want)) + 1e-4)
    wants = (norm, mean, var)
    for g, i in zip(got[readers:], fetch):
        size = (np.abs(norm) + np.abs(d["s"]), np.abs(d["x"]).mean(1), 1.0 + var)[i]
        assert np.all(np.abs(g.reshape(wants[i].shape) - wants[i]) <= 2 * u * size + 1e-6)
