"""Matrix products of a program that do not depend on each other, in one launch (ProductGroup, flex_group_kernel): one row, column
or k; extents at the edges of the 64x64 tiles; products of very different K, so that some are split and some are not; more products
than a launch takes; products that need another's result; eager runs and replays.

Bounds: as in test_gpu_gemm_flex (sums of k products in fp32, one rounding of the result)."""
import numpy as np
import pytest

from cinn_amd import runtime
from cinn_amd.common import BFloat16, DefaultAMDGPUTarget, Float, bfloat16_bits_to_float32, float32_to_bfloat16_bits
from cinn_amd.frontend import Computation, NetBuilder

from launch_counts import GROUP, launches

pytestmark = pytest.mark.gpu

TYPES = {"float32": Float(32), "float16": Float(16), "bfloat16": BFloat16()}
ULP = {"float32": 2.0 ** -24, "float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}


class Net:
    def __init__(self, kind):
        self.kind, self.b, self.data, self.rng = kind, NetBuilder("group"), {}, np.random.default_rng(7)

    def input(self, name, shape, scale=1.0):
        v = (self.rng.standard_normal(shape) * scale).astype(np.float32)
        v = float32_to_bfloat16_bits(v) if self.kind == "bfloat16" else v.astype(self.kind)
        self.data[name] = v
        return self.b.create_input(TYPES[self.kind], list(shape), name)

    def compile(self, outs):
        self.stream = runtime.Stream()
        comp = Computation.build_and_compile(DefaultAMDGPUTarget(), self.b, outputs=outs, stream=self.stream)
        for name, v in self.data.items():
            comp.get_tensor(name).from_numpy(v)
        return comp

    def value(self, v):
        return (bfloat16_bits_to_float32(v) if self.kind == "bfloat16" else v).astype(np.float64)

    def get(self, comp, out):
        return self.value(comp.get_tensor(out.id).numpy())

    def check(self, got, a, b, shift=0.0):
        k = a.shape[1]
        want, scale = a @ b + shift, np.abs(a) @ np.abs(b) + np.abs(shift)
        bound = (2.0 ** -24 * np.sqrt(k) + 2.0 ** -22) * scale + ULP[self.kind] * np.abs(want) + 2.0 ** -25
        assert got.shape == want.shape and np.all(np.abs(got - want) <= bound)


@pytest.mark.parametrize("kind", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("rows,inp,out", [(1, 1, 1), (1, 70, 3), (33, 17, 65), (65, 63, 129), (64, 65, 64), (127, 1001, 62), (700, 333, 190),
                                          (5001, 33, 17), (40, 2050, 1), (300, 130, 2001)])
def test_a_layers_three_products_and_two_more(gpu, rows, inp, out, kind):
    net = Net(kind)
    x, w, dy, c, v = (net.input(n, s) for n, s in (("x", (rows, inp)), ("w", (inp, out)), ("dy", (rows, out)), ("c", (out,)), ("v", (inp, out))))
    b = net.b
    outs = [b.add(b.matmul(x, w), c), b.matmul(dy, w, False, True), b.matmul(x, dy, True, False), b.matmul(x, v), b.matmul(dy, v, False, True)]
    comp = net.compile(outs)
    x, w, dy, c, v = (net.value(net.data[n]) for n in ("x", "w", "dy", "c", "v"))
    for replay in (False, True, False, True, True):
        for o in outs:
            t = comp.get_tensor(o.id)
            t.from_numpy(np.ones_like(t.numpy()))
        (comp.execute_graph if replay else comp.execute)()
        net.stream.synchronize()
        got = [net.get(comp, o) for o in outs]
        for at, (p, q, shift) in enumerate(((x, w, c), (dy, w.T, 0.0), (x.T, dy, 0.0), (x, v, 0.0), (dy, v.T, 0.0))):
            net.check(got[at], p, q, shift)


# which of these are one launch: small ones are, and those of one small tile in all products, until a tile of 128 or the small tiles of
# fp32 are estimated to be faster one by one
@pytest.mark.parametrize("kind", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("rows,inp,out,groups", [(37, 75, 247, 1), (665, 233, 670, 1), (33, 17, 65, 1), (127, 1001, 62, 1), (4887, 301, 2123, 0)])
def test_a_layers_three_products_in_one_launch(gpu, rows, inp, out, groups, kind):
    net = Net(kind)
    x, w, dy = (net.input(n, s) for n, s in (("x", (rows, inp)), ("w", (inp, out)), ("dy", (rows, out))))
    comp = net.compile([net.b.matmul(x, w), net.b.matmul(dy, w, False, True), net.b.matmul(x, dy, True, False)])
    with launches() as count:
        comp.execute()
        net.stream.synchronize()
    assert count(GROUP) == groups


@pytest.mark.parametrize("kind", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("m,k", [(1, 1), (50, 65), (130, 257), (800, 70)])
def test_products_that_need_another_ones_result(gpu, m, k, kind):
    net = Net(kind)
    # x u has values of about 1: the squares' sum of 800 of them is within fp16's 65504
    x, u, v, w = (net.input(n, s, k ** -0.5) for n, s in (("x", (m, k)), ("u", (k, k)), ("v", (k, k)), ("w", (k, k))))
    b = net.b
    first = b.matmul(x, u)
    outs = [first, b.matmul(first, v), b.matmul(x, w), b.matmul(first, w, False, True), b.matmul(first, first, True, False)]
    comp = net.compile(outs)
    for _ in range(3):
        comp.execute()
    net.stream.synchronize()
    got = [net.get(comp, o) for o in outs]
    x, u, v, w = (net.value(net.data[n]) for n in ("x", "u", "v", "w"))
    for at, (p, q) in enumerate(((x, u), (got[0], v), (x, w), (got[0], w.T), (got[0].T, got[0]))):
        net.check(got[at], p, q)
