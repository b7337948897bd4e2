"""Groups of little data that stand between library calls share a launch with a later or an earlier kernel (OrderForMerging): never
before what they read, never after what reads them, and not past a group that may update in place what they read."""
import numpy as np
import pytest

from cinn_amd.common import DefaultAMDGPUTarget, Float
from cinn_amd.frontend import Computation, NetBuilder

pytestmark = pytest.mark.gpu


def run(b, outs, feeds):
    comp = Computation.build_and_compile(DefaultAMDGPUTarget(), b, outputs=outs)
    for name, v in feeds.items():
        comp.get_tensor(name).from_numpy(v)
    for _ in range(2):
        comp.execute()
    names = [comp.instruction_info(i)[0] for i in range(comp.num_instructions())]
    return [comp.get_tensor(o.id).numpy() for o in outs], names


def inputs(b, shapes, seed=3):
    rng = np.random.default_rng(seed)
    feeds = {n: rng.uniform(0.5, 1.5, s).astype(np.float32) for n, s in shapes.items()}
    return feeds, [b.create_input(Float(32), list(s), n) for n, s in shapes.items()]


def near(got, want):  # sums of 64 products in fp32, or a few operations
    np.testing.assert_allclose(got, want, rtol=2.0 ** -18, atol=0)


def test_kernels_between_products_share_launches(gpu):
    b = NetBuilder("between")
    feeds, (x, w, u, v) = inputs(b, {"x": (64, 64), "w": (64, 64), "u": (48,), "v": (96,)})
    y = b.matmul(x, w)
    early = b.sqrt(u)                 # needs neither product: joins the kernel behind the second
    z = b.matmul(y, w)
    late = b.sqrt(b.add(z, x))
    last = b.matmul(late, w)
    other = b.multiply(v, v)          # needs nothing: joins the kernel before the last product
    got, names = run(b, [early, late, last, other], feeds)
    assert len(names) == 4 and sum("and_2_more" in n for n in names) == 1, names
    x, w, u, v = (feeds[n].astype(np.float64) for n in ("x", "w", "u", "v"))
    near(got[0], np.sqrt(u))
    near(got[1], np.sqrt((x @ w) @ w + x))
    near(got[2], np.sqrt((x @ w) @ w + x) @ w)
    near(got[3], v * v)


def test_a_kernel_stays_between_what_it_reads_and_what_reads_it(gpu):
    b = NetBuilder("chain")
    feeds, (x, w, u) = inputs(b, {"x": (64, 64), "w": (64, 64), "u": (64,)})
    w = b.scale(w, 2.0 ** -6)
    y = b.matmul(x, w)
    row = b.reduce_sum(y, [0])        # needs the first product, and the second needs it
    z = b.matmul(b.add(y, b.multiply(row, u)), w)
    tail = b.sqrt(z)
    got, _ = run(b, [row, z, tail], feeds)
    x, w, u = (feeds[n].astype(np.float64) for n in ("x", "w", "u"))
    w *= 2.0 ** -6
    row = (x @ w).sum(0)
    near(got[0], row)
    near(got[1], (x @ w + row * u) @ w)
    near(got[2], np.sqrt((x @ w + row * u) @ w))


def test_an_update_does_not_pass_other_readers_of_its_input(gpu):
    """new = 0.9 state + 0.1 u may be bound to state's memory: what reads the old state element by element is in the same kernel (fused
    with it, in one thread) or before it.  Readers of other elements: test_merge_updates"""
    b = NetBuilder("update")
    feeds, (x, w, state, u) = inputs(b, {"x": (64, 64), "w": (64, 64), "state": (64,), "u": (64,)})
    seen = b.multiply(state, state)
    y = b.matmul(x, w)
    z = b.matmul(b.add(y, seen), w)
    new = b.add(b.scale(state, 0.9), b.scale(u, 0.1))
    tail = b.exp(b.scale(b.matmul(z, w), 2.0 ** -20))
    comp = Computation.build_and_compile(DefaultAMDGPUTarget(), b, outputs=[y, z, new, tail])
    names = [comp.instruction_info(i) for i in range(comp.num_instructions())]
    writer = [i for i, (_, args) in enumerate(names) if new.id in args]
    readers = [i for i, (_, args) in enumerate(names) if state.id in args]
    assert len(writer) == 1 and writer[0] == max(readers), names
    for name, v in feeds.items():
        comp.get_tensor(name).from_numpy(v)
    comp.execute()
    near(comp.get_tensor(new.id).numpy(), 0.9 * feeds["state"].astype(np.float64) + 0.1 * feeds["u"])
