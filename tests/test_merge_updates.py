"""A group that may update a program input in place - it reads the input and its result has the input's type and size, so that a
caller may have bound both to the same memory - never shares a launch with another reader of that input, whose blocks
would run next to its own: neither where the two follow each other nor where a group is moved (RunEnd, OrderForMerging)."""
import pytest

from cinn_amd.common import DefaultAMDGPUTarget, Float
from cinn_amd.frontend import Computation, NetBuilder

READERS = {
    "slice": lambda b, s: b.slice(s, [0], [7], [50]),
    "sum": lambda b, s: b.reduce_sum(s, [1]),
    "softmax": lambda b, s: b.softmax(s, axes=[-1]),
    "sum_of_a_view": lambda b, s: b.reduce_sum(b.reshape(s, [32, 128]), [1]),
    "sum_of_a_view_of_a_view": lambda b, s: b.reduce_sum(b.reshape(b.reshape(s, [4096]), [128, 32]), [1]),
}


def instructions(b, outs):
    comp = Computation.build_and_compile(DefaultAMDGPUTarget(), b, outputs=outs)
    return [comp.instruction_info(i)[1] for i in range(comp.num_instructions())]


@pytest.mark.parametrize("reader", sorted(READERS))
@pytest.mark.parametrize("between", ["products", "nothing"])
@pytest.mark.parametrize("result", ["itself", "a view"])
def test_reader_and_update_have_launches_of_their_own(reader, between, result):
    b = NetBuilder("update")
    x, w, state, u = (b.create_input(Float(32), [64, 64], name) for name in ("x", "w", "state", "u"))
    seen = READERS[reader](b, state)
    outs = [seen]
    if between == "products":
        outs.append(b.matmul(x, w))
    new = b.add(b.scale(state, 0.9), b.scale(u, 0.1))
    returned = new if result == "itself" else b.reshape(new, [4096])
    outs.append(returned)
    if between == "products":
        outs.append(b.matmul(outs[1], w))
    args = instructions(b, outs)
    reads = [i for i, a in enumerate(args) if seen.id in a]
    updates = [i for i, a in enumerate(args) if new.id in a or returned.id in a]
    assert len(reads) == 1 and updates and reads[0] < min(updates), args


# an update that reads more than it writes over, as a softmax: kept apart by what stands between the two in the program, which no
# move takes out of the way; next to each other they share a launch, as they always have
@pytest.mark.parametrize("reader", sorted(set(READERS) - {"softmax", "sum"}))  # (those of whole rows are fused with the softmax, in one thread)
@pytest.mark.parametrize("first", ["reader", "update"])
@pytest.mark.parametrize("between", ["products", "nothing"])
def test_update_by_rows(reader, first, between):
    b = NetBuilder("rows")
    x, w, state = (b.create_input(Float(32), [64, 64], name) for name in ("x", "w", "state"))
    parts = {"reader": lambda: READERS[reader](b, state), "update": lambda: b.softmax(state, axes=[-1])}
    second = "update" if first == "reader" else "reader"
    outs = {first: parts[first]()}
    if between == "products":
        y = outs["y"] = b.matmul(x, w)
    outs[second] = parts[second]()
    if between == "products":
        outs["z"] = b.matmul(y, w)
    args = instructions(b, list(outs.values()))
    at = {name: [i for i, a in enumerate(args) if outs[name].id in a] for name in ("reader", "update")}
    assert len(at["reader"]) == len(at["update"]) == 1
    if between == "products":
        assert at[first][0] < at[second][0], args
    else:
        assert at[first] == at[second], args


def test_readers_that_update_nothing_share_a_launch():
    b = NetBuilder("readers")
    x, w, state = (b.create_input(Float(32), [64, 64], name) for name in ("x", "w", "state"))
    total = b.reduce_sum(state, [1])
    y = b.matmul(x, w)
    part = b.slice(state, [0], [7], [50])
    args = instructions(b, [total, y, part, b.matmul(y, w)])
    assert len(args) == 3 and any(total.id in a and part.id in a for a in args), args
