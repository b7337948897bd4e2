"""Where the bias of a layer in training is added (names of the calls of compiled programs, no GPU needed): in the product, or by the
generated kernel that reads a small sum."""
import pytest

from cinn_amd.common import Float
from cinn_amd.frontend import NetBuilder

from helpers import compile_only


@pytest.mark.parametrize("bits", [16, 32])
@pytest.mark.parametrize("m,n,reader,inside", [
    (71, 331, None, (True, True)),         # fp16, fp32
    (71, 331, "relu", (False, False)),
    (71, 331, "matmul", (True, False)),    # a call of the library adds nothing on its way
    (771, 2122, "relu", (True, False)),
])
def test_where_the_bias_is_added(m, n, reader, inside, bits):
    b, k = NetBuilder("layer"), 48
    x, w, c = (b.create_input(Float(bits), s, e) for e, s in (("x", [m, k]), ("w", [k, n]), ("c", [n])))
    y = b.add(b.matmul(x, w), c)
    if reader == "relu":
        y = b.relu(y)
    elif reader == "matmul":
        y = b.matmul(y, b.create_input(Float(bits), [n, 16], "v"))
    comp = compile_only(b, [y])
    names = [comp.instruction_info(i)[0] for i in range(comp.num_instructions())]
    assert any("matmul_bias" in e for e in names) == inside[bits == 32], names
