"""A program's graph replay runs what its eager run ran: an fp32 product whose K is split and the channel sums of a training
batch norm keep their partial sums in scratch that the eager run has sized, whether or not the library's page of zeros
exists (neither reads it, so it does not in a process that has run nothing else - hence the child process).  Equal bit for
bit, replayed several times with eager work between."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

CHILD = """
import numpy as np
from cinn_amd import runtime
from cinn_amd.common import DefaultAMDGPUTarget, Float
from cinn_amd.frontend import Computation, NetBuilder

rng = np.random.default_rng(3)


def check(name, build):
    feeds, results = {}, []
    for replay in (False, True):
        b, stream = NetBuilder(name), runtime.Stream()

        def given(n, shape):
            feeds.setdefault(n, rng.standard_normal(shape).astype(np.float32))
            return b.create_input(Float(32), list(shape), n)
        outs = build(b, given)
        comp = Computation.build_and_compile(DefaultAMDGPUTarget(), b, outputs=outs, stream=stream)
        for n, t in feeds.items():
            comp.get_tensor(n).from_numpy(t)
        for i in range(4 if replay else 1):
            (comp.execute_graph if replay else comp.execute)()
            stream.synchronize()
            results.append([comp.get_tensor(o.id).numpy() for o in outs])
            for o in outs:
                comp.get_tensor(o.id).from_numpy(np.zeros(o.shape(), np.float32))
    for r in results[1:]:
        for got, want in zip(r, results[0]):
            assert np.array_equal(got, want), (name, np.abs(got - want).max())
    print(name, flush=True)


for m, n, k in ((3, 768, 768), (128, 128, 4096), (70, 90, 3001)):
    check("product %d" % m, lambda b, given: [b.matmul(given("x", (m, k)), given("y", (k, n)))])


def batch_norm(b, given):
    x = given("x", (8, 23, 21, 40))
    v = [given(n, (40,)) for n in ("scale", "bias", "mean", "var")]
    y, mean, var = b.batchnorm(x, *v, is_test=False, data_layout="NHWC")[:3]
    return [y, mean, var] + list(b.batch_norm_grad(given("dy", x.shape()), x, v[0], mean, var, data_layout="NHWC"))


check("batch norm", batch_norm)
"""


def test_replay_equals_eager_run_in_a_process_of_its_own(gpu):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    done = subprocess.run([sys.executable, "-c", CHILD], cwd=root, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=100,
                          universal_newlines=True)
    assert done.returncode == 0 and done.stdout.rstrip().endswith("batch norm"), done.stdout[-2000:]
