"""A structure's surrogate energy does not depend on how many structures share
the call: the surrogate rounds FP32 features to BF16, so features have to keep
their bits whatever the batch's size."""
import numpy as np
import pytest

import gapx
import mlp_oracle as mo
from gapx import synth
from helpers import workload_model

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if gapx.device_count() == 0:
        pytest.skip("no GPU visible")


@pytest.mark.parametrize("flags", [gapx.MIXED, gapx.GRAD | gapx.MIXED, 0], ids=["mixed", "mixed_grad", "fp64"])
def test_alone_and_in_a_population(flags):
    m = gapx.Model.from_model(workload_model("ternary4k"))
    net = gapx.MLP(seed=3)
    net.set_params(mo.init_params(23).astype(np.float32).astype(np.float64))
    s = synth.jittered_structures(1, 24, 24, 0.07, (1, 8, 22), seed=31)[0]
    ref = None
    for copies in (1, 20, 60, 200):  # eight, two and one waves per atom in GAP runs
        ctx = gapx.Context(m)
        ctx.load([s] * copies, 6.0)
        ctx.run_surrogate(net, flags)
        r = ctx.results()
        out = (ctx.features(dedx=False)[0].reshape(copies, 24, -1), r["eatom"].reshape(copies, 24), r["energy"])
        print(copies, r["energy"][0], flush=True)
        ref = ref or [a[0] for a in out]
        for a, b in zip(out, ref):
            assert all(np.array_equal(x, b) for x in a), copies
        ctx.close()
    net.close()
    m.close()
