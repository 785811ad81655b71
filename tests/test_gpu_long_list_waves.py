"""The waves per atom that a load gives the generic forward: long lists take four
where one-wave workgroups would leave few waves on a CU (their LDS, or too few
atoms), short ones and grid tables follow the number of atoms alone; and results
do not depend on it (FP64, 1e-12 of the largest value)."""
import numpy as np
import pytest

import gapx
from gapx import synth
from test_gpu_descriptor_forms import FORMS, model_for

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if gapx.device_count() == 0:
        pytest.skip("no GPU visible")


def cell(n, vpa):
    return synth.jittered_structures(1, n, n, 1.0 / vpa, (1, 8, 22), n, jitter=0.1)[0]


# five cutoffs (6, 5, 4, 4.5, 3.5): slots for 1.25 x 181 neighbours leave 6 (FP64)
# and 13 (FP32) one-wave workgroups on a CU, for 1.25 x 65 neighbours 16 and more
@pytest.mark.parametrize("form,vpa,n,fp64,mixed", [
    ("no_grid", 5.0, 1300, 4, 4), ("no_grid", 5.0, 2100, 4, 4), ("no_grid", 5.0, 4200, 4, 4),
    ("no_grid", 14.0, 1300, 2, 2), ("no_grid", 14.0, 2100, 1, 1), ("no_grid", 14.0, 4200, 1, 1),
    ("eta4_zeta4", 5.0, 1300, 2, 2), ("eta4_zeta4", 5.0, 4200, 1, 1)])
def test_waves_of_the_forward(form, vpa, n, fp64, mixed):
    small = synth.structure(23, 23 * 14.0, (1, 8, 22), np.random.default_rng(5), min_dist=1.3)
    m = gapx.Model.from_model(model_for(FORMS[form], small, np.random.default_rng(6)))
    ctx = gapx.Context(m)
    ctx.load([cell(n, vpa)], 6.0)
    assert ctx.tuning(gapx.GRAD)["waves_fwd"] == fp64
    assert ctx.tuning(gapx.GRAD | gapx.MIXED)["waves_fwd"] == mixed
    ctx.run(gapx.GRAD)
    a, x = ctx.results(), ctx.features(dedx=False)[0]
    ctx.set_tuning(gapx.GRAD, waves_fwd=1, waves_bwd=1, gpr_rows=64, gpr_blocks=1, halves=0)
    ctx.run(gapx.GRAD)
    b, y = ctx.results(), ctx.features(dedx=False)[0]
    print(form, vpa, n, flush=True)
    assert np.abs(x - y).max() <= 1e-12 * np.abs(y).max()
    for k in ("energy", "forces", "stress", "eatom"):
        assert np.abs(a[k] - b[k]).max() <= 1e-12 * max(1.0, np.abs(b[k]).max()), k
