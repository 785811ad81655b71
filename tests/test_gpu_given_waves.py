"""Launch shapes of the descriptor kernels that a caller gives run as given,
whatever the batch's size, and the ones a load picks by the batch's size (eight
waves per atom for small batches, down to one) agree with one wave per atom."""
import numpy as np
import pytest

import gapx
from gapx import synth
from test_gpu_descriptor_forms import FORMS, model_for

pytestmark = pytest.mark.gpu

NAMES = ["eta3_zeta5", "eta5_zeta2", "eta9_zeta2", "eta4_two_radial_cutoffs", "no_grid"]


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if gapx.device_count() == 0:
        pytest.skip("no GPU visible")


def cell(form):
    s = synth.structure(23, 23 * 14.0, (1, 8, 22), np.random.default_rng(5), min_dist=1.3)
    return s, gapx.Model.from_model(model_for(FORMS[form], s, np.random.default_rng(6)))


def evaluate(m, s, copies, flags, **shape):
    ctx = gapx.Context(m)
    ctx.load([s] * copies, 6.0)
    if shape:
        ctx.set_tuning(flags, gpr_rows=64, gpr_blocks=1, halves=0, **shape)
    ctx.run(flags)
    n = len(s["species"])
    r = ctx.results()
    return dict(x=ctx.features(dedx=False)[0][:n], forces=r["forces"][:n], eatom=r["eatom"][:n], energy=r["energy"][:1])


# the same waves add the same numbers in the same order: every bit agrees
@pytest.mark.parametrize("flags", [gapx.GRAD, gapx.GRAD | gapx.MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("form", NAMES)
def test_given_waves_do_not_follow_the_size(form, flags):
    s, m = cell(form)
    for w in (1, 2, 4):
        few, many = (evaluate(m, s, copies, flags, waves_fwd=w, waves_bwd=w) for copies in (1, 60))
        print(form, w, flush=True)
        for k in few:
            assert np.array_equal(few[k], many[k]), (w, k)


# FP64 sums in another order: 1e-12 of the largest value.  Mixed: the bars
# between mixed and FP64 (1e-4 of the largest force, 1e-5 of the sum of |E_i|).
@pytest.mark.parametrize("form", NAMES)
def test_shapes_by_size_against_one_wave(form):
    s, m = cell(form)
    for copies in (1, 31, 140):
        for flags in (gapx.GRAD, gapx.GRAD | gapx.MIXED):
            a, b = evaluate(m, s, copies, flags), evaluate(m, s, copies, flags, waves_fwd=1, waves_bwd=1)
            print(form, copies, flags, flush=True)
            fp64 = flags == gapx.GRAD
            bar = {k: 1e-12 * max(1.0, np.abs(b[k]).max()) for k in b} if fp64 else \
                dict(forces=1e-4 * np.abs(b["forces"]).max(), energy=1e-5 * np.abs(b["eatom"]).sum(),
                     eatom=1e-5 * np.abs(b["eatom"]).sum())
            for k in bar:
                assert np.abs(a[k] - b[k]).max() <= bar[k], (copies, flags, k)
