"""MD with one launch between evaluations (largest structure up to 8192 atoms)
against the four-launch form: small structures run alone and beside one of
8200 atoms, which takes the whole batch to the four launches.  The step's
arithmetic is the same; the forces' sums differ in order (1e-12 relative), so
positions, momenta and log agree to 1e-9 after 18 steps (two blocks of steps,
the second one partial)."""
import numpy as np
import pytest

import gapx
from gapx import synth
from test_gpu_descriptor_forms import FORMS, model_for

pytestmark = pytest.mark.gpu
MASS = {1: 1.008, 8: 15.999, 22: 47.867}


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if gapx.device_count() == 0:
        pytest.skip("no GPU visible")


@pytest.mark.parametrize("sizes,taut,fixcm,log", [((1, 5, 64), 500.0, True, True), ((255, 256, 257), 5.0, False, True),
                                                  ((300,), 0.0, True, False)])
def test_one_launch_matches_four(sizes, taut, fixcm, log):
    small = [synth.jittered_structures(1, n, n, 1.0 / 18.0, (1, 8, 22), n)[0] for n in sizes]
    big = synth.jittered_structures(1, 8200, 8200, 1.0 / 18.0, (1, 8, 22), 1)[0]
    m = gapx.Model.from_model(model_for(FORMS["eta1_zeta1"], small[-1], np.random.default_rng(3)))
    n = sum(sizes)

    def run(structs):
        mass = np.concatenate([[MASS[int(z)] for z in s["species"]] for s in structs])
        p0 = np.random.default_rng(4).normal(size=(len(mass), 3)) * np.sqrt(mass * 300.0 * gapx.KB)[:, None]
        ctx = gapx.Context(m)
        ctx.load(structs, 6.0)
        out = ctx.md(mass, 18, dt_fs=0.5, temperature=300.0, taut_fs=taut, fixcm=fixcm, momenta=p0, log=log)
        return ctx.positions()[:n], ctx.momenta()[:n], (out[:, :len(sizes)] if log else None)

    one, four = run(small), run(small + [big])
    dx, dp = np.abs(one[0] - four[0]).max(), np.abs(one[1] - four[1]).max()
    print(sizes, dx, dp, flush=True)
    assert dx <= 1e-9 and dp <= 1e-9
    if log:
        assert np.abs(one[2] - four[2]).max() <= 1e-9 * max(1.0, np.abs(four[2]).max())
