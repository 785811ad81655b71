"""Grid-form backward from the per-eta LDS records: every number of zetas, in
FP64 against the CPU oracle at the parity bar and mixed against FP64 at the
bars of the other forms, for an ordinary and a long list and one to four waves
per atom (the records' place in LDS follows the radial lines and the waves)."""
import numpy as np
import pytest

import gapx
import oracle
from gapx import synth
from test_gpu_descriptor_forms import grid_sf, model_for

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if gapx.device_count() == 0:
        pytest.skip("no GPU visible")


ZETAS = {1: (2,), 2: (1, 4), 3: (1, 2, 4), 4: (1, 2, 4, 8), 5: (1, 2, 4, 8, 16)}


# about 64 and 180 neighbours
@pytest.mark.parametrize("vpa", [14.1, 5.0])
@pytest.mark.parametrize("nz", sorted(ZETAS))
@pytest.mark.parametrize("n_eta", [2, 9])
def test_records(n_eta, nz, vpa):
    rng = np.random.default_rng(100 * n_eta + 10 * nz + int(vpa))
    s = synth.jittered_structures(1, 12, 12, 1.0 / vpa, (1, 8, 22), n_eta + nz, jitter=0.1)[0]
    om = model_for(grid_sf(n_eta, ZETAS[nz], n_rad=5 + nz), s, rng)
    ref = oracle.gap_calc(om, s["species"], s["lat"], s["pos"], 6.0, mode="sparse", nthreads=4)
    scale = max(1.0, np.abs(ref["forces"]).max())
    ctx = gapx.Context(gapx.Model.from_model(om))
    ctx.load([s], 6.0)
    for w in (1, 2, 4):
        print(n_eta, nz, vpa, w, flush=True)
        for f in (gapx.GRAD, gapx.GRAD | gapx.MIXED):
            ctx.set_tuning(f, waves_fwd=w, waves_bwd=w)
        ctx.run(gapx.GRAD)
        r = ctx.results()
        assert abs(r["energy"][0] - ref["energy"]) / 12 < 1e-9
        assert np.abs(r["forces"] - ref["forces"]).max() < 1e-7 * scale
        assert np.abs(r["stress"][0] - ref["stress"]).max() < max(1e-6, 1e-8 * np.abs(ref["stress"]).max())
        ctx.run(gapx.GRAD | gapx.MIXED)
        x = ctx.results()
        assert np.abs(x["forces"] - r["forces"]).max() < 1e-4 * np.abs(r["forces"]).max()
        assert abs(x["energy"][0] - r["energy"][0]) < 1e-5 * np.abs(r["eatom"]).sum()
