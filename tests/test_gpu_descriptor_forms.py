"""Descriptor kernels over the forms their dispatch tells apart: grid tables
of one to nine etas and one to five zetas (the backward holds g in registers
up to four etas, in FP32 eight, and reads LDS records above), tables without a
grid, radial lines of one or several cutoff groups, and neighbour lists whose
last 64 are empty, few or nearly full.

FP64 against the CPU oracle at the parity bar.  Mixed runs against FP64: every
slot force is a sum of FP32 terms with a relative error of about 50 roundings
(3e-6) each; terms of both signs cancel by about a factor of 30, so forces
hold to 1e-4 of the largest one, energies (summed without such cancellation)
to 1e-5 of the sum of |E_i|.
"""
import numpy as np
import pytest

import gapx
import oracle
from gapx import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if gapx.device_count() == 0:
        pytest.skip("no GPU visible")


def grid_sf(n_eta, zetas, rc=6.0, rad_cuts=(6.0,), n_rad=7):
    t, a, c, z = synth.sf_table(n_rad, synth.logspace(0.005, 0.4, n_eta), zetas, rc)
    c = c.copy()
    c[:n_rad] = np.resize(rad_cuts, n_rad)
    return t, a, c, z


def ring_sf():
    """No grid: angular lines of several cutoffs and shifted radial lines."""
    rows = [(1, 0.05, 6.0, 1), (3, 2.0, 5.0, 1), (1, 1.0, 4.0, 1), (2, 0.02, 6.0, 1), (4, 0.02, 4.5, 2),
            (2, 0.3, 3.5, 4), (4, 0.1, 6.0, 1)]
    t, a, c, z = (np.array(x) for x in zip(*rows))
    return t.astype(np.int32), a.astype(float), c.astype(float), z.astype(float)


FORMS = {
    "eta1_zeta1": grid_sf(1, (1,)),
    "eta3_zeta5": grid_sf(3, (1, 2, 4, 8, 16)),
    "eta4_zeta4": grid_sf(4, (1, 2, 4, 16)),
    "eta5_zeta2": grid_sf(5, (1, 2)),
    "eta8_zeta3": grid_sf(8, (1, 2, 4)),
    "eta9_zeta2": grid_sf(9, (2, 4)),
    "eta4_two_radial_cutoffs": grid_sf(4, (1, 2, 4, 8), rad_cuts=(6.0, 4.5)),
    "radial_only_wide": grid_sf(1, (1,), n_rad=37),
    "radial_whole_chunk": grid_sf(2, (1, 4), n_rad=16),
    "no_grid": ring_sf(),
}


def model_for(sf, s, rng):
    t, a, c, z = sf
    D = 2 * len(t)
    om = oracle.Model(z=np.array([1, 8, 22], np.int32), w=np.array([1.0, -0.5, 2.0]), sf_type=t, sf_alpha=a, sf_cut=c,
                      theta=np.ones(D), mm=np.zeros((8, D)), coeff=rng.normal(0, 0.3, 8),
                      sf_zeta=None if np.all(z == 1) else z)
    x = oracle.descriptors(om, s["species"], s["lat"], s["pos"], 6.0)
    om.theta = 2.0 * x.std(axis=0) + 1e-3
    om.mm = x[rng.choice(len(x), size=8, replace=len(x) < 8)] + rng.normal(0, 0.2, size=(8, D)) * om.theta
    return om


# neighbours per atom about 30, 64 +- a few, 75, 130
@pytest.mark.parametrize("vpa", [30.0, 14.1, 12.0, 7.0])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_forms(form, vpa):
    rng = np.random.default_rng(int(vpa * 10))
    s = synth.structure(23, 23 * vpa, (1, 8, 22), rng, min_dist=1.3)
    om = model_for(FORMS[form], s, rng)
    ref = oracle.gap_calc(om, s["species"], s["lat"], s["pos"], 6.0, mode="sparse", nthreads=4)
    m = gapx.Model.from_model(om)
    print(form, vpa, flush=True)
    for w in (1, 2, 4):
        ctx = gapx.Context(m)
        ctx.load([s], 6.0)
        ctx.set_tuning(gapx.GRAD, waves_fwd=w, waves_bwd=w)
        ctx.set_tuning(gapx.GRAD | gapx.MIXED, waves_fwd=w, waves_bwd=w)
        ctx.run(gapx.GRAD)
        r = ctx.results()
        assert abs(r["energy"][0] - ref["energy"]) / 23 < 1e-9
        assert np.abs(r["forces"] - ref["forces"]).max() < 1e-7
        assert np.abs(r["stress"][0] - ref["stress"]).max() < max(1e-6, 1e-8 * np.abs(ref["stress"]).max())
        ctx.run(gapx.GRAD | gapx.MIXED)
        x = ctx.results()
        assert np.abs(x["forces"] - r["forces"]).max() < 1e-4 * np.abs(r["forces"]).max()
        assert abs(x["energy"][0] - r["energy"][0]) < 1e-5 * np.abs(r["eatom"]).sum()


def test_default_shapes_by_size(monkeypatch):
    """Loads without given shapes take them from the batch's size: small
    batches four to eight waves per atom and as many splits as there are
    chunks, larger ones fewer.  Every size gives what one wave per atom and
    one split give (FP64 sums in another order: 1e-12 of the largest value)."""
    rng = np.random.default_rng(9)
    first = synth.structure(8, 8 * 14.0, (1, 8, 22), rng)
    m = gapx.Model.from_model(model_for(FORMS["eta4_zeta4"], first, rng))
    seen = set()
    for n in (2, 8, 65, 257, 321, 385, 641, 769, 1537, 3100):
        s = synth.jittered_structures(1, n, n, 1.0 / 14.0, (1, 8, 22), n)[0]
        ctx = gapx.Context(m)
        ctx.load([s], 6.0)
        t = ctx.tuning(gapx.GRAD)
        seen.add((t["waves_fwd"], t["waves_bwd"]))
        print(n, t, flush=True)
        ctx.run(gapx.GRAD)
        a = ctx.results()
        ctx.set_tuning(gapx.GRAD, waves_fwd=1, waves_bwd=1, gpr_rows=64, gpr_blocks=1, halves=0)
        ctx.run(gapx.GRAD)
        b = ctx.results()
        for k in ("energy", "forces", "stress", "eatom"):
            assert np.abs(a[k] - b[k]).max() <= 1e-12 * max(1.0, np.abs(b[k]).max()), (n, k)
        ctx.load([s], 6.0)  # given shapes stay across loads
        assert ctx.tuning(gapx.GRAD)["gpr_blocks"] == 1
    assert {w for w, _ in seen} == {1, 2, 4} and {w for _, w in seen} == {1, 2, 4}
