"""CAR2ACSF from a caller's neighbour table: independent of the evaluations the
model made before, and of table entries far beyond every cutoff.  Lines centred
far beyond their cutoff likewise, in every call."""
import numpy as np
import pytest

import gapx
import oracle
from gapx import synth
from test_gpu_descriptor_forms import FORMS, model_for

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if gapx.device_count() == 0:
        pytest.skip("no GPU visible")


def table(s, w, rcut=6.0):
    """NEIGHBOR(na, max_neighbor, 6) of a structure and its counts."""
    t = np.stack(np.meshgrid(*[np.arange(-3, 4)] * 3, indexing="ij"), -1).reshape(-1, 3) @ s["lat"]
    rows = []
    for i, p in enumerate(s["pos"]):
        q = (s["pos"][:, None] + t).reshape(-1, 3)
        j = np.repeat(np.arange(len(s["pos"])), len(t))
        d = np.linalg.norm(q - p, axis=1)
        near = (d <= rcut) & (d > 1e-9)
        rows.append(np.column_stack([q, d, w[s["species"][j]], j + 1.0])[near])
    nb = np.zeros((len(rows), max(map(len, rows)) + 2, 6))
    for i, r in enumerate(rows):
        nb[i, :len(r)] = r
    return nb, np.array([len(r) for r in rows], np.int32)


WEIGHT = np.zeros(120)
WEIGHT[[1, 8, 22]] = 1.0, -0.5, 2.0


def case(form):
    s = synth.structure(9, 9 * 14.0, (1, 8, 22), np.random.default_rng(3), min_dist=1.3)
    return s, gapx.Model.from_model(model_for(FORMS[form], s, np.random.default_rng(4)))


@pytest.mark.parametrize("form", ["eta3_zeta5", "no_grid"])
def test_same_bits_after_any_evaluation(form):
    s, m = case(form)
    nb, count = table(s, WEIGHT)
    ref = m.car2acsf(s["pos"], nb, count)
    for copies in (1, 60, 150, 700):
        m.calc_batch([s] * copies)
        out = m.car2acsf(s["pos"], nb, count)
        print(form, copies, flush=True)
        for a, b in zip(out, ref):
            assert np.array_equal(a, b), copies


# entries beyond every cutoff count nothing (a line's term needs r <= rc); the
# sums in another order: 1e-12 of the largest value
@pytest.mark.parametrize("far", [7.5, 1e9, 1e30, 1e200, np.inf])
@pytest.mark.parametrize("form", ["eta3_zeta5", "eta4_two_radial_cutoffs", "no_grid"])
def test_entries_beyond_the_cutoffs(form, far):
    s, m = case(form)
    nb, count = table(s, WEIGHT)
    ref = m.car2acsf(s["pos"], nb, count)
    for ahead in (False, True):  # behind each atom's row at a unit vector's place, before it at their own
        wide = nb.copy()
        for i, c in enumerate(count):
            entry = np.r_[s["pos"][i] + [far if ahead else 1.0, 0, 0], far, 1.0, 1.0]
            wide[i, :c + 1] = np.vstack([entry, nb[i, :c]] if ahead else [nb[i, :c], entry])
        out = m.car2acsf(s["pos"], wide, count + 1)
        print(form, far, ahead, flush=True)
        for a, b in zip(out, ref):
            assert np.isfinite(a).all()
            assert np.abs(a - b).max() <= 1e-12 * max(1.0, np.abs(b).max())


# a radial line centred there has no term; FP64 against the oracle at the parity
# bar, mixed against FP64 (1e-5 of the sum of |E_i|, 1e-4 of the largest force)
@pytest.mark.parametrize("rs", [1e9, 1e30, 1e200])
@pytest.mark.parametrize("form", ["eta3_zeta5", "no_grid"])
def test_lines_centred_beyond_their_cutoff(form, rs):
    t, a, c, z = FORMS[form]
    sf = (np.r_[t, 3].astype(np.int32), np.r_[a, rs], np.r_[c, 6.0], np.r_[z, 1.0])
    s = synth.structure(9, 9 * 14.0, (1, 8, 22), np.random.default_rng(3), min_dist=1.3)
    om = model_for(sf, s, np.random.default_rng(4))
    ref = oracle.gap_calc(om, s["species"], s["lat"], s["pos"], 6.0, mode="sparse", nthreads=4)
    m = gapx.Model.from_model(om)
    ctx = gapx.Context(m)
    ctx.load([s], 6.0)
    ctx.run(gapx.GRAD)
    r = ctx.results()
    assert abs(r["energy"][0] - ref["energy"]) / 9 < 1e-9
    assert np.abs(r["forces"] - ref["forces"]).max() < 1e-7
    ctx.run(gapx.GRAD | gapx.MIXED)
    x = ctx.results()
    assert abs(x["energy"][0] - r["energy"][0]) < 1e-5 * np.abs(r["eatom"]).sum()
    assert np.abs(x["forces"] - r["forces"]).max() < 1e-4 * np.abs(r["forces"]).max()
