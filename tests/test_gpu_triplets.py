"""Neighbour and triplet lists at the sizes where their kernels change form:
one, two and four chunks of 64 neighbours held in registers, pairs from LDS
above 256, triplet entries of 16 bits (capacity up to 256) and of 32, bins with
no atoms beside full ones, more images than lanes.  FP64 against the CPU
oracle at the parity bar (the lists do not depend on the precision)."""
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


def cell(n, vpa, seed):
    return synth.jittered_structures(1, n, n, 1.0 / vpa, (1, 8, 22), seed, jitter=0.1)[0]


def skinny(seed):
    """Two atoms in a cell of 2.2 x 2.6 x 30 A: hundreds of images, most bins empty."""
    rng = np.random.default_rng(seed)
    lat = np.array([[2.2, 0, 0], [0.4, 2.6, 0], [1.0, -2.0, 30.0]])
    return dict(species=np.array([1, 22], np.int32), lat=lat, pos=np.array([[0.1, 0.2, 0.3], [1.0, 1.5, 4.0]])
                + rng.uniform(0, 0.1, (2, 3)))


def isolated():
    """No neighbours for one atom, one for the others."""
    lat = np.eye(3) * 40.0
    return dict(species=np.array([1, 8, 22], np.int32), lat=lat, pos=np.array([[1.0, 1, 1], [20, 20, 20], [21.2, 20, 20]]))


CASES = {
    "k62": cell(8, 15.2, 1), "k66": cell(27, 14.0, 2), "k128": cell(8, 7.1, 3), "k134": cell(8, 6.8, 4),
    "k190": cell(8, 4.8, 5), "k240": cell(8, 3.7, 5), "k256": cell(8, 3.4, 6), "k298": cell(8, 3.0, 7),
    "skinny": skinny(8), "isolated": isolated(),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_lists(name):
    s = CASES[name]
    n = len(s["species"])
    rng = np.random.default_rng(len(name))
    om = model_for(FORMS["eta1_zeta1"], s, rng)
    ref = oracle.gap_calc(om, s["species"], s["lat"], s["pos"], 6.0, mode="sparse", nthreads=4)
    m = gapx.Model.from_model(om)
    ctx = gapx.Context(m)
    ctx.load([s], 6.0)
    ctx.run(gapx.GRAD)
    r = ctx.results()
    print(name, ctx.counts(), flush=True)
    assert abs(r["energy"][0] - ref["energy"]) / n < 1e-9
    scale = max(1.0, np.abs(ref["forces"]).max())
    assert np.abs(r["forces"] - ref["forces"]).max() < 1e-7 * scale
    assert np.abs(r["stress"][0] - ref["stress"]).max() < max(1e-6, 1e-8 * np.abs(ref["stress"]).max())


# one, four and eight waves per atom by the batch's size: the list is the one a
# single wave builds (k66's cell of 27 atoms, alone and repeated past the lines
# at 768 and 1536 atoms; same features, so the same sums in FP64)
@pytest.mark.parametrize("name", ["k66", "k190", "isolated", "skinny"])
def test_waves_by_size(name):
    s = CASES[name]
    n = len(s["species"])
    m = gapx.Model.from_model(model_for(FORMS["eta1_zeta1"], s, np.random.default_rng(2)))
    out = []
    for copies in (1, 800 // n + 1, 1600 // n + 1):
        ctx = gapx.Context(m)
        ctx.load([s] * copies, 6.0)
        ctx.set_tuning(gapx.GRAD, waves_fwd=1, waves_bwd=1, gpr_rows=64, gpr_blocks=1, halves=0)
        ctx.run(gapx.GRAD)
        r = ctx.results()
        pairs, triplets = ctx.counts()
        out.append((pairs // copies, triplets // copies, r["energy"][0], r["forces"][:n], r["eatom"][:n],
                    ctx.features(dedx=False)[0][:n]))
        assert pairs % copies == 0 and triplets % copies == 0
        print(name, copies, out[-1][:3], flush=True)
    for o in out[1:]:
        assert o[:2] == out[0][:2]
        assert np.array_equal(o[5], out[0][5])  # lists in the same order: the same sums
        for a, b in zip(o[2:5], out[0][2:5]):
            assert np.abs(a - b).max() <= 1e-12 * max(1.0, np.abs(b).max())


@pytest.mark.parametrize("copies", [1, 400])
def test_lists_near_the_limit(copies):
    """Close to the longest list FP32 descriptors take (2912), eight and one
    waves per atom; pair counts exactly."""
    s = cell(4, 905.0 / 2850.0, 11)
    frac = s["pos"] @ np.linalg.inv(s["lat"])
    h = np.linalg.inv(s["lat"]).T  # rows: reciprocal vectors
    reach = [int(np.ceil(6.0 * np.linalg.norm(h[k]))) + 1 for k in range(3)]
    t = np.stack(np.meshgrid(*[np.arange(-r, r + 1) for r in reach], indexing="ij"), -1).reshape(-1, 3)
    d = np.linalg.norm(((frac[None, :, None] - frac[None, None]) + t[:, None, None]) @ s["lat"], axis=-1)
    want = int(((d <= 6.0) & (d > 1e-9)).sum())
    assert np.abs(d - 6.0).min() > 1e-9
    ty, a, c, z = FORMS["eta1_zeta1"]
    D = 2 * len(ty)
    om = oracle.Model(z=np.array([1, 8, 22], np.int32), w=np.array([1.0, -0.5, 2.0]), sf_type=ty, sf_alpha=a,
                      sf_cut=np.where(ty == 1, c, 1.0), theta=np.ones(D) * 1e4, mm=np.zeros((8, D)),
                      coeff=np.ones(8))
    m = gapx.Model.from_model(om)
    ctx = gapx.Context(m)
    ctx.load([s] * copies, 6.0)
    ctx.run(gapx.MIXED)
    r = ctx.results()
    print(copies, want, ctx.counts(), flush=True)
    assert ctx.counts()[0] == want * copies
    assert np.isfinite(r["energy"]).all()
