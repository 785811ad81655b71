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
