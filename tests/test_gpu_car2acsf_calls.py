"""CAR2ACSF from a caller's neighbour table: independent of the evaluations the
model made before."""
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
