"""Loading, updating and fetching through a context's pinned staging."""
import numpy as np
import pytest

import gapx
from gapx import synth
from helpers import workload_model

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pop():
    if gapx.device_count() == 0:
        pytest.skip("no GPU visible")
    return gapx.Model.from_model(workload_model("population")), synth.population(40, seed=4004)


def evaluate(m, structs, flags):
    ctx = gapx.Context(m)
    ctx.load(structs, 6.0)
    ctx.run(flags)
    r = ctx.results()
    ctx.close()
    return [r]


def test_loads_through_growing_staging(pop):
    """Batches below and above the staging's first room, single structures,
    packed lists (numpy int32/float64 arrays) and other forms (lists, float32
    or Fortran-ordered arrays), lattice and position updates without a run in
    between: every form gives bit for bit what a fresh context gives."""
    m, structs = pop
    small, large = structs[:3], synth.population(120, seed=4005)
    odd = [dict(species=[int(z) for z in s["species"]], lat=np.asfortranarray(s["lat"]), pos=s["pos"].tolist())
           for s in small]
    ctx = gapx.Context(m)
    for batch, plain in ((small, small), (large, large), (odd, small), (small[:1], small[:1]), (large, large)):
        ctx.load(batch, 6.0)
        ctx.run(gapx.GRAD)
        r = ctx.results()
        f = evaluate(m, plain, gapx.GRAD)[0]
        for k in ("energy", "forces", "stress", "eatom"):
            assert np.array_equal(r[k], f[k]), k
    pos = np.concatenate([s["pos"] for s in large])
    ctx.update(pos + 0.01)
    ctx.update(pos + 0.02, lat=np.stack([s["lat"] * 1.01 for s in large]))
    assert np.array_equal(ctx.positions(), pos + 0.02)
    ctx.run(gapx.GRAD)
    moved = [dict(species=s["species"], lat=s["lat"] * 1.01, pos=s["pos"] + 0.02) for s in large]
    f = evaluate(m, moved, gapx.GRAD)[0]
    assert np.array_equal(ctx.results()["forces"], f["forces"])
    ctx.close()
