"""Lists on both sides of every count at which the triplet builder takes another
number of 64-neighbour chunks (64, 128, 192, 256, above it from LDS), with eight,
four and one wave per atom (up to 768, 1536 and more atoms).

Clusters in a wide cell, every atom within the others' cutoff.  One cluster in
FP64 against the CPU oracle at the parity bar; batches of copies hold the same
lists in the same order, so the features agree bit for bit and the rest to 1e-12."""
import numpy as np
import pytest

import gapx
import oracle
from test_gpu_triplets_narrow import cluster, model

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if gapx.device_count() == 0:
        pytest.skip("no GPU visible")


@pytest.mark.parametrize("k", [63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257])
def test_chunks(k):
    s = cluster(k + 1)
    n = k + 1
    om = model([s])
    ref = oracle.gap_calc(om, s["species"], s["lat"], s["pos"], 6.0, mode="sparse", nthreads=8)
    m = gapx.Model.from_model(om)
    first = None
    for copies in (1, 800 // n + 1, 1600 // n + 1):
        ctx = gapx.Context(m)
        ctx.load([s] * copies, 6.0)
        ctx.set_tuning(gapx.GRAD, waves_fwd=1, waves_bwd=1, gpr_rows=64, gpr_blocks=1, halves=0)
        ctx.run(gapx.GRAD)
        r = ctx.results()
        pairs, triplets = ctx.counts()
        print(k, copies, pairs, triplets, flush=True)
        assert pairs == copies * n * k and triplets % copies == 0
        x = ctx.features(dedx=False)[0].reshape(copies, n, -1)
        if first is None:
            first = (triplets, x[0], r)
            scale = max(1.0, np.abs(ref["forces"]).max())
            assert abs(r["energy"][0] - ref["energy"]) / n < 1e-9
            assert np.abs(r["forces"] - ref["forces"]).max() < 1e-7 * scale
        assert triplets == copies * first[0]
        assert np.array_equal(x, np.broadcast_to(first[1], x.shape))
        f = r["forces"].reshape(copies, n, 3)
        assert np.abs(f - first[2]["forces"]).max() <= 1e-12 * max(1.0, np.abs(f).max())
        assert np.abs(r["energy"] - first[2]["energy"]).max() <= 1e-12 * np.abs(r["eatom"][:n]).sum()
