"""Triplet entries of 16 bits up to the widest list that has them (capacity 256,
248 neighbours once a run has grown to it), and the change to 32 bits and back
between the runs of one context, eager and replayed from a graph.  Clusters in a
wide cell: their first capacity is 32, so every list here is one that grew.

FP64 against the CPU oracle at the parity bar, forces scaled by the largest."""
import numpy as np
import pytest

import gapx
import oracle
from test_gpu_descriptor_forms import FORMS

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if gapx.device_count() == 0:
        pytest.skip("no GPU visible")


def cluster(n, scale=1.0):
    """n points of a jittered cubic lattice nearest to its centre, within 3 A at scale 1."""
    g = np.stack(np.meshgrid(*[np.arange(-5, 6)] * 3, indexing="ij"), -1).reshape(-1, 3) * 1.0
    g = g[np.argsort((g ** 2).sum(1), kind="stable")[:n]]
    rng = np.random.default_rng(n)
    g = g + rng.uniform(-0.15, 0.15, g.shape)
    g *= 2.95 / np.linalg.norm(g, axis=1).max()
    return dict(species=rng.choice(np.array([1, 8, 22], np.int32), n).astype(np.int32), lat=np.eye(3) * 60.0,
                pos=30.0 + scale * g)


def model(structures):
    """Centres and length scales from all of the structures."""
    rng = np.random.default_rng(1)
    t, a, c, z = FORMS["eta1_zeta1"]
    D = 2 * len(t)
    om = oracle.Model(z=np.array([1, 8, 22], np.int32), w=np.array([1.0, -0.5, 2.0]), sf_type=t, sf_alpha=a, sf_cut=c,
                      theta=np.ones(D), mm=np.zeros((12, D)), coeff=rng.normal(0, 0.3, 12))
    x = np.concatenate([oracle.descriptors(om, s["species"], s["lat"], s["pos"], 6.0) for s in structures])
    om.theta = 2.0 * x.std(axis=0) + 1e-3
    om.mm = x[rng.choice(len(x), size=12)] + rng.normal(0, 0.2, size=(12, D)) * om.theta
    return om


def check(om, s, pos, r, ctx):
    ref = oracle.gap_calc(om, s["species"], s["lat"], pos, 6.0, mode="sparse", nthreads=8)
    n = len(pos)
    d = np.linalg.norm(pos[:, None] - pos[None], axis=-1)
    assert ctx.counts()[0] == int(((d <= 6.0) & (d > 0)).sum())
    assert abs(r["energy"][0] - ref["energy"]) / n < 1e-9
    scale = max(1.0, np.abs(ref["forces"]).max())
    assert np.abs(r["forces"] - ref["forces"]).max() < 1e-7 * scale
    assert np.abs(r["stress"][0] - ref["stress"]).max() < max(1e-6, 1e-8 * np.abs(ref["stress"]).max())
    return int(((d <= 6.0) & (d > 0)).sum(1).max())


# 240 and 248 neighbours: capacities 248 and 256 (16 bits); 249: 264 (32 bits)
@pytest.mark.parametrize("k", [186, 200, 240, 247, 248, 249])
def test_grown_lists(k):
    s = cluster(k + 1)
    om = model([s])
    ctx = gapx.Context(gapx.Model.from_model(om))
    ctx.load([s], 6.0)
    ctx.run(gapx.GRAD)
    r = ctx.results()
    print(k, ctx.counts(), flush=True)
    assert check(om, s, s["pos"], r, ctx) == k


@pytest.mark.parametrize("graph", [False, True], ids=["eager", "graph"])
def test_growth_across_the_entry_widths(graph):
    s, loose, looser = (cluster(300, scale) for scale in (1.0, 2.5, 3.2))
    om = model([s, loose, looser])
    ctx = gapx.Context(gapx.Model.from_model(om))
    ctx.load([looser], 6.0)
    ctx.use_graph(graph)
    seen = []
    for c in (looser, loose, loose, s, s, looser, loose):  # 16 bits, grown; 32 bits; the same lists in 32 bits
        ctx.update(c["pos"])
        ctx.run(gapx.GRAD)
        seen.append(check(om, s, c["pos"], ctx.results(), ctx))
        print(graph, seen[-1], flush=True)
    assert 32 < seen[0] < seen[1] <= 248 < seen[3]
