"""Energy-only runs contract through a kernel of their own (no feature-major
halves, no second product) with the same chunk turns as the one with gradients:
compared with it and with FP64 over row tiles of 64 and 128, FP16 and BF16
operands, up to and above 128 features, and splits of 1, 2, 3 and more chunks.

With and without gradient the products, exponentials and sums are the same
operations in the same order; 2^-22 of sum |c_k| leaves each weight one FP32
rounding of another instruction choice.  Against FP64: S = xt . mt from hi + lo
halves is off by 3 * 2^-(2 b + 1) sum_d |xt_d mt_kd| with b = 11 (FP16) or 8 (BF16)
significant bits, and by 2^-24 of it per FP32 addition of D; the features' FP32
sums (relative 2^-22 each) move d2 / 2 by at most 2^-22 sum_d |x_d / theta_d|
|xt_d - mt_kd|.  E_i moves by at most sum |c_k| times those.
"""
import numpy as np
import pytest

import gapx
import oracle
from gapx import synth
from test_gpu_descriptor_forms import grid_sf

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if gapx.device_count() == 0:
        pytest.skip("no GPU visible")


# 45 lines (D = 90, padded to 96, 64 points per chunk pair) and 65 (130, 160, 32)
TABLES = {"D96": grid_sf(4, (1, 2, 4, 16), n_rad=13), "D160": grid_sf(8, (1, 2, 4), n_rad=17)}
POINTS = 250  # 256 padded


def case(table):
    rng = np.random.default_rng(17)
    s = synth.jittered_structures(1, 150, 150, 1.0 / 14.0, (1, 8, 22), 3)[0]
    t, a, c, z = TABLES[table]
    D = 2 * len(t)
    om = oracle.Model(z=np.array([1, 8, 22], np.int32), w=np.array([1.0, -0.5, 2.0]), sf_type=t, sf_alpha=a, sf_cut=c,
                      theta=np.ones(D), mm=np.zeros((POINTS, D)), coeff=rng.normal(0, 0.3, POINTS), sf_zeta=z)
    x = oracle.descriptors(om, s["species"], s["lat"], s["pos"], 6.0)
    om.theta = 12.0 * x.std(axis=0) + 1e-3
    om.mm = x[rng.choice(len(x), size=POINTS)] + rng.normal(0, 0.03, size=(POINTS, D)) * om.theta
    return s, om


@pytest.mark.parametrize("bf16", [False, True], ids=["fp16", "bf16"])
@pytest.mark.parametrize("table", sorted(TABLES))
def test_energies_with_and_without_gradient(table, bf16):
    s, om = case(table)
    m = gapx.Model.from_model(om)
    assert not m.precision()["mixed_contraction_fp64"]
    ctx = gapx.Context(m)
    ctx.load([s], 6.0)
    ctx.run(0)
    exact = ctx.results()["eatom"]
    x = ctx.features(dedx=False)[0]
    mu = (om.mm / om.theta).mean(axis=0)
    xt, mt = x / om.theta - mu, om.mm / om.theta - mu
    size = (np.abs(xt) @ np.abs(mt).T).max()
    drift = 2.0 ** -22 * max((np.abs(x[i] / om.theta) * np.abs(xt[i] - mt)).sum(axis=1).max() for i in range(len(x)))
    c1 = np.abs(om.coeff).sum()
    bar = c1 * (size * (3 * 2.0 ** -(17 if bf16 else 23) + x.shape[1] * 2.0 ** -24) + drift + 2.0 ** -22)
    assert bar < 0.05 * np.abs(exact).max(), "the bound says nothing"
    mixed = gapx.MIXED | (gapx.BF16 if bf16 else 0)
    dp = (x.shape[1] + 31) // 32 * 32
    for rows in ((64, 128) if dp <= 128 else (128,)):
        tiles = 256 // rows
        for splits in (8, 4, 3, 2, 1):
            out = []
            for flags in (mixed, mixed | gapx.GRAD):
                ctx.set_tuning(flags, gpr_rows=rows, gpr_blocks=tiles * splits, halves=0)
                ctx.run(flags)
                out.append(ctx.results())
            a, b = out
            print(table, bf16, rows, splits, np.abs(a["eatom"] - b["eatom"]).max(), np.abs(a["eatom"] - exact).max(), bar,
                  flush=True)
            assert np.abs(a["eatom"] - b["eatom"]).max() <= 2.0 ** -22 * c1
            assert np.abs(a["eatom"] - exact).max() <= bar
            assert abs(a["energy"][0] - a["eatom"].sum()) <= 1e-12 * np.abs(a["eatom"]).sum()
            assert not a["forces"].any() and not a["stress"].any()
