"""The two tile sizes of the variance's quadratic form: a batch whose tiles
fill the chip (128 x 128, here with a half tile left over in both directions)
against the same structures a few at a time (64 x 64).  Both sum the same
products in the same order, the features come from one wave per atom in both:
sigma^2 agrees to 1e-13 (FP64, values in [0, 1]); against the oracle 1e-10."""
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


# atoms per structure, structures, sparse points: 155 x 5 and 156 x 5 row and
# column tiles of 64 (odd numbers of both, or of columns), 256 x 4 (whole tiles)
@pytest.mark.parametrize("n,count,M", [(100, 99, 300), (67, 149, 310), (128, 128, 256)])
def test_tiles_agree(n, count, M):
    structs = synth.jittered_structures(count, n, n, 1.0 / 20.0, (1, 8, 22), 5)
    rng = np.random.default_rng(M)
    om = model_for(FORMS["eta1_zeta1"], structs[0], rng)
    x = np.concatenate([oracle.descriptors(om, s["species"], s["lat"], s["pos"], 6.0) for s in structs[:6]])
    pick = rng.choice(len(x), size=M)
    om.mm = x[pick] + rng.normal(0, 0.2, size=(M, x.shape[1])) * om.theta
    om.coeff = rng.normal(0, 0.3, M)
    Q = np.linalg.inv(oracle.covariance(om, om.mm) + 0.05 * np.eye(M))
    m = gapx.Model.from_model(om)
    m.set_qmm(Q)

    def run(part):
        ctx = gapx.Context(m)
        ctx.load(part, 6.0)
        ctx.set_tuning(gapx.GRAD, waves_fwd=1, waves_bwd=1)
        ctx.run(gapx.GRAD)
        return ctx.variance()[1]

    whole = run(structs)
    parts = np.concatenate([run(structs[k:k + 6]) for k in range(0, count, 6)])
    print(len(whole), M, np.abs(whole - parts).max(), flush=True)
    assert len(whole) == n * count
    assert np.abs(whole - parts).max() <= 1e-13
    _, ref = oracle.gpr_variance(om, x, Q)
    assert np.abs(whole[:len(x)] - ref).max() <= 1e-10
