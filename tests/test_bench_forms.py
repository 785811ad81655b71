"""bench.py names the backward's form by the table's etas, and the committed
counter summary has the kernels that the benchmark's workloads launch (CPU
only: no kernel runs)."""
import os
import sys

import numpy as np
import pytest

from conftest import ROOT

sys.path.insert(0, ROOT)
import bench  # noqa: E402
from gapx import synth  # noqa: E402


@pytest.mark.parametrize("n_eta,mixed,form", [(1, True, 24), (2, True, 24), (3, True, 4), (4, True, 4),
                                              (1, False, 4), (5, True, 14), (8, True, 14), (9, True, 24),
                                              (4, False, 4), (5, False, 24), (8, False, 24)])
def test_backward_form_follows_the_etas(n_eta, mixed, form):
    t = {"waves_bwd": 2}
    assert bench.stage_kernel("descriptors_bwd", mixed, t, True, 128, 1000, 4000, n_eta=n_eta) == \
        ("k_desc_bwd<%s, 2, %d, true, false>" % ("float" if mixed else "double", form), 1000 * 128)


def test_etas_of_a_table():
    t, a, c, z = synth.sf_table(5, synth.logspace(0.005, 0.4, 8), (1, 2, 4, 16), 6.0)
    assert bench.angular_etas(dict(sf_type=np.asarray(t), sf_alpha=np.asarray(a))) == 8


@pytest.mark.parametrize("label,n_atoms,des_len,nsparse,n_eta", [("ternary32k", 32768, 256, 8000, 8),
                                                                 ("ternary4k", 4096, 128, 4000, 4)])
def test_profiled_kernels_are_found(label, n_atoms, des_len, nsparse, n_eta):
    for stage in ("descriptors_fwd", "descriptors_bwd"):
        found = []
        for w in (1, 2, 4):
            t = {"waves_fwd": w, "waves_bwd": w}
            name, grid = bench.stage_kernel(stage, True, t, True, des_len, n_atoms, nsparse, n_eta=n_eta)
            found.append(bench.measured_traffic(label, name, grid) is not None)
        assert any(found), stage
