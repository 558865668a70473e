"""Radius-4 joint bilateral filter: its weights in pairs of floats.

On the CPU (jbf_pair_weight_check.c restates the arithmetic): the quotient
equals IEEE division, and every weight that is kept equals the reference
expression (float)exp(-(double)di2 / kI) (jointbilateralfilter3D_K,
GFIRST_GPU_Kernels.cu:508-539). Sampled here; over every float di2 at sigma_I
0.025 (1.05e9 values) no weight differed. On the GPU: the kernel equals the
oracle bit for bit where volumes, rows of lanes and value ranges end.
"""
import os
import subprocess

import numpy as np
import pytest

from gfirst_amd.geometry import Geometry

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("jbf") / "jbf_pair_weight_check")
    subprocess.run(["gcc", "-O2", "-mfma", "-ffp-contract=off", "-o", exe,
                    os.path.join(HERE, "jbf_pair_weight_check.c"), "-lm"], check=True)
    return exe


@pytest.mark.parametrize("args", [("div", 2), ("exp", 61, 0.025), ("exp", 61, 1e-3),
                                  ("exp", 61, 100.0)])
def test_kept_weights_equal_reference(checker, args):
    out = subprocess.run([checker, *map(str, args)], check=True, capture_output=True, text=True)
    cases, left, bad, worst = out.stdout.split()
    assert int(cases) > 10_000_000 and int(bad) == 0
    assert int(left) < int(cases) // 1000 and float(worst) < 1


# side, planes: smaller than the radius, one interior voxel, one block and one lane more
@pytest.mark.gpu
@pytest.mark.parametrize("res,nzs", [(4, 5), (5, 3), (5, 6), (26, 11), (27, 9), (70, 6)])
@pytest.mark.parametrize("kind", ["noise", "shell", "edges"])
def test_volume_and_value_edges_vs_oracle(gctx, orc, res, nzs, kind):
    g = Geometry(res, nzs, 9, 4, 1, 1, 2.0, 3.0 * res, 1.0 * res)
    rng = np.random.default_rng(res + nzs)
    inp = rng.uniform(0, 3, g.nvox).astype(np.float32)
    guide = rng.uniform(0.4, 0.6, g.nvox).astype(np.float32)
    if kind == "shell":  # weights around the smallest normal float, below it, and 0
        guide = rng.choice(np.asarray([0, 0.46, 0.466, 0.47, 0.5, 0.511, 0.512, 1], np.float32),
                           g.nvox)
    if kind == "edges":
        guide[rng.uniform(size=g.nvox) < 0.01] = np.inf
        guide[rng.uniform(size=g.nvox) < 0.01] = np.nan
        guide[rng.uniform(size=g.nvox) < 0.05] = -3e38
        guide[rng.uniform(size=g.nvox) < 0.05] = 1e-42
    for mref in (1.0, 0.7, 2.0 ** -21):
        with np.errstate(all="ignore"):
            exp = orc.jbf(g, inp, guide, mref)
        assert np.array_equal(gctx.jbf3d(g, inp, guide, mref), exp, equal_nan=True), mref
