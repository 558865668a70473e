"""Projector at the edges of its tiles, groups and waves: equal to the oracle
bit for bit (the arithmetic and its order are the oracle's, so the tolerance
is 0), for every tuned shape and for the untuned one.
"""
import numpy as np
import pytest

from gfirst_amd.geometry import Geometry

pytestmark = pytest.mark.gpu

# res, nzs, nrad, nang, span, nseg, pitch, diam, fov
GEOMS = {
    "3-bins": Geometry(8, 5, 3, 3, 1, 3, 2.0, 13.0, 8.0),        # fewer bins than a lane takes
    "17-angles": Geometry(20, 13, 30, 17, 3, 5, 2.0, 27.0, 20.0),  # a partial chunk, 2 bins over
    "leaves": Geometry(16, 33, 19, 6, 3, 11, 2.0, 17.0, 16.0),   # most LORs leave at the ends
    "below": Geometry(20, 65, 33, 48, 3, 21, 2.0, 28.0, 20.0),   # 2350 blocks of narrow waves
    "above": Geometry(20, 65, 33, 50, 3, 21, 2.0, 28.0, 20.0),   # 2444: wide waves
    "even-bins": Geometry(24, 64, 64, 64, 3, 15, 1.0, 33.0, 24.0),
}


@pytest.mark.parametrize("name", list(GEOMS))
def test_edges_vs_oracle(gctx, orc, name):
    g = GEOMS[name]
    rng = np.random.default_rng(len(name))
    img = rng.uniform(0, 2, g.nvox).astype(np.float32)
    y = rng.poisson(2.0, g.ndata).astype(np.float32)
    y[rng.uniform(size=g.ndata) < 0.1] = -1000.0  # invalid bins
    bg = rng.uniform(0, 1, g.ndata).astype(np.float32)
    for S, s in ((1, 0), (g.nang - 1, 0), (3, 2)):
        proj = orc.forward(g, img, s, S)
        corr = orc.ratio(g, proj, y, bg, s, S)
        for sg, rz in ((0, 0), (4, 4), (6, 16), (8, 32)):
            if sg:
                gctx.set_tuning(g, S, zsum_sg=sg, rot_z=rz)
            what = "subset %d of %d, %d planes, rotation %d" % (s, S, sg, rz)
            assert np.array_equal(gctx.forward_project(g, img, s, S), proj), what
            assert np.array_equal(gctx.forward_ratio(g, img, y, bg, s, S), corr), what
