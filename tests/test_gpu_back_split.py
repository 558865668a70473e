"""Backprojector whose waves share a tile's views: equal to the oracle bit for
bit (the samples and the order of their sums are the oracle's, so the tolerance
is 0) where turns of 8 views, chunks of 64 views and angle tables end."""
import numpy as np
import pytest

from gfirst_amd.geometry import Geometry

pytestmark = pytest.mark.gpu


# views: 1 angle of 1 segment, less and more than a turn, a chunk, a chunk + 1,
# more angles than the table in LDS holds
@pytest.mark.parametrize("nang,nseg,S", [(3, 1, 3), (7, 1, 1), (9, 1, 1), (64, 1, 4), (13, 5, 1),
                                         (30, 7, 1), (25, 7, 1), (26, 7, 1)])
@pytest.mark.parametrize("gaps", [0.0, 0.02, 0.5])
def test_turn_edges_vs_oracle(gctx, orc, nang, nseg, S, gaps):
    g = Geometry(17, 21, 19, nang, 3, nseg, 2.0, 27.0, 17.0)
    rng = np.random.default_rng(nang + nseg)
    corr = rng.uniform(0, 3, g.ndata).astype(np.float32)
    corr[rng.uniform(size=g.ndata) < 0.05] = -1000.0
    valid = rng.uniform(size=g.ndata) >= gaps
    gctx.set_tuning(g, S, 1, 8, back_lds=False, back_ahead=2)
    for s in (0, S - 1):
        ne, de = orc.back(g, corr, np.where(valid, 1, -1000).astype(np.float32), s, S)
        n, d = gctx.back_project(g, corr, valid.astype(np.uint8), s, S)
        assert np.array_equal(n, ne) and np.array_equal(d, de), s
