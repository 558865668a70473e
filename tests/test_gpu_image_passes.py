"""Blur, update, maximum and ratio at the edges of their strips of four: equal
to the oracle bit for bit (same operations in the same order, tolerance 0)."""
import numpy as np
import pytest

from gfirst_amd.geometry import Geometry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res,nzs,nrad", [(4, 3, 5), (7, 4, 9), (8, 5, 12), (9, 3, 11),
                                          (17, 6, 18), (33, 3, 39), (64, 4, 67)])
def test_strip_edges_vs_oracle(gctx, orc, res, nzs, nrad):
    g = Geometry(res, nzs, nrad, 5, 1, 1, 2.0, 1.7 * res + 4, 1.0 * res)
    rng = np.random.default_rng(res)
    x = rng.uniform(0, 2, g.nvox).astype(np.float32)
    num = rng.uniform(0, 3, g.nvox).astype(np.float32)
    den = rng.uniform(0, 2, g.nvox).astype(np.float32)
    den[rng.uniform(size=g.nvox) < 0.2] = 0.0
    assert np.array_equal(gctx.blur_xy(g, x, 1.5), orc.blur_xy(g, x, 1.5))
    assert np.array_equal(gctx.update(g, x, num, den, 1.5), orc.update(g, x, num, den, 1.5))
    for at in (0, g.nvox - 1):
        y = x.copy()
        y[at] = 7.0
        assert gctx.image_max(g, y) == 7.0
    assert gctx.image_max(g, -x) == 0.0
    proj = rng.uniform(0, 1, g.ndata).astype(np.float32)
    proj[rng.uniform(size=g.ndata) < 0.3] = 0.0
    yT = rng.poisson(2.0, g.ndata).astype(np.float32)
    for bg in (None, rng.uniform(-0.01, 0.02, g.ndata).astype(np.float32)):
        zero = np.zeros(g.ndata, np.float32)
        assert np.array_equal(gctx.ratio(g, proj, yT, zero if bg is None else bg, 1, 2),
                              orc.ratio(g, proj, yT, zero if bg is None else bg, 1, 2))
