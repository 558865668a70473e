"""Backprojector where one slice's window takes more than 16 rows and eight
slices' windows more than 32: equal to the oracle bit for bit (the samples and
the order of their sums are the oracle's, so the tolerance is 0), without a
tuning and with every tuned shape."""
import numpy as np
import pytest

import gfirst_amd as ga
from gfirst_amd.geometry import Geometry

pytestmark = pytest.mark.gpu

SHAPES = [None, (4, True, 1), (8, True, 1), (16, True, 1), (1, False, 2), (1, False, 4),
          (2, False, 1)]


# rows of 1 / 4 / 8 slices: 25 / 28 / 32, 28 / 31 / 35, 31 / 34 / 38; angles of 45 degrees, where a
# tile's corners are farthest apart, among the four
@pytest.mark.parametrize("nseg", [17, 19, 21])
def test_steep_tilts_vs_oracle(orc, nseg):
    g = Geometry(16, 65, 17, 4, 3, nseg, 2.0, 20.0, 16.0)
    rng = np.random.default_rng(nseg)
    corr = rng.uniform(0, 3, g.ndata).astype(np.float32)
    corr[rng.uniform(size=g.ndata) < 0.03] = -1000.0
    valid = rng.uniform(size=g.ndata) < 0.95
    ne, de = orc.back(g, corr, np.where(valid, 1, -1000).astype(np.float32), 0, 1)
    with ga.Context(0) as ctx:
        for shape in SHAPES:
            if shape is not None:
                ctx.set_tuning(g, 1, shape[0], 8, back_lds=shape[1], back_ahead=shape[2])
            n, d = ctx.back_project(g, corr, valid.astype(np.uint8), 0, 1)
            assert np.array_equal(n, ne), shape
            assert np.array_equal(d, de), shape
