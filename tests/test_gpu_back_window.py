"""Backprojector through per-wave LDS windows: the sums equal the oracle's bit
for bit where tiles, windows and value ranges end.

The kernel adds A and 1 with fused multiply-adds and keeps the calibration in
a sentinel value; both are exact, so the tolerance is 0 (NaN equals NaN).
"""
import numpy as np
import pytest

from gfirst_amd.geometry import Geometry

pytestmark = pytest.mark.gpu

# res, nzs, nrad, nang, span, nseg, pitch, diam, fov
GEOMS = {
    "one-tile": Geometry(8, 3, 9, 4, 1, 3, 2.0, 13.0, 8.0),        # fewest planes, span 1
    "tile+1": Geometry(9, 17, 11, 6, 3, 5, 2.0, 15.0, 9.0),        # one column into a second tile
    "tile-1": Geometry(23, 16, 20, 5, 3, 3, 2.0, 37.0, 23.0),      # planes a power of two
    "steep": Geometry(16, 65, 17, 6, 3, 15, 2.0, 20.0, 16.0),      # tilt 2 planes a voxel: fits
    "steeper": Geometry(16, 65, 17, 6, 3, 23, 2.0, 20.0, 16.0),    # 3.2 planes a voxel: gathers
    "16-rows": Geometry(24, 33, 25, 4, 3, 9, 2.0, 28.0, 24.0),     # windows of 16 rows and more
    "wide-in": Geometry(20, 12, 40, 6, 3, 3, 1.54, 33.0, 20.0),    # 1.30 bins a voxel: fits
    "wide-out": Geometry(20, 12, 40, 6, 3, 3, 1.50, 33.0, 20.0),   # 1.33 bins a voxel: gathers
}
SHAPES = [None, (4, True, 1), (5, True, 1), (6, True, 1), (8, True, 1), (16, True, 1),
          (1, False, 2), (1, False, 4), (2, False, 1), (6, False, 1)]


def run(gctx, orc, g, S, s, corr, valid):
    ne, de = orc.back(g, corr, np.where(valid, 1, -1000).astype(np.float32), s, S)
    for shape in SHAPES:
        if shape is not None:
            gctx.set_tuning(g, S, shape[0], 8, back_lds=shape[1], back_ahead=shape[2])
        n, d = gctx.back_project(g, corr, valid.astype(np.uint8), s, S)
        assert np.array_equal(n, ne, equal_nan=True), ("numer", shape)
        assert np.array_equal(d, de, equal_nan=True), ("denom", shape)


@pytest.mark.parametrize("name", list(GEOMS))
def test_edges_vs_oracle(gctx, orc, name):
    g = GEOMS[name]
    rng = np.random.default_rng(len(name))
    corr = rng.uniform(0, 3, g.ndata).astype(np.float32)
    corr[rng.uniform(size=g.ndata) < 0.03] = -1000.0
    corr[rng.uniform(size=g.ndata) < 0.03] = 0.0
    corr[rng.uniform(size=g.ndata) < 0.03] *= -0.01
    valid = rng.uniform(size=g.ndata) < 0.9
    for S, s in ((1, 0), (2, 1)):
        run(gctx, orc, g, S, s, corr, valid)


@pytest.mark.parametrize("kind", ["tiny", "huge", "nan", "inf", "sentinel", "all-invalid"])
def test_values_out_of_range_vs_oracle(gctx, orc, kind):
    """Ratios for which the fused sums are not exact take the reference's
    expression; so does a ratio equal to the sentinel itself."""
    g = GEOMS["tile+1"]
    rng = np.random.default_rng(7)
    corr = rng.uniform(0, 2, g.ndata).astype(np.float32)
    valid = rng.uniform(size=g.ndata) < 0.95
    at = rng.uniform(size=g.ndata) < 0.01
    special = {"tiny": [-1e-30, 1e-38, -1e-42], "huge": [3e37, -3e37, 1e20], "nan": [np.nan],
               "inf": [np.inf, -np.inf], "sentinel": [float.fromhex("-0x1.5a5a5ap126")],
               "all-invalid": [1.0]}[kind]
    corr[at] = rng.choice(np.asarray(special, np.float32), int(at.sum()))
    if kind == "all-invalid":
        valid[:] = False
    run(gctx, orc, g, 1, 0, corr, valid)
    # the next call on ordinary values is not affected
    run(gctx, orc, g, 1, 0, np.ones(g.ndata, np.float32), np.ones(g.ndata, bool))


def test_near_unit_calibration_vs_oracle(gctx, orc):
    """Isolated invalid bins: samples that weigh one by less than 1/1001 still
    count, with a calibration below 1."""
    g = Geometry(64, 24, 64, 16, 3, 7, 2.0, 106.1, 64.0)
    rng = np.random.default_rng(11)
    corr = rng.uniform(0, 2, g.ndata).astype(np.float32)
    valid = np.ones(g.ndata, bool)
    valid[::17] = False
    _, d = orc.back(g, corr, np.where(valid, 1, -1000).astype(np.float32), 0, 1)
    assert (d != np.round(d)).any()  # the case occurs
    run(gctx, orc, g, 1, 0, corr, valid)
