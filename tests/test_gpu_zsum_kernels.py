"""The z-sum kernel that a tuning names is the one that runs: narrow waves and
waves of 4, 6 and 8 planes, each equal to the oracle bit for bit at the edges of
its tiles, in passes of one angle and in a session whose last chunk is one angle."""
import numpy as np
import pytest

import gfirst_amd as ga
from gfirst_amd.geometry import Geometry

pytestmark = pytest.mark.gpu

# res, nzs, nrad, nang, span, nseg, pitch, diam, fov
GEOMS = {
    "3-bins": Geometry(8, 5, 3, 3, 1, 3, 2.0, 13.0, 8.0),          # fewer bins than a lane takes
    "17-angles": Geometry(20, 13, 30, 17, 3, 5, 2.0, 27.0, 20.0),  # 16 angles and 1, 2 bins over
    "leaves": Geometry(16, 33, 19, 6, 3, 11, 2.0, 17.0, 16.0),     # most LORs leave at the ends
    "2350-blocks": Geometry(20, 65, 33, 45, 3, 21, 2.0, 28.0, 20.0),
}
KERNELS = (2, 4, 6, 8)


def data(g):
    rng = np.random.default_rng(g.nang)
    y = rng.poisson(2.0, g.ndata).astype(np.float32)
    bg = rng.uniform(0, 1, g.ndata).astype(np.float32)
    return rng.uniform(0, 2, g.nvox).astype(np.float32), y, bg


@pytest.mark.parametrize("name", list(GEOMS))
def test_operators_vs_oracle(gctx, orc, name):
    g = GEOMS[name]
    img, y, bg = data(g)
    for S, s in ((1, 0), (g.nang, g.nang - 1), (2, 1)):
        proj = orc.forward(g, img, s, S)
        corr = orc.ratio(g, proj, y, bg, s, S)
        for sg in KERNELS:
            gctx.set_tuning(g, S, zsum_sg=sg)
            assert gctx.tuning(g, S)["zsum_sg"] == sg
            assert np.array_equal(gctx.forward_project(g, img, s, S), proj), (S, sg)
            assert np.array_equal(gctx.forward_ratio(g, img, y, bg, s, S), corr), (S, sg)


@pytest.mark.parametrize("name", ["17-angles", "2350-blocks"])
def test_session_vs_oracle(gctx, orc, name):
    """Log-likelihood relative to the sum of |terms|: 1e-12 (the device's log and a
    tree-ordered FP64 sum against a sequential host sum)."""
    g = GEOMS[name]
    _, y, bg = data(g)
    norm = np.ones(g.ndata, np.float32)
    yr, br = np.float32(g.res) * y, np.float32(g.res) * bg
    x0 = orc.cylinder(g, 1.0)
    proj = orc.forward(g, orc.blur_xy(g, x0, 1.5))
    exp = None
    for sg in KERNELS:
        gctx.set_tuning(g, 1, zsum_sg=sg)
        r = gctx.recon(g, ga.recon_params(mode=1, niter=1, nsub=1), np.concatenate([y, bg]), None,
                       norm)
        if exp is None:
            cal = orc.calib(g, r.get(ga.OUT_PROJ_BLANK), norm)
            exp, terms = orc.loglik(g, proj, yr, br, cal)
            x = orc.update(g, x0, *orc.back(g, orc.ratio(g, proj, yr, br), cal), 1.5)
        r.run()
        assert abs(r.loglik() - exp) <= 1e-12 * terms, sg
        assert np.array_equal(r.get(ga.OUT_XD), x), sg
        r.close()


def test_narrow_waves_are_refused_above_their_range(gctx):
    g = Geometry(20, 65, 33, 46, 3, 21, 2.0, 28.0, 20.0)  # 2444 blocks
    gctx.set_tuning(g, 1, zsum_sg=4)
    with pytest.raises(ga.GfrError):
        gctx.set_tuning(g, 1, zsum_sg=2)
    assert gctx.tuning(g, 1)["zsum_sg"] == 4
    gctx.set_tuning(g, 2, zsum_sg=2)  # 23 angles


@pytest.mark.parametrize("name", ["17-angles", "2350-blocks"])
def test_measured_tuning_round_trips(name):
    """What the tuner chose can be written back and reads the same."""
    g = GEOMS[name]
    _, y, _ = data(g)
    with ga.Context(0) as ctx:
        r = ctx.recon(g, ga.recon_params(mode=1, niter=1, nsub=2),
                      np.concatenate([y, np.zeros_like(y)]), None, np.ones(g.ndata, np.float32))
        r.close()
        t = ctx.tuning(g, 2)
        assert t["measured"] and t["zsum_sg"] in KERNELS
        keys = ("back_zb", "zsum_sg", "back_lds", "back_waves", "rot_z", "back_bw", "back_ahead")
        ctx.set_tuning(g, 2, **{k: t[k] for k in keys})
        assert {k: ctx.tuning(g, 2)[k] for k in keys} == {k: t[k] for k in keys}
