"""Log-likelihood of sessions and batches whose subsets differ by an angle, on
both sides of the size where passes change from narrow z-sum waves to wide ones:
equal to the oracle's per pass, and a batch's to a session's.

Relative to the sum of |terms|: 1e-12 (the device's log and a tree-ordered FP64
sum against a sequential host sum), as for even subsets."""
import numpy as np
import pytest

import gfirst_amd as ga
from gfirst_amd.geometry import Geometry

pytestmark = pytest.mark.gpu

S = 2
# 745 sinograms of 33 bins, 94 narrow blocks for every two angles
ANGLES = {"narrow": 89,   # 45 and 44 angles: 2350 blocks of narrow waves
          "limit": 91}    # 46 and 45 angles: 2444 (wide waves) and 2350


def study(nang):
    g = Geometry(20, 65, 33, nang, 3, 21, 2.0, 28.0, 20.0)
    rng = np.random.default_rng(nang)
    y = rng.poisson(rng.uniform(0.1, 4.0, g.ndata)).astype(np.float32)
    bg = rng.uniform(0, 0.3, g.ndata).astype(np.float32)
    norm = rng.uniform(0.8, 1.2, g.ndata).astype(np.float32)
    norm[rng.uniform(size=g.ndata) < 0.02] = 0.0
    return g, y, bg, norm


@pytest.mark.parametrize("tuned", [True, False], ids=["tuned", "untuned"])
@pytest.mark.parametrize("name", list(ANGLES))
def test_loglik_vs_oracle(orc, monkeypatch, name, tuned):
    if not tuned:
        monkeypatch.setenv("GFR_AUTOTUNE", "0")
    g, y, bg, norm = study(ANGLES[name])
    with ga.Context(0) as ctx:
        r = ctx.recon(g, ga.recon_params(mode=1, niter=1, nsub=S), np.concatenate([y, bg]), None,
                      norm)
        cal = orc.calib(g, r.get(ga.OUT_PROJ_BLANK), norm)
        yr, br = np.float32(g.res) * y, np.float32(g.res) * bg
        x = orc.cylinder(g, 1.0)
        for s in range(S):
            r.step()
            proj = orc.forward(g, orc.blur_xy(g, x, 1.5), s, S)
            exp, terms = orc.loglik(g, proj, yr, br, cal, s, S)
            assert abs(r.loglik() - exp) <= 1e-12 * terms, s
            x = orc.update(g, x, *orc.back(g, orc.ratio(g, proj, yr, br, s, S), cal, s, S), 1.5)
        assert np.array_equal(r.get(ga.OUT_XD), x)
        r.close()


@pytest.mark.parametrize("name", list(ANGLES))
def test_batch_of_more_subsets_than_its_lanes(name):
    """Frames of 2, 3 and 5 subsets on lanes made for 2."""
    g, y, bg, norm = study(ANGLES[name])
    with ga.Context(0) as ctx:
        bt = ctx.batch(g, ga.batch_params(max_frames=3, min_nsub=S, lanes=2), norm)
        ids = [(n, bt.add(1, n, y, bg)) for n in (2, 3, 5)]
        bt.run()
        for n, f in ids:
            r = ctx.recon(g, ga.recon_params(mode=1, niter=1, nsub=n), np.concatenate([y, bg]),
                          None, norm)
            r.run()
            assert bt.loglik(f) == r.loglik(), n
            assert np.array_equal(bt.get(f), r.get(ga.OUT_XD)), n
            r.close()
        bt.close()
