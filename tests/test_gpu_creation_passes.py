"""Creation passes over whole sinograms: 4 bins an item at any length and
alignment, from host or device memory, give the bits of the definition."""
import numpy as np
import pytest

import gfirst_amd as ga
from gfirst_amd.geometry import Geometry

pytestmark = pytest.mark.gpu

ODD = Geometry(8, 5, 9, 7, 1, 3, 2.0, 13.0, 8.0)  # 693 bins: halves of a pair at odd offsets


def test_mask_at_its_threshold(gctx, orc):
    g = ODD
    t = np.float32(0.01)
    vals = np.asarray([t, np.nextafter(t, np.float32(1)), np.nextafter(t, np.float32(0)), 0, -1,
                       1, np.nan, np.inf], np.float32)
    rng = np.random.default_rng(3)
    pb, nm = (rng.choice(vals, g.ndata).astype(np.float32) for _ in range(2))
    with np.errstate(invalid="ignore"):
        expect = (pb.astype(np.float64) > 0.01) & (nm.astype(np.float64) > 0.01)
    assert np.array_equal(gctx.calib_mask(g, pb, nm).astype(bool), expect)


@pytest.mark.parametrize("storage", [ga.STORE_F32, ga.STORE_F16, ga.STORE_BF16])
def test_device_pair_equals_host_pair(gctx, storage):
    g = ODD
    rng = np.random.default_rng(4)
    d2 = rng.poisson(3.0, 2 * g.ndata).astype(np.float32)
    norm = rng.uniform(0.5, 1.5, g.ndata).astype(np.float32)
    p = ga.recon_params(mode=1, niter=2, nsub=3, storage=storage)

    def image(pair, nrm):
        r = gctx.recon(g, p, pair, None, nrm)
        r.run()
        out = r.get(ga.OUT_XD)
        r.close()
        return out

    assert np.array_equal(image(d2, norm), image(gctx.to_device(d2), gctx.to_device(norm)))
    for at in (0, g.ndata - 1, 2 * g.ndata - 1):  # first, last bin of the counts, of the background
        wrong = d2.copy()
        wrong[at] = np.nan
        for pair in (wrong, gctx.to_device(wrong)):
            with pytest.raises(ga.GfrError):
                image(pair, norm)
