"""Without a measurement gfr_tuning_get reports the shapes that launches take, and
writing them back fixes those shapes."""
import numpy as np
import pytest

import gfirst_amd as ga
from gfirst_amd.geometry import C0, C1, Geometry

pytestmark = pytest.mark.gpu

# geometry, subsets -> sinograms per z-sum wave, planes per rotation block, then
# the backprojector's slices, windows, views at a time (by the launcher's rules)
EXPECTED = {
    "small": (C0, 4, (2, 4, 1, 0, 2)),        # 256 waves of 8 slices, few z-sum blocks
    "inveon": (C1, 16, (6, 16, 8, 1, 1)),     # 5120 waves
    "few-lors": (C1, 40, (4, 16, 8, 1, 1)),   # 2.2M LORs a pass, 4320 narrow blocks
    "two-angles": (C1, 80, (2, 4, 8, 1, 1)),  # 2160 narrow blocks
    "steep": (Geometry(16, 65, 17, 6, 3, 19, 2.0, 20.0, 16.0), 1, (2, 4, 1, 0, 1)),  # gathers
    "576-waves": (Geometry(64, 72, 64, 32, 3, 5, 2.0, 106.1, 64.0), 4, (2, 4, 1, 0, 4)),
}


@pytest.mark.parametrize("name", list(EXPECTED))
def test_reported_shapes_are_in_force(name):
    g, S, expected = EXPECTED[name]
    keys = ("zsum_sg", "rot_z", "back_zb", "back_lds", "back_ahead")
    with ga.Context(0) as ctx:
        t = ctx.tuning(g, S)
        assert not t["measured"]
        assert tuple(t[k] for k in keys) == expected
        corr = np.random.default_rng(1).uniform(0, 2, g.ndata).astype(np.float32)
        valid = np.ones(g.ndata, np.uint8)
        n, d = ctx.back_project(g, corr, valid, 0, S)
        ctx.set_tuning(g, S, **{k: t[k] for k in keys})
        t2 = ctx.tuning(g, S)
        assert t2["measured"] and tuple(t2[k] for k in keys) == expected
        n2, d2 = ctx.back_project(g, corr, valid, 0, S)
        assert np.array_equal(n, n2) and np.array_equal(d, d2)
