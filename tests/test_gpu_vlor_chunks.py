"""Soft assignment by chunks of an angle's bins: equal to the oracle bit for bit
(same operations in record order, tolerance 0) where chunks, angles, subsets
and lists end."""
import numpy as np
import pytest

from gfirst_amd.geometry import Geometry

pytestmark = pytest.mark.gpu

# bins of an angle: 99 (less than a chunk of 1024), 1024 (one chunk), 1025 * 3
GEOMS = {"short": Geometry(8, 5, 9, 7, 1, 3, 2.0, 13.0, 8.0),
         "whole": Geometry(8, 16, 64, 5, 3, 1, 2.0, 70.0, 8.0),
         "more": Geometry(8, 25, 123, 4, 3, 1, 2.0, 130.0, 8.0)}


@pytest.mark.parametrize("name", list(GEOMS))
@pytest.mark.parametrize("kind", ["none", "few", "many", "ends", "one-bin"])
def test_chunk_edges_vs_oracle(gctx, orc, name, kind):
    g = GEOMS[name]
    nd = g.ndata
    rng = np.random.default_rng(len(name + kind))
    rec = rng.integers(-2, nd + 3, size={"none": 0, "few": 40}.get(kind, 6000) * 2)
    if kind == "ends":  # first and last bins of angles and of the sinogram
        q = np.arange(nd)[(np.arange(nd) % g.nrad == 0) | (np.arange(nd) % g.nrad == g.nrad - 1)]
        rec = rng.choice(q + 1, size=8000)
    rec = rec.reshape(-1, 2).astype(np.int32)
    if kind == "one-bin":
        rec[:, 0] = nd // 2
        rec[::7, 1] = nd // 2
    yT = (rng.poisson(1.0, nd) * g.res).astype(np.float32)
    proj = rng.uniform(0, 2, nd).astype(np.float32)
    proj[::5] = 0.0
    bt = orc.vlor_blankt(g, yT, orc.vlor_precount(g, rec))
    v = gctx.vlor(g, rec, yT)
    for s, S in ((0, 1), (1, 2), (g.nang - 1, g.nang)):
        assert np.array_equal(v.assign(proj, s, S), orc.vlor_assign(g, rec, bt, proj, s, S)), (s, S)
    v.close()
