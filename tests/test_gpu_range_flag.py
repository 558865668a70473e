"""A ratio outside the range of the fast backprojection's sums sends its own pass
through the reference's expression, and no later pass: neither of the session,
nor of another frame of the batch. Timed: that expression takes several times as
long as the fast sums, a pass without such a ratio takes as long as in a run that
never had one (half as much again is allowed for)."""
import time

import numpy as np
import pytest

import gfirst_amd as ga
from gfirst_amd.geometry import C1

pytestmark = pytest.mark.gpu

S = 16


@pytest.fixture(scope="module")
def study():
    """Counts, and the same with one tiny negative one in subset 0, whose ratio
    lies between -2^-32 and 0."""
    g = C1
    y = np.random.default_rng(3).poisson(0.5, g.ndata).astype(np.float32)
    odd = y.copy()
    odd[(g.nsinogs // 2 * g.nang) * g.nrad + g.nrad // 2] = -1e-15
    return g, y, odd, np.ones(g.ndata, np.float32)


def test_sessions(gctx, study):
    g, y, odd, norm = study
    ms = {}
    for name, v in (("clean", y), ("odd", odd)):
        r = gctx.recon(g, ga.recon_params(mode=1, niter=1, nsub=S),
                       np.concatenate([v, np.zeros_like(v)]), None, norm)
        r.profile(True)
        passes = []
        for _ in range(8):
            r.step()
            passes.append(r.phase_times()["back"][0])
        r.close()
        ms[name] = passes
        print(name, ["%.3f" % t for t in passes])
    assert ms["odd"][0] > 2 * ms["clean"][0]  # the case occurs
    assert np.median(ms["odd"][1:]) < 1.5 * np.median(ms["clean"][1:])


def test_frames_of_a_batch(gctx, study):
    g, y, odd, norm = study
    ms = {}
    for name, v in (("clean", y), ("odd", odd)):
        bt = gctx.batch(g, ga.batch_params(max_frames=2, min_nsub=S, lanes=1), norm)
        for f in (v, y):
            bt.add(1, S, f)
        steps = []
        for _ in range(8):
            t = time.perf_counter()
            bt.step()
            bt.sync()
            steps.append(1e3 * (time.perf_counter() - t))
        bt.close()
        ms[name] = steps
        print(name, ["%.3f" % t for t in steps])
    assert np.median(ms["odd"][1:]) < 1.5 * np.median(ms["clean"][1:])
