"""The work that a user of this package has it do, as timed cases.

Every case goes through the package's public entry points (Context, Recon,
Batch, Vlor): the operators a program calls one by one in place of the
reference's wrappers, and whole reconstructions. `kind` names the entry point;
the other keys are the geometry and the call's own arguments.

Inputs are drawn on the GPU from the seed: a mouse-like phantom (a body and
six organs, ellipsoids) whose line integrals are taken in closed form, Poisson
counts of those, a normalization in [0.8, 1.2] and, where `gaps` is set, the
diagonal stripes that missing detector blocks leave in a sinogram.
"""
import math

import numpy as np
import torch

import gfirst_amd as ga
from gfirst_amd.geometry import Geometry, nseg_for

_GEOM = ("res", "nzs", "nrad", "nang", "span", "nseg", "pitch", "diam_det", "fov")


def _geometry_keys(g):
    return {k: getattr(g, k) for k in _GEOM}


def _geometry(case):
    return Geometry(*[case[k] for k in _GEOM])


def listed():
    small, inveon, ref = (_geometry_keys(g) for g in (ga.C0, ga.C1, ga.REF))
    return [
        # Projection-only run of a small study: every view of one image.
        dict(small, name="project-small", kind="project", subset=0, nsub=1),
        # The same for the scanner as the reference compiles it (span 11, 147 bins,
        # 168 angles): a whole sinogram in one call, the projector's largest.
        dict(ref, name="project-ref", kind="project", subset=0, nsub=1),
        # One subset's projection and ratio with a randoms background, span 3.
        dict(inveon, name="ratio-inveon", kind="ratio", subset=5, nsub=16),
        # Backprojection of one subset of a small study: the smallest call.
        dict(small, name="back-small", kind="back", subset=1, nsub=4, gaps=False),
        # Backprojection with an odd bin count and detector gaps in the data.
        dict(ref, name="back-ref", kind="back", subset=3, nsub=12, gaps=True),
        # The heaviest operator of an Inveon-size subset.
        dict(inveon, name="back-inveon", kind="back", subset=2, nsub=16, gaps=False),
        # Joint bilateral filter of a triples estimate, guided by the doubles image.
        dict(inveon, name="jbf-inveon", kind="jbf"),
        # Soft assignment of one subset's triple events to their bins.
        dict(inveon, name="vlor-inveon", kind="vlor", subset=7, nsub=16, nrec=860000),
        # Whole small reconstruction from host arrays (2 iterations x 4 subsets),
        # as a program that replaces the executable calls it.
        dict(small, name="osem-small", kind="osem", nsub=4, niter=2, storage=0, host=True, bg=True),
        # One iteration (16 subsets) of an Inveon-size study whose sinograms are on
        # the GPU in half precision, session and result copy included.
        dict(inveon, name="osem-inveon", kind="osem", nsub=16, niter=1, storage=1, host=False,
             bg=False),
        # One joint doubles + triples iteration with the VLOR assignment.
        dict(inveon, name="joint-inveon", kind="joint", nsub=16, niter=1, nrec=860000),
        # Six frames of a dynamic study with uneven subset counts, advanced together.
        dict(inveon, name="batch-inveon", kind="batch", niter=1, frames=6, storage=1),
    ]


def draw(rng):
    """A scanner between the small study's and the Inveon-size one, odd sizes
    included, and one of the calls above on it."""

    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    res = log(48, 128)
    rings = log(16, 80)
    span = rng.choice([3, 3, 5, 7, 9, 11])
    pitch = rng.choice([1.63, 2.0])
    fov = res * rng.uniform(0.75, 1.0)
    nzs = 2 * rings - 1
    nseg = nseg_for(span, rng.randint(rings // 2, rings - 1))
    while nseg > 1 and nzs - 2 * ((nseg // 2 - 1) * span + span // 2 + 1) <= 0:
        nseg -= 2
    g = dict(res=res, nzs=nzs, nrad=min(147, max(32, int(res * rng.uniform(0.85, 1.15)))),
             nang=log(48, 168), span=span, nseg=max(1, nseg), pitch=pitch,
             diam_det=round(fov * rng.uniform(1.6, 1.9), 3), fov=round(fov, 3))
    kind = rng.choice(["project", "ratio", "back", "back", "jbf", "vlor", "osem", "osem", "joint",
                       "batch"])
    nsub = rng.choice([4, 6, 8, 12, 16, 24])
    one = dict(subset=rng.randrange(nsub), nsub=nsub)
    more = {
        "project": lambda: rng.choice([dict(subset=0, nsub=1), one]),
        "ratio": lambda: one,
        "back": lambda: dict(one, gaps=rng.random() < 0.5),
        "jbf": lambda: {},
        "vlor": lambda: dict(one, nrec=log(20000, 860000)),
        "osem": lambda: dict(nsub=nsub, niter=1, storage=rng.choice([0, 1, 2]), host=False,
                             bg=rng.random() < 0.5),
        "joint": lambda: dict(nsub=rng.choice([8, 12, 16]), niter=1, nrec=log(20000, 860000)),
        "batch": lambda: dict(niter=1, frames=rng.randint(2, 6), storage=rng.choice([0, 1, 2])),
    }[kind]()
    return dict(g, kind=kind, **more)


# --- inputs ------------------------------------------------------------------

_contexts = {}


def _context(which):
    """One library context per way of working: a program that calls operators
    holds one, a program that runs sessions holds one."""
    if which not in _contexts:
        _contexts[which] = ga.Context(0)
    return _contexts[which]


class _DeviceView:
    """Lets torch see a DeviceArray's memory, and keeps it alive."""

    def __init__(self, arr):
        self.arr = arr
        self.__cuda_array_interface__ = dict(shape=(arr.n,), typestr=arr.dtype.str,
                                             data=(arr.ptr, False), version=2)


def _tensor(arr):
    return torch.as_tensor(_DeviceView(arr), device="cuda")


def _to_library(ctx, t, dtype=np.float32):
    arr = ctx.array(t.numel(), dtype)
    _tensor(arr).copy_(t.reshape(-1))
    return arr


def _zeros(ctx, n):
    arr = ctx.array(n)
    _tensor(arr).zero_()
    return arr


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


class _Views:
    """Sinogram coordinates: per sinogram its plane and axial step, per angle
    sine and cosine, in double precision on the GPU."""

    def __init__(self, g):
        self.zmin, self.sign, self.first = [], [], []
        planes, steps, acc = [], [], 0
        pi = float(np.float32(3.1415926))
        for k in range(g.nseg):
            i = (k + 1) // 2
            zm = 0 if i == 0 else (i - 1) * g.span + g.span // 2 + 1
            sg = 0 if i == 0 else (1 if k % 2 == 0 else -1)
            n = g.nzs - 2 * zm
            self.zmin.append(zm)
            self.sign.append(sg)
            self.first.append(acc)
            planes.append(np.arange(zm, g.nzs - zm))
            steps.append(np.full(n, (g.fov / g.res) * sg * zm / (0.5 * g.diam_det)))
            acc += n
        self.nsino = acc
        dev = dict(device="cuda", dtype=torch.float64)
        self.plane = torch.tensor(np.concatenate(planes), **dev)
        self.step = torch.tensor(np.concatenate(steps), **dev)
        ang = -np.arange(g.nang) / g.nang * pi + pi
        self.sin, self.cos = torch.tensor(np.sin(ang), **dev), torch.tensor(np.cos(ang), **dev)
        self.bins = torch.arange(g.nrad, **dev) - (g.nrad - 1) / 2.0


def _phantom(g, gen):
    """Body and organs: (centre, semi axes, added value) in voxels, z last."""
    vx, vz = g.fov / g.res, g.pitch / 2.0
    u = torch.rand(6, 8, generator=gen, device="cuda").cpu().numpy().astype(np.float64)
    mid = np.array([(g.res - 1) / 2.0] * 2 + [(g.nzs - 1) / 2.0])
    rad = min(12.5 / vx, 0.42 * g.res)
    zhalf = min(45.0 / vz, 0.5 * g.nzs)
    out = [(mid, np.array([rad, rad, zhalf]), 1.0)]
    for a in u:
        semi = np.array([rad * (0.16 + 0.24 * a[0]), rad * (0.16 + 0.24 * a[1]),
                         zhalf * (0.08 + 0.2 * a[2])])
        r = a[3] * (rad - semi[:2].max())
        c = mid + np.array([r * math.cos(6.2832 * a[4]), r * math.sin(6.2832 * a[4]),
                            (2 * a[5] - 1) * (zhalf - semi[2])])
        out.append((c, semi, 0.5 + 7.0 * a[6]))
    return out


def _image(g, ellipsoids):
    z, y, x = (torch.arange(n, device="cuda", dtype=torch.float64) for n in (g.nzs, g.res, g.res))
    img = torch.zeros(g.nzs, g.res, g.res, device="cuda")
    for c, s, v in ellipsoids:
        d = (((z - c[2]) / s[2]) ** 2)[:, None, None] + (((y - c[1]) / s[1]) ** 2)[None, :, None] + \
            (((x - c[0]) / s[0]) ** 2)[None, None, :]
        img += v * (d <= 1.0)
    return img


def _integrals(g, ellipsoids):
    """Line integrals of the phantom (in samples of one voxel's length) for
    every bin, closed form: [sinogram][angle][bin]."""
    V = _Views(g)
    mid, fx = (g.res - 1) / 2.0, (0.5 * g.pitch) / (g.fov / g.res)
    f = torch.float32
    st, ct = V.sin.to(f)[None, :, None], V.cos.to(f)[None, :, None]
    x0 = (fx * V.bins).to(f)[None, None, :]
    out = torch.zeros(V.nsino, g.nang, g.nrad, device="cuda")
    rows = max(1, 16_000_000 // (g.nang * g.nrad))
    for a in range(0, V.nsino, rows):
        p = V.plane[a:a + rows].to(f)[:, None, None]
        dz = V.step[a:a + rows].to(f)[:, None, None]
        for c, s, v in ellipsoids:
            ox, oy = (x0 * ct + (mid - c[0])) / s[0], (x0 * st + (mid - c[1])) / s[1]
            dx, dy = st / s[0], -ct / s[1]
            oz, ez = (p - c[2]) / s[2], dz / s[2]
            qa = (dx * dx + dy * dy) + ez * ez
            qb = (ox * dx + oy * dy) + oz * ez
            qc = (ox * ox + oy * oy) + (oz * oz - 1.0)
            out[a:a + rows] += (2.0 * v) * torch.sqrt(torch.clamp(qb * qb - qa * qc, min=0.0)) / qa
    return out


def _support(g):
    """The image's cylinder (radius RES/2), as an ellipsoid without ends."""
    c = np.array([g.res // 2, g.res // 2, 0.0], np.float64)
    return [(c, np.array([g.res / 2.0, g.res / 2.0, 1e6]), 1.0)]


def _normalization(g, gen, gaps):
    """[angle][bin] factors per sinogram in [0.8, 1.2]; with gaps, 0 on the
    diagonals that two missing detector blocks leave."""
    V = _Views(g)
    n = 0.8 + 0.4 * torch.rand(V.nsino, g.nang, g.nrad, device="cuda", generator=gen)
    if gaps:
        a = torch.arange(g.nang, device="cuda")[:, None]
        r = torch.arange(g.nrad, device="cuda")[None, :]
        k = (r * g.nang) // g.nrad
        n *= ~(((k + a) % (g.nang // 2) < 2) | ((k - a) % (g.nang // 2) < 2))
    return n


def _counts(mean, total, gen):
    return torch.poisson(mean * (total / mean.sum(dtype=torch.float64)).to(torch.float32),
                         generator=gen)


def _records(weights, n, gen):
    """n pairs of 1-based bins drawn from the sinogram's distribution; one in
    twenty names a hit outside the scanner (0)."""
    edge = torch.cumsum(weights.reshape(-1).double(), 0)
    at = torch.rand(2 * n, device="cuda", generator=gen, dtype=torch.float64) * edge[-1]
    i = torch.searchsorted(edge, at).clamp_(max=edge.numel() - 1) + 1
    i *= torch.rand(2 * n, device="cuda", generator=gen) >= 0.05
    return i.to(torch.int32).reshape(n, 2)


def _total_counts(views):
    """5e7 counts over an Inveon-size sinogram, in proportion elsewhere."""
    return 0.57 * views.numel()


def _inputs(case, seed):
    """What the call is given, as GPU tensors."""
    g, gen, kind = _geometry(case), _generator(seed), case["kind"]
    body = _phantom(g, gen)
    if kind == "project":
        return dict(img=_image(g, body))
    if kind == "jbf":
        guide, img = _image(g, body), _image(g, _phantom(g, gen))
        noise = torch.rand(2, *guide.shape, device="cuda", generator=gen)
        return dict(guide=guide * (0.7 + 0.6 * noise[0]), img=img * (0.4 + 1.2 * noise[1]))
    mean = _integrals(g, body)
    if kind == "batch":
        return dict(norm=_normalization(g, gen, False),
                    y=[_counts(mean, _total_counts(mean) * 0.2 * (1 + k), gen)
                       for k in range(case["frames"])])
    if kind == "osem":
        bg = 0.05 * float(mean.mean()) if case["bg"] else 0.0
        y = _counts(mean + bg, _total_counts(mean), gen)
        back = torch.full_like(y, float(y.mean()) * bg / float(mean.mean() + bg))
        return dict(y=torch.stack([y, back]), norm=_normalization(g, gen, False))
    other = _integrals(g, _phantom(g, gen)) if kind in ("joint", "vlor") else None
    if kind == "joint":
        zero = torch.zeros_like(mean)
        return dict(y=torch.stack([_counts(mean, _total_counts(mean), gen), zero]),
                    t=torch.stack([_counts(other, 0.02 * _total_counts(mean), gen), zero]),
                    rec=_records(other, case["nrec"], gen), norm=_normalization(g, gen, False))
    # Mid-reconstruction estimate: the phantom over a faint remainder of the
    # uniform start.
    blank = _integrals(g, _support(g))
    est = mean + 0.02 * blank
    if kind == "vlor":
        return dict(proj=other + 0.02 * blank, rec=_records(other, case["nrec"], gen),
                    y=g.res * _counts(other, 0.02 * _total_counts(mean), gen))
    if kind == "ratio":
        scale = g.res * _total_counts(mean) / float(mean.sum(dtype=torch.float64))
        bg = 0.05 * float(mean.mean()) * scale
        y = g.res * _counts(mean + 0.05 * float(mean.mean()), _total_counts(mean), gen)
        return dict(img=_image(g, body) * scale, y=y, bg=torch.full_like(y, bg))
    # back: measured over estimated counts, -1000 where nothing is expected
    c = _total_counts(mean) / float(est.sum(dtype=torch.float64))
    y = torch.poisson(est * c, generator=gen)
    corr = torch.where(est >= 0.01, y / (est * c).clamp(min=1e-12), -1000.0)
    mask = (blank > 0.01) & (_normalization(g, gen, case["gaps"]) > 0.01)
    return dict(corr=corr, mask=mask.to(torch.uint8))


def prepare(case, seed):
    g, kind, d = _geometry(case), case["kind"], _inputs(case, seed)
    s = dict(case=case, g=g)
    if kind in ("osem", "joint", "batch"):
        ctx = s["ctx"] = _context("sessions")
        if kind == "batch":
            s["subsets"] = [(8, 16, 24)[k % 3] for k in range(case["frames"])]
            s["y"] = [_to_library(ctx, y) for y in d["y"]]
            s["batch"] = ctx.batch(g, ga.batch_params(storage=case["storage"],
                                                      max_frames=case["frames"], min_nsub=8),
                                   d["norm"].cpu().numpy())
        elif kind == "osem" and case["host"]:
            s["y"], s["norm"] = (d[k].cpu().numpy() for k in ("y", "norm"))
        else:
            s["y"], s["norm"] = _to_library(ctx, d["y"]), _to_library(ctx, d["norm"])
            if kind == "joint":
                s["t"], s["rec"] = _to_library(ctx, d["t"]), d["rec"].cpu().numpy()
        s["params"] = None if kind == "batch" else ga.recon_params(
            mode=3 if kind == "joint" else 1, niter=case["niter"], nsub=case["nsub"],
            storage=case.get("storage", ga.STORE_F32))
    else:
        ctx = s["ctx"] = _context("operators")
        if kind == "vlor":
            y = _to_library(ctx, d["y"])
            torch.cuda.synchronize()
            s["vlor"] = ctx.vlor(g, d["rec"].cpu().numpy(), y)
            s["in"] = [_to_library(ctx, d["proj"])]
        elif kind == "back":
            s["in"] = [_to_library(ctx, d["corr"]), _to_library(ctx, d["mask"], np.uint8)]
        else:
            s["in"] = [_to_library(ctx, d[k]) for k in ("img", "guide", "y", "bg") if k in d]
        voxels = kind in ("back", "jbf")
        s["out"] = [_zeros(ctx, g.nvox if voxels else g.ndata) for _ in range(2 if kind == "back" else 1)]
        s["result"] = [_tensor(o) for o in s["out"]]
        if kind == "jbf":
            s["max"] = ctx.image_max(g, s["in"][1])
    torch.cuda.synchronize()
    return s


def run(s):
    case, ctx, g = s["case"], s["ctx"], s["g"]
    kind = case["kind"]
    if kind == "batch":
        b = s["batch"]
        ids = [b.add(case["niter"], n, y) for n, y in zip(s["subsets"], s["y"])]
        b.run()
        out = [b.get(f) for f in ids]
        for f in ids:
            b.remove(f)
        return out
    if kind == "osem" and case["host"]:
        return ctx.osem_run(g, s["params"], s["y"], None, s["norm"])[0]
    if kind in ("osem", "joint"):
        r = ctx.recon(g, s["params"], s["y"], s.get("t"), s["norm"], s.get("rec"))
        r.run()
        out = [r.get(w) for w in ((ga.OUT_XD, ga.OUT_XT) if kind == "joint" else (ga.OUT_XD,))]
        r.close()
        return out
    if kind == "project":
        ctx.forward_project(g, s["in"][0], case["subset"], case["nsub"], out=s["out"][0])
    elif kind == "ratio":
        ctx.forward_ratio(g, *s["in"], case["subset"], case["nsub"], out=s["out"][0])
    elif kind == "back":
        ctx.back_project(g, *s["in"], case["subset"], case["nsub"], *s["out"])
    elif kind == "vlor":
        s["vlor"].assign(s["in"][0], case["subset"], case["nsub"], out=s["out"][0])
    else:
        ctx.jbf3d(g, s["in"][0], s["in"][1], s["max"], out=s["out"][0])
    return s["result"]


# --- what a pass cannot do without -------------------------------------------


def _angles(g, subset, nsub):
    return (g.nang - subset + nsub - 1) // nsub


def work(case):
    """Bytes: inputs once, outputs once. Operations: 9 per bilinear and 4 per
    axial interpolation of a projection's samples, 10 per voxel and view of a
    backprojection (only planes inside the segment), 10 per neighbour of the
    bilateral filter."""
    g, kind = _geometry(case), case["kind"]
    zmins = [0 if k == 0 else ((k + 1) // 2 - 1) * g.span + g.span // 2 + 1 for k in range(g.nseg)]
    planes = sum(g.nzs - 2 * z for z in zmins)

    def forward(na):
        return na * (g.res + 1) * g.nrad * (4.0 * planes + 9.0 * g.nzs)

    def back(na):
        return 10.0 * na * g.res * g.res * planes

    jbf = 10.0 * 729 * max(0, g.nzs - 4) * max(0, g.res - 4) ** 2
    lors = planes * g.nrad  # per angle
    if kind == "jbf":
        return dict(bytes=12.0 * g.nvox, flops=jbf)
    if kind in ("project", "ratio", "back", "vlor"):
        na = _angles(g, case["subset"], case["nsub"])
        if kind == "vlor":  # the touched bins' projections, the records, the subset's bins
            return dict(bytes=16.0 * case["nrec"] + 4.0 * lors * na, flops=8.0 * case["nrec"])
        if kind == "back":
            return dict(bytes=5.0 * lors * na + 8.0 * g.nvox, flops=back(na))
        return dict(bytes=4.0 * g.nvox + (12.0 if kind == "ratio" else 4.0) * lors * na,
                    flops=forward(na))
    one = case["niter"] * (forward(g.nang) + back(g.nang))
    if kind == "batch":
        n = case["frames"]
        return dict(bytes=n * (4.0 * lors * g.nang + 4.0 * g.nvox), flops=n * one)
    if kind == "joint":
        return dict(bytes=20.0 * lors * g.nang + 8.0 * g.nvox + 8.0 * case["nrec"],
                    flops=2 * one + case["niter"] * case["nsub"] * jbf)
    return dict(bytes=12.0 * lors * g.nang + 4.0 * g.nvox, flops=one)


# --- the same computations in double precision -------------------------------


def _lerp(a, b, t):
    return a + t * (b - a)


def _axis(c, n):
    """Clamp-to-edge linear filter: lower and upper sample and the weight."""
    f = torch.floor(c)
    i = f.long()
    return i.clamp(0, n - 1), (i + 1).clamp(0, n - 1), c - f


def _project64(g, V, img, angles):
    """[sinogram][angle][bin] sums of RES + 1 trilinear samples."""
    mid, fx = (g.res - 1) / 2.0, (0.5 * g.pitch) / (g.fov / g.res)
    lo, hi = math.floor(-0.5 * g.res), math.floor(0.5 * g.res)
    ell = torch.arange(lo, hi + 1, device="cuda", dtype=torch.float64)
    z0, z1, az = _axis(V.plane[None, :] + ell[:, None] * V.step[None, :], g.nzs)
    az = az[:, :, None]
    out = torch.empty(V.nsino, len(angles), g.nrad, device="cuda", dtype=torch.float64)
    flat = img.reshape(g.nzs, -1)
    for k, it in enumerate(angles):
        st, ct = V.sin[it], V.cos[it]
        x0, x1, ax = _axis(fx * V.bins[None, :] * ct + mid + ell[:, None] * st, g.res)
        y0, y1, ay = _axis(fx * V.bins[None, :] * st + mid - ell[:, None] * ct, g.res)
        plane = _lerp(_lerp(flat[:, y0 * g.res + x0], flat[:, y0 * g.res + x1], ax),
                      _lerp(flat[:, y1 * g.res + x0], flat[:, y1 * g.res + x1], ax), ay)
        acc = torch.zeros(V.nsino, g.nrad, device="cuda", dtype=torch.float64)
        for i in range(len(ell)):
            p = plane[:, i]
            acc += _lerp(p[z0[i]], p[z1[i]], az[i])
        out[:, k] = acc
    return out


def _back64(g, V, corr, valid, angles):
    """Sums over views of the interpolated ratio and calibration."""
    mid, fx = (g.res - 1) / 2.0, (g.fov / g.res) / (g.pitch / 2.0)
    xy = torch.arange(g.res, device="cuda", dtype=torch.float64) - mid
    z = torch.arange(g.nzs, device="cuda", dtype=torch.float64)[:, None]
    both = torch.stack([corr, torch.where(valid, 1.0, -1000.0).double()])
    num = torch.zeros(g.nzs, g.res * g.res, device="cuda", dtype=torch.float64)
    den = torch.zeros_like(num)
    for s in range(g.nseg):
        zm = V.zmin[s]
        fz = (g.fov / g.res) * V.sign[s] * zm / (0.5 * g.diam_det)
        n = g.nzs - 2 * zm
        for k, it in enumerate(angles):
            st, ct = V.sin[it], V.cos[it]
            u = ((xy[:, None] * st + xy[None, :] * ct) * fx + (g.nrad - 1) / 2.0).reshape(-1)
            yr = (xy[:, None] * ct - xy[None, :] * st).reshape(1, -1)
            t = z + yr * fz
            inside = (t + 0.5 >= zm) & (t + 0.5 < g.nzs - zm)
            r0, r1, au = _axis(u, g.nrad)
            p0, p1, aw = _axis(t, g.nzs)
            rows = torch.full((2, g.nzs, g.nrad), -1000.0, device="cuda", dtype=torch.float64)
            rows[:, zm:g.nzs - zm] = both[:, V.first[s]:V.first[s] + n, k]
            c = _lerp(rows[:, :, r0], rows[:, :, r1], au)
            a, b = (_lerp(torch.gather(v, 0, p0), torch.gather(v, 0, p1), aw) for v in c)
            keep = inside & (a >= 0) & (b >= 0)
            num += torch.where(keep, a, 0.0)
            den += torch.where(keep, b, 0.0)
    return num, den


def _blur64(g, img, psf):
    k = torch.arange(-4, 5, dtype=torch.float64) * 1.662 / (psf + 0.1)
    w = torch.exp(-k * k)
    w = (w / w.sum()).cuda()
    x = img.reshape(g.nzs, 1, g.res, g.res)
    y = torch.nn.functional.pad(x, (0, 0, 4, 4))
    y = sum(w[j] * y[:, :, j:j + g.res] for j in range(9))
    out = x.clone()
    if g.res > 8:
        out[..., 4:-4] = sum(w[j] * y[..., j:j + g.res - 8] for j in range(9))
    return out.reshape(g.nzs, g.res, g.res)


def _update64(g, x, num, den, psf):
    f = _blur64(g, torch.where(den < 0.001, 1.0, num / den.clamp(min=0.001)), psf)
    w = torch.exp(-torch.arange(-2, 3, dtype=torch.float64) ** 2)
    w = (w / w.sum()).cuda()
    r2, f = g.res * g.res, f.reshape(-1)
    pad = torch.nn.functional.pad(f, (2 * r2, 2 * r2))
    m2, m1, c, p1, p2 = (pad[j * r2:j * r2 + f.numel()] for j in range(5))
    # a voxel takes the rule of the slice that the voxel before it lies in
    k = ((torch.arange(f.numel(), device="cuda") - 1).clamp(min=0)) // r2
    v = w[0] * m2 + w[1] * m1 + w[2] * c + w[3] * p1 + w[4] * p2
    v = torch.where((k == 1) | (k == g.nzs - 2), 0.333 * (m1 + c + p1), v)
    v = torch.where(k == 0, 0.5 * (c + p1), v)
    v = torch.where(k == g.nzs - 1, 0.5 * (m1 + c), v)
    x = (x.reshape(-1) * v).reshape(g.nzs, g.res, g.res)
    x[0], x[-1] = x[1], x[-2]
    return x


def _jbf64(g, img, guide, top, r=4, sigma=0.75, sigma_i=0.025):
    ks, ki = (2 * sigma) ** 2, (2 * sigma_i) ** 2
    norm, total = torch.zeros_like(img), torch.zeros_like(img)

    def cut(n, d):  # voxels whose neighbour at offset d lies below the upper face
        return slice(r, min(n, n - d)), slice(r + d, min(n, n + d))

    for dz in range(-r, r + 1):
        for dy in range(-r, r + 1):
            for dx in range(-r, r + 1):
                at, of = zip(cut(g.nzs, dz), cut(g.res, dy), cut(g.res, dx))
                h = torch.exp(-((guide[of] - guide[at]) / top) ** 2 / ki -
                              (dz * dz + dy * dy + dx * dx) / ks)
                norm[at] += h
                total[at] += h * img[of]
    return torch.where(norm > 1e-8, total / norm.clamp(min=1e-8), 0.0)


def _ratio64(p, y, bg):
    den = p + (0.0 if bg is None else bg.clamp(min=0.0))
    return torch.where(den >= 0.01, y / den.clamp(min=0.01), -1000.0)


def _osem64(case, g, V, d):
    x = torch.zeros(g.nzs, g.res, g.res, device="cuda", dtype=torch.float64)
    i = torch.arange(g.res, device="cuda") - g.res // 2
    x[:] = ((i[:, None] ** 2 + i[None, :] ** 2) <= (g.res // 2) ** 2).double()
    blank = _project64(g, V, x, list(range(g.nang))).float()
    valid = (blank > 0.01) & (d["norm"] > 0.01)
    del blank
    y, bg = d["y"]
    if case["storage"]:
        half = torch.float16 if case["storage"] == ga.STORE_F16 else torch.bfloat16
        y, bg = y.to(half), bg.to(half)
    for _ in range(case["niter"]):
        for sub in range(case["nsub"]):
            at = list(range(sub, g.nang, case["nsub"]))
            p = _project64(g, V, _blur64(g, x, 1.5), at)
            corr = _ratio64(p, g.res * y[:, at].double(), g.res * bg[:, at].double())
            x = _update64(g, x, *_back64(g, V, corr, valid[:, at], at), 1.5)
    return x


def _place(full, part, angles):
    """The subset's bins in a sinogram of zeros, flat as the library lays it out."""
    full[:, angles] = part
    return full.reshape(-1)


def exact(case, seed):
    """None for a batch and a joint study (their passes are those of `osem`,
    `vlor` and `jbf`, and many)."""
    g, kind = _geometry(case), case["kind"]
    if kind in ("batch", "joint"):
        return None
    d, V = _inputs(case, seed), _Views(g)
    if kind == "osem":
        x = _osem64(case, g, V, d).reshape(-1).cpu().numpy()
        return x if case["host"] else [x]
    if kind == "jbf":
        return [_jbf64(g, d["img"].double(), d["guide"].double(), float(d["guide"].max())).reshape(-1)]
    at = list(range(case["subset"], g.nang, case["nsub"]))
    full = torch.zeros(V.nsino, g.nang, g.nrad, device="cuda", dtype=torch.float64)
    if kind == "project":
        return [_place(full, _project64(g, V, d["img"].double(), at), at)]
    if kind == "ratio":
        p = _project64(g, V, d["img"].double(), at)
        return [_place(full, _ratio64(p, d["y"][:, at].double(), d["bg"][:, at].double()), at)]
    if kind == "back":
        n, t = _back64(g, V, d["corr"][:, at].double(), d["mask"][:, at] > 0, at)
        return [n.reshape(-1), t.reshape(-1)]
    # vlor: each event's weight, split between its two bins by their projections
    i = d["rec"].long() - 1
    i = i[((i > 0) & (i < full.numel())).all(1)]
    hits = torch.bincount(i.reshape(-1), minlength=full.numel()).double()
    share = torch.where(hits > 0, d["y"].reshape(-1).double() / (g.res * hits.clamp(min=1)), 0.0)
    pair = d["proj"].reshape(-1).double()[i]
    total = pair.sum(1)
    weight = torch.where(total > 0.01, share[i].sum(1) / total.clamp(min=0.01), 0.0)
    got = torch.zeros(full.numel(), device="cuda", dtype=torch.float64)
    got.index_add_(0, i.reshape(-1), (pair * weight[:, None]).reshape(-1))
    return [_place(full, got.reshape(V.nsino, g.nang, g.nrad)[:, at], at)]
