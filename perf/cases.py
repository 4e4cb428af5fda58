"""Timed cases of the volumetric merging estimators, each one pass through the public Python entry points.

Every input is made on the GPU from a seed. The kinds of case:

  frame      camera rays of one frame against photon points and photon beams (upbp_eval)
  stress     random camera rays against a dense set of photon beams, half SHORT, half LONG
  rays       rays without a common origin: the continuation segments of scattered camera paths
  upbp       a frame evaluated with the UPBP MIS weights (upbp_eval_upbp)
  adjoint    a differentiable rendering step: forward, squared loss, gradients (autograd)
  batch      many small independent scenes in one persistent plan (hipGraph replay)
  iteration  one progressive iteration: trace light paths, build both structures, evaluate a frame
  pp3d       vertex merging in media through the hashed grid
  surf       vertex merging on surfaces through the hashed grid
  knn        structure builds with k-nearest-neighbour radii

`exact` evaluates the plain estimators, their gradients and the KNN radii in 64 bits by brute force.
"""
from __future__ import annotations

import math
import types

import numpy as np
import torch

from smallupbp_amd import _abi, autograd, native, scenes

DEV = "cuda"
SPHERE_C, SPHERE_R = (0.5, 0.5, 0.5), 0.3
EYE = (0.5, 0.5, -2.0)
# media tables: box 0, vacuum 1, sphere 2 (sigma_a, sigma_s, mean cosine, continuation)
CLEAR = ((0.0, 0.0, 0.0), (0.0, 0.0, 0.0), 0.0, 1.0)
BOX_SPHERE = [((0.02, 0.02, 0.02), (0.2, 0.2, 0.2), 0.0, 0.8), CLEAR, ((0.05, 0.05, 0.05), (2.0, 2.0, 2.0), 0.0, 0.8)]
CHROMATIC = [((0.02, 0.03, 0.01), (0.2, 0.25, 0.3), 0.0, 0.8), CLEAR, ((0.05, 0.04, 0.06), (2.0, 1.8, 2.2), 0.0, 0.8)]
UNIT_CUBE = [((0.1, 0.1, 0.1), (0.5, 0.5, 0.5), 0.0, 0.8), CLEAR]
DENSE_BOX = [((0.1, 0.1, 0.1), (1.0, 1.0, 1.0), 0.0, 0.8), CLEAR]
TRACE_MEDIA = [((0.05, 0.1, 0.02), (1.2, 1.0, 0.8), 0.0, 0.9), CLEAR, ((0.1, 0.05, 0.2), (3.0, 2.5, 2.0), 0.0, 0.8)]


def listed():
    return [
        # a thumbnail or preview tile: the smallest call, where launches and waits are what it costs
        {"name": "frame_64x36", "kind": "frame", "width": 64, "height": 36, "photons": 20_000, "beams": 2_000,
         "sphere": True, "short": False, "g": 0.0},
        # photon points only in one cube: the plain beam radiance estimate
        {"name": "frame_256_points", "kind": "frame", "width": 256, "height": 256, "photons": 100_000, "beams": 0,
         "sphere": False, "short": False, "g": 0.0},
        # a full-HD frame of a preview render, photon points of varying radius and SHORT photon beams
        {"name": "frame_1080p", "kind": "frame", "width": 1920, "height": 1080, "photons": 1_000_000,
         "beams": 200_000, "sphere": True, "short": False, "g": 0.0},
        # the heaviest beam gather: a million query beams against two million photon beams
        {"name": "stress_1m_2m", "kind": "stress", "queries": 1_000_000, "beams": 2_000_000},
        # continuation rays of scattered camera paths, forward-scattering media: no two share an origin
        {"name": "rays_200k", "kind": "rays", "queries": 200_003, "photons": 300_000, "beams": 60_000, "g": 0.5},
        # one UPBP camera pass of a full-HD frame
        {"name": "upbp_1080p", "kind": "upbp", "width": 1920, "height": 1080, "paths": 400_000, "beams": 200_000},
        # one optimisation step of the media coefficients and photon powers
        {"name": "adjoint_512", "kind": "adjoint", "width": 512, "height": 512, "photons": 500_000,
         "beams": 100_000},
        # many independent scenes served at once, their sizes uneven
        {"name": "batch_16", "kind": "batch", "instances": 16, "photons": 35_000, "queries": 500_000},
        # progressive rendering: everything is rebuilt each iteration
        {"name": "iteration_640x360", "kind": "iteration", "width": 640, "height": 360, "paths": 200_000,
         "beam_paths": 25_000},
        # merging a million camera vertices in media
        {"name": "pp3d_1m", "kind": "pp3d", "queries": 1_000_000, "paths": 1_000_000, "radius": 0.01},
        # merging a million camera vertices on surfaces
        {"name": "surf_1m", "kind": "surf", "queries": 1_000_000, "paths": 1_000_000, "radius": 0.01},
        # builds whose radii come from the 10th nearest neighbour
        {"name": "knn_150k", "kind": "knn", "photons": 150_000, "beams": 30_000, "knn": 10},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "stress", "rays", "upbp", "adjoint", "batch", "iteration", "pp3d",
                       "surf", "knn"])
    if kind == "frame":
        w = _log(rng, 48, 1920)
        h = max(9, int(w * rng.uniform(0.5, 0.75)) | 1)
        photons, beams = _log(rng, 5_000, 1_000_000), _log(rng, 1_000, 200_000)
        drop = rng.randrange(4)
        return {"kind": kind, "width": w, "height": min(h, 1080), "photons": 0 if drop == 1 else photons,
                "beams": 0 if drop == 2 else beams, "sphere": rng.random() < 0.6, "short": rng.random() < 0.3,
                "g": rng.choice([0.0, 0.0, 0.6, -0.3])}
    if kind == "stress":
        return {"kind": kind, "queries": _log(rng, 30_000, 900_000), "beams": _log(rng, 50_000, 1_500_000)}
    if kind == "rays":
        return {"kind": kind, "queries": _log(rng, 1_000, 200_000), "photons": _log(rng, 10_000, 300_000),
                "beams": _log(rng, 2_000, 60_000), "g": rng.choice([0.0, 0.5, 0.8])}
    if kind == "upbp":
        w = _log(rng, 100, 1600)
        return {"kind": kind, "width": w, "height": max(9, w * 9 // 16), "paths": _log(rng, 10_000, 400_000),
                "beams": _log(rng, 2_000, 200_000)}
    if kind == "adjoint":
        w = _log(rng, 64, 512)
        return {"kind": kind, "width": w, "height": max(9, int(w * rng.uniform(0.6, 1.0))),
                "photons": _log(rng, 20_000, 500_000), "beams": _log(rng, 5_000, 100_000)}
    if kind == "batch":
        return {"kind": kind, "instances": rng.randint(4, 24), "photons": _log(rng, 8_000, 40_000),
                "queries": _log(rng, 20_000, 400_000)}
    if kind == "iteration":
        w = _log(rng, 160, 800)
        return {"kind": kind, "width": w, "height": max(9, w * 9 // 16), "paths": _log(rng, 20_000, 250_000),
                "beam_paths": _log(rng, 5_000, 25_000)}
    if kind in ("pp3d", "surf"):
        return {"kind": kind, "queries": _log(rng, 30_000, 900_000), "paths": _log(rng, 60_000, 900_000),
                "radius": round(rng.uniform(0.006, 0.011), 5)}
    return {"kind": kind, "photons": _log(rng, 10_000, 150_000), "beams": _log(rng, 2_000, 30_000),
            "knn": rng.choice([3, 10, 10, 16])}


# ---- inputs, made on the GPU -------------------------------------------------------------
class _Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed) * 7919 + 17)

    def uni(self, shape, lo=0.0, hi=1.0):
        return torch.rand(shape, generator=self.g, device=DEV, dtype=torch.float64) * (hi - lo) + lo

    def normal(self, shape):
        return torch.randn(shape, generator=self.g, device=DEV, dtype=torch.float64)

    def integers(self, lo, hi, n):
        return torch.randint(lo, hi, (n,), generator=self.g, device=DEV)

    def dirs(self, n):
        z = self.uni(n, -1.0, 1.0)
        phi = self.uni(n, 0.0, 2.0 * math.pi)
        s = torch.sqrt(torch.clamp(1.0 - z * z, min=0.0))
        return _unit(torch.stack([s * torch.cos(phi), s * torch.sin(phi), z], -1))


def _unit(v):
    return (v / v.norm(dim=-1, keepdim=True)).float()


def _media(rows, g=None):
    if g is not None:
        rows = [(a, s, g if any(s) else 0.0, c) for a, s, _, c in rows]
    return scenes.make_media(rows)


def _tables(media):
    """sigma_a, sigma_s, sigma_t (f64), the smallest positive sigma_t and its channel, scattering flag, g."""
    sa = torch.tensor(np.abs(media["absorption"].astype(np.float64)), device=DEV)
    ss = torch.tensor(np.abs(media["scattering"].astype(np.float64)), device=DEV)
    st = sa + ss
    mn, k = torch.where(st > 0, st, torch.full_like(st, math.inf)).min(1)
    mn = torch.where(torch.isfinite(mn), mn, torch.zeros_like(mn))
    return sa, ss, st, mn, k, (ss > 0).any(1), torch.tensor(media["mean_cosine"].astype(np.float64), device=DEV)


def _frame_rays(width, height):
    x = (torch.arange(width, device=DEV, dtype=torch.float64) + 0.5) / width
    y = 0.5 + (torch.arange(height, device=DEV, dtype=torch.float64) + 0.5 - height * 0.5) / width
    yy, xx = torch.meshgrid(y, x, indexing="ij")
    return _camera(torch.stack([xx.reshape(-1), yy.reshape(-1), torch.zeros(width * height, device=DEV)], -1))


def _camera(target):
    e = torch.tensor(EYE, device=DEV, dtype=torch.float64)
    return e.expand_as(target).float().contiguous(), _unit(target - e)


def _sphere_span(o, d):
    oc = o.double() - torch.tensor(SPHERE_C, device=DEV, dtype=torch.float64)
    b = (d.double() * oc).sum(-1)
    disc = b * b - ((oc * oc).sum(-1) - SPHERE_R ** 2)
    s = torch.sqrt(torch.clamp(disc, min=0.0))
    return disc > 0, -b - s, -b + s


def _box_span(o, d):
    inv = 1.0 / d.double()
    a, b = -o.double() * inv, (1.0 - o.double()) * inv
    return torch.minimum(a, b).amax(-1), torch.maximum(a, b).amin(-1)


def _segments(media, o, d, sphere):
    """CSR offsets and [S,8] records (what Scene::Intersect stores) of rays through the unit box medium and the
    sphere medium in it, and the same as [Q,4] arrays (tmin, tmax, medium, valid)."""
    n = o.shape[0]
    tin, tout = _box_span(o, d)
    tin = torch.clamp(tin, min=0.0)
    hit = tout > tin
    zero = torch.zeros_like(tin)
    if sphere:
        hs, a, b = _sphere_span(o, d)
        a, b = torch.maximum(a, tin), torch.minimum(b, tout)
        hs = hs & hit & (b > a)
        a, b = torch.where(hs, a, tout), torch.where(hs, b, tout)
    else:
        hs, a, b = torch.zeros(n, dtype=torch.bool, device=DEV), tout, tout
    far = torch.full_like(tin, 10.0)
    t0 = torch.stack([zero, tin, a, b], 1)
    t1 = torch.stack([torch.where(hit, tin, far), a, b, tout], 1)
    ok = torch.stack([~hit | (tin > 0), hit & (a > tin), hs, hs & (tout > b)], 1)
    mid = torch.tensor([1, 0, 2, 0], device=DEV).expand(n, 4)
    t0, t1 = t0.float(), t1.float()
    ok = ok & (t1 > t0)
    ok[:, 0] |= ~ok.any(1)  # every ray has a segment
    mid = torch.where(ok, mid, torch.zeros_like(mid))
    counts = ok.sum(1)
    off = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    off[1:] = torch.cumsum(counts, 0)
    _, _, st, mn, _, sc, _ = _tables(media)
    m = mid[ok]
    ln = (t1 - t0)[ok].double()
    seg = torch.zeros((int(off[-1]), 8), dtype=torch.float32, device=DEV)
    seg[:, 0], seg[:, 1] = t0[ok], t1[ok]
    pdf = torch.where(sc[m], torch.clamp(torch.exp(-mn[m] * ln), min=1e-35), torch.ones_like(ln)).float()
    seg[:, 2], seg[:, 3] = pdf, pdf
    seg[:, 4:7] = torch.exp(-st[m] * ln[:, None]).float()
    seg.view(torch.int32)[:, 7] = m.to(torch.int32)
    return off, seg, (t0, t1, mid, ok)


def _photons(gen, n, lognormal=None, radius=None):
    pos = gen.uni((n, 3)).float()
    inc = gen.dirs(n)
    power = gen.uni((n, 3), 0.0, 1e-4).float()
    r = None
    if lognormal:
        r = torch.clamp(torch.exp(math.log(lognormal) + 0.4 * gen.normal(n)), 5e-4, 0.05).float()
    return scenes.Photons(pos, inc, power, r, 0.0 if radius is None else radius)


def _beams(gen, n, media, sphere, radius, short_fraction=1.0, short_mean=None):
    o = gen.uni((n, 3)).float()
    d = gen.dirs(n)
    _, bound = _box_span(o, d)
    med = torch.zeros(n, dtype=torch.int64, device=DEV)
    if sphere:
        hs, a, b = _sphere_span(o, d)
        inside = ((o.double() - torch.tensor(SPHERE_C, device=DEV, dtype=torch.float64)) ** 2).sum(-1) < SPHERE_R ** 2
        stop = torch.where(inside, b, torch.where(hs & (a > 0), a, torch.full_like(a, math.inf)))
        bound = torch.minimum(bound, stop)
        med[inside] = 2
    mn = _tables(media)[3]
    short = gen.uni(n) < short_fraction
    mean = 1.0 / mn[med] if short_mean is None else torch.full((n,), short_mean, device=DEV, dtype=torch.float64)
    length = torch.where(short, torch.minimum(-torch.log1p(-gen.uni(n)) * mean, bound), bound)
    flags = torch.where(short, scenes.SHORT_BEAM, scenes.LONG_BEAM).to(torch.int32)
    return scenes.Beams(o, d, torch.clamp(length, min=1e-4).float(), gen.uni((n, 3), 0.0, 1e-4).float(), flags,
                        med.to(torch.int32), radius)


def _frame_inputs(c, seed):
    gen = _Gen(seed)
    kind = c["kind"]
    sphere = kind in ("rays", "adjoint") or bool(c.get("sphere"))
    short = bool(c.get("short"))
    if kind == "stress":
        media = _media(DENSE_BOX)
        o, d = _camera(torch.cat([gen.uni((c["queries"], 2)), torch.zeros((c["queries"], 1), device=DEV)], 1))
        ph, bm = None, _beams(gen, c["beams"], media, False, 0.003, 0.5, 0.05)
    elif kind == "rays":
        media = _media(BOX_SPHERE, c["g"])
        o, d = gen.uni((c["queries"], 3)).float(), gen.dirs(c["queries"])
        ph = _photons(gen, c["photons"], lognormal=0.005)
        bm = _beams(gen, c["beams"], media, True, 0.003)
    else:
        media = _media(CHROMATIC if kind == "adjoint" else BOX_SPHERE if sphere else UNIT_CUBE, c.get("g"))
        o, d = _frame_rays(c["width"], c["height"])
        ph = None
        if c["photons"]:
            ph = _photons(gen, c["photons"], lognormal=0.005) if sphere else _photons(gen, c["photons"], radius=0.01)
        bm = _beams(gen, c["beams"], media, sphere, 0.003) if c["beams"] else None
    off, seg, pad = _segments(media, o, d, sphere)
    return types.SimpleNamespace(gen=gen, media=media, o=o, d=d, off=off, seg=seg, pad=pad, photons=ph, beams=bm,
                                 short=short, common=kind != "rays")


def _built(ctx, ph, bm, **kw):
    """Both structures on a context whose stream does not wait for torch's."""
    torch.cuda.synchronize()
    bre = beams = None
    if ph is not None:
        bre = native.EmbreeBre(ctx)
        bre.build(ph, **kw)
    if bm is not None:
        beams = native.PhotonBeamsEvaluator(ctx)
        beams.build(bm)
    return bre, beams


def _view(x):
    return native.QueryBatchView(x.o, x.d, x.off, x.seg, scenes.SHORT_BEAM if x.short else scenes.LONG_BEAM)


# ---- records of the UPBP and vertex-merging inputs (32-bit words) ---------------------------
def _mis(gen, n):
    m = torch.zeros((n, 16), dtype=torch.float32, device=DEV)
    for k in (0, 1, 2, 5, 6):
        m[:, k] = gen.uni(n, 0.5, 2.0).float()
    m[:, 3], m[:, 4] = gen.uni(n, 1.0, 3.0).float(), gen.uni(n, 1.0, 3.0).float()
    m[:, 7], m[:, 8] = gen.uni(n, 0.2, 1.0).float(), gen.uni(n, -1.0, 1.0).float()
    for k in (9, 10, 11, 12):
        m[:, k] = gen.uni(n, 0.1, 2.0).float()
    m[:, 13] = 1.0
    fl = (gen.uni(n) < 0.1).int() * scenes.MIS_SPECULAR | (gen.uni(n) < 0.7).int() * scenes.MIS_IN_MEDIUM_WITH_BEAMS
    m.view(torch.int32)[:, 14] = fl.to(torch.int32)
    return m


def _light_vertices(gen, paths):
    """Light sub-paths of 1..4 vertices after the source: [n,28] float words, path ends, source mask."""
    counts = gen.integers(1, 5, paths) + 1
    ends = torch.cumsum(counts, 0)
    n = int(ends[-1])
    path = torch.repeat_interleave(torch.arange(paths, device=DEV), counts)
    length = torch.arange(n, device=DEV) - (ends - counts)[path]
    lv = torch.zeros((n, 28), dtype=torch.float32, device=DEV)
    lv[:, 0:3] = gen.uni((n, 3), 0.0, 1e-4).float()
    lv[:, 3:6] = gen.dirs(n)
    lv[:, 6] = gen.uni(n, 0.5, 1.0).float()
    lv[:, 12:28] = _mis(gen, n)
    src = length == 0
    w = lv.view(torch.int32)
    w[:, 7], w[:, 8], w[:, 9] = path.to(torch.int32), length.to(torch.int32), 1
    w[:, 26] = torch.where(src, scenes.MIS_ON_LIGHT_SOURCE, w[:, 26])
    lv[:, 21:25] = torch.where(src[:, None], 0.0, lv[:, 21:25])
    return lv, ends.to(torch.int32), src


def _camera_paths(gen, n):
    length = gen.integers(1, 4, n)
    off = torch.cumsum(length + 1, 0) - (length + 1)
    return length, off, _mis(gen, int((length + 1).sum()))


def _mis_inputs(camera, lv, ends, queries=None, beams=None):
    p = dict(techniques=_abi.PB2D | _abi.BB1D | _abi.BPT | _abi.PP3D | _abi.SURF, query_beam_type=_abi.LONG_BEAM,
             photon_beam_type=_abi.SHORT_BEAM, min_path_length=0, max_path_length=20, surf_factor=0.7,
             pp3d_factor=0.9, pb2d_factor=0.6, bb1d_factor=1.3, bb1d_min_mfp=0.5, min_dist_to_med=0.0,
             has_bb1d_beams=1)
    mi = types.SimpleNamespace(camera=camera, light_vertices=lv, path_ends=ends, params=p)
    return _abi.mis_inputs(mi, _abi.MEM_DEVICE, {"queries": queries, "camera": camera, "light_vertices": lv,
                                                 "path_ends": ends, "beams": beams})


def _upbp_state(c, seed):
    gen = _Gen(seed)
    media = _media(BOX_SPHERE)
    lv, ends, src = _light_vertices(gen, c["paths"])
    n, nb = lv.shape[0], c["beams"]
    ph = scenes.Photons(gen.uni((n, 3)).float(), lv[:, 3:6].contiguous(), lv[:, 0:3].contiguous(), None, 0.005)
    bm = _beams(gen, nb, media, True, 0.003)
    bmis = torch.zeros((nb, 8), dtype=torch.float32, device=DEV)
    w = bmis.view(torch.int32)
    w[:, 0] = gen.integers(0, n, nb).to(torch.int32)
    w[:, 1] = 2 | (gen.uni(nb) < 0.3).to(torch.int32)
    for k, (a, b) in ((2, (0.5, 1.0)), (3, (0.5, 1.0)), (4, (0.5, 2.0))):
        bmis[:, k] = gen.uni(nb, a, b).float()
    o, d = _frame_rays(c["width"], c["height"])
    off, seg, _ = _segments(media, o, d, True)
    q = o.shape[0]
    length, coff, cam = _camera_paths(gen, q)
    qm = torch.zeros((q, 6), dtype=torch.int32, device=DEV)
    qm[:, 0:2] = coff.view(torch.int32).view(q, 2)
    qm[:, 2] = length.to(torch.int32)
    qm[:, 3] = ((length > 1) & (gen.uni(q) < 0.5)).to(torch.int32)
    qm.view(torch.float32)[:, 4] = gen.uni(q, 0.5, 2.0).float()
    ctx = native.Context(0)
    ctx.set_media(media)
    bre, beams = _built(ctx, ph, bm, in_medium=(~src).to(torch.uint8))
    qv = native.QueryBatchView(o, d, off, seg)
    return {"ctx": ctx, "bre": bre, "beams": beams, "qv": qv, "mis": _mis_inputs(cam, lv, ends, qm, bmis)}


def _on_planes(gen, n):
    """Points on three faces of the unit box and the face normals."""
    k = gen.integers(0, 3, n)
    p = gen.uni((n, 3))
    nrm = torch.zeros((n, 3), dtype=torch.float64, device=DEV)
    for i, (ax, sgn, at) in enumerate(((1, 1.0, 0.0), (2, -1.0, 1.0), (0, 1.0, 0.0))):
        p[k == i, ax] = at
        nrm[k == i, ax] = sgn
    return p.float(), nrm


def _hemisphere(gen, nrm):
    d = gen.dirs(nrm.shape[0]).double()
    side = torch.where((d * nrm).sum(-1) < 0, -1.0, 1.0)
    return d * torch.where(gen.uni(nrm.shape[0]) < 0.08, -side, side)[:, None]


def _merge_state(c, seed):
    gen = _Gen(seed)
    media = _media(BOX_SPHERE)
    surf = c["kind"] == "surf"
    lv, ends, src = _light_vertices(gen, c["paths"])
    n, q = lv.shape[0], c["queries"]
    conn = (gen.uni(n) < 0.9) & ~src
    w = lv.view(torch.int32)
    w[:, 10] = conn.to(torch.int32) * scenes.LV_CONNECTABLE
    if surf:
        pos, nrm = _on_planes(gen, n)
        lv[:, 3:6] = _hemisphere(gen, nrm).float()
    else:
        pos = gen.uni((n, 3)).float()
        w[:, 10] |= (~src).to(torch.int32) * scenes.LV_IN_MEDIUM
    length, coff, cam = _camera_paths(gen, q)
    if surf:
        qp, qn = _on_planes(gen, q)
        z = qn + 0.05 * gen.normal((q, 3))
        z = z / z.norm(dim=1, keepdim=True)
        a = torch.where(z[:, :1].abs() > 0.99, torch.tensor([[0.0, 1.0, 0.0]], device=DEV, dtype=torch.float64),
                        torch.tensor([[1.0, 0.0, 0.0]], device=DEV, dtype=torch.float64))
        y = torch.linalg.cross(z, a)
        y = y / y.norm(dim=1, keepdim=True)
        x = torch.linalg.cross(y, z)
        fix = _hemisphere(gen, qn)
        diff, phong = gen.uni((q, 3), 0.05, 0.8), gen.uni((q, 3), 0.05, 0.5)
        lum = torch.tensor([0.212671, 0.715160, 0.072169], device=DEV, dtype=torch.float64)
        ad, ap = diff @ lum, phong @ lum
        rec = torch.zeros((q, 32), dtype=torch.float32, device=DEV)
        rec[:, 0:3], rec[:, 4:7], rec[:, 8:11], rec[:, 12:15] = qp, x.float(), y.float(), z.float()
        rec[:, 7] = torch.clamp((diff + phong).amax(1), max=1.0).float()
        rec[:, 11], rec[:, 15] = (ad / (ad + ap)).float(), (ap / (ad + ap)).float()
        rec[:, 16:19] = torch.stack([(fix * x).sum(-1), (fix * y).sum(-1), (fix * z).sum(-1)], -1).float()
        rec[:, 19] = gen.uni(q, 1.0, 80.0).float()
        rec[:, 20:23], rec[:, 24:27] = diff.float(), phong.float()
        at, off_at = 3, 28
    else:
        qp = gen.uni((q, 3), -0.05, 1.05).float()
        rec = torch.zeros((q, 12), dtype=torch.float32, device=DEV)
        rec[:, 0:3], rec[:, 4:7] = qp, gen.dirs(q)
        p = qp.double()
        inside = ((p >= 0) & (p <= 1)).all(1)
        ball = ((p - torch.tensor(SPHERE_C, device=DEV, dtype=torch.float64)) ** 2).sum(1) <= SPHERE_R ** 2
        rec.view(torch.int32)[:, 3] = torch.where(ball, 2, torch.where(inside, 0, 1)).to(torch.int32)
        at, off_at = 7, 8
    w = rec.view(torch.int32)
    w[:, at] = length.to(torch.int32)
    w[:, off_at:off_at + 2] = coff.view(torch.int32).view(q, 2)
    ctx = native.Context(0)
    ctx.set_media(media)
    torch.cuda.synchronize()
    grid = native.HashGrid(ctx)
    grid.build(pos, lv.view(torch.uint8).view(-1), c["radius"], c["paths"], _abi.SURF if surf else _abi.PP3D)
    return {"ctx": ctx, "grid": grid, "queries": rec.view(torch.uint8).view(-1), "mis": _mis_inputs(cam, lv, ends)}


def _batch_inputs(c, seed):
    """Independent unit-box scenes of uneven size: photons lognormal, a fifth as many beams, random camera rays."""
    gen = _Gen(seed)
    sizes = np.random.Generator(np.random.Philox(c["photons"] + 1000 * c["instances"]))  # of the case, not the seed
    out = []
    for _ in range(c["instances"]):
        n = int(np.clip(sizes.lognormal(math.log(c["photons"]), 1.0), 2_500, 12 * c["photons"]))
        q = int(sizes.uniform(c["queries"] / 100, c["queries"]))
        co = gen.uni((2, 3), 0.05, 3.0).cpu().numpy()
        media = scenes.make_media([(tuple(co[0]), tuple(co[1]), 0.0, 0.8), CLEAR])
        ph = _photons(gen, n, lognormal=0.005)
        bm = _beams(gen, n // 5, media, False, 0.003)
        o, d = _camera(torch.cat([gen.uni((q, 2)), torch.zeros((q, 1), device=DEV)], 1))
        off, seg, pad = _segments(media, o, d, False)
        out.append(types.SimpleNamespace(media=media, o=o, d=d, off=off, seg=seg, pad=pad, photons=ph, beams=bm,
                                         short=False, common=True))
    return out


def _knn_inputs(c, seed):
    gen = _Gen(seed)
    media = _media(BOX_SPHERE)
    return media, _photons(gen, c["photons"], radius=0.5), _beams(gen, c["beams"], media, True, 0.25)


# ---- the cases -----------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind == "upbp":
        return dict(_upbp_state(case, seed), kind=kind)
    if kind in ("pp3d", "surf"):
        return dict(_merge_state(case, seed), kind=kind)
    if kind == "batch":
        ctx = native.Context(0)
        xs = _batch_inputs(case, seed)
        ctx.set_media(np.concatenate([x.media for x in xs]))
        inst, outs = [], []
        for i, x in enumerate(xs):
            bre, beams = _built(ctx, x.photons, x.beams)
            op, ob = (torch.empty((x.o.shape[0], 3), device=DEV) for _ in range(2))
            inst.append((bre, beams, _view(x), 2 * i, op, ob))
            outs.append((op, ob))
        torch.cuda.synchronize()
        return {"kind": kind, "ctx": ctx, "plan": native.BatchPlan(ctx, inst), "outs": outs}
    if kind == "iteration":
        sc = scenes.light_scene(media_rows=TRACE_MEDIA, max_path_length=10, bb1d_min_mfp=0.1, seed=int(seed) + 1,
                                beam_path_count=case["beam_paths"])
        o, d = _frame_rays(case["width"], case["height"])
        off, seg, _ = _segments(sc.media, o, d, True)
        ctx = native.Context(0)
        stream = torch.cuda.Stream()
        ctx.set_stream(stream.cuda_stream)
        ctx.set_media(sc.media)
        return {"kind": kind, "ctx": ctx, "stream": stream, "scene": sc, "paths": case["paths"],
                "capacity": (4 * case["paths"], 8 * case["beam_paths"]), "qv": native.QueryBatchView(o, d, off, seg)}
    if kind == "knn":
        media, ph, bm = _knn_inputs(case, seed)
        ctx = native.Context(0)
        ctx.set_media(media)
        return {"kind": kind, "ctx": ctx, "photons": ph, "beams": bm, "knn": case["knn"]}
    x = _frame_inputs(case, seed)
    if kind == "adjoint":
        host = scenes.Queries(x.o.cpu().numpy(), x.d.cpu().numpy(), x.off.cpu().numpy(),
                              x.seg.cpu().numpy().view(scenes.SEGMENT_DTYPE).reshape(-1))
        w = scenes.Workload("adjoint", x.media, x.photons, x.beams, host)
        torch.cuda.synchronize()
        sigma_s, sigma_a = autograd.media_params(x.media)
        return {"kind": kind, "scene": autograd.DiffScene(w), "sigma_s": sigma_s, "sigma_a": sigma_a,
                "power": x.photons.power.clone(), "target": x.gen.uni((x.o.shape[0], 3)).float()}
    ctx = native.Context(0)
    ctx.set_media(x.media)
    bre, beams = _built(ctx, x.photons, x.beams)
    return {"kind": kind, "ctx": ctx, "bre": bre, "beams": beams, "qv": _view(x)}


def run(s):
    kind = s["kind"]
    if kind == "upbp":
        return native.eval_upbp(s["ctx"], s["bre"], s["beams"], s["qv"], s["mis"])
    if kind in ("pp3d", "surf"):
        return s["grid"].eval(s["queries"], s["mis"])
    if kind == "batch":
        s["plan"].run(use_graph=True)
        return s["outs"]
    if kind == "adjoint":
        p = [s[k].detach().requires_grad_(True) for k in ("sigma_s", "sigma_a", "power")]
        lp, lb = autograd.estimate(s["scene"], *p)
        loss = ((lp + lb - s["target"]) ** 2).sum()
        loss.backward()
        return {"photons": lp.detach(), "beams": lb.detach(), "grads": [x.grad for x in p]}
    if kind == "iteration":
        return _iteration(s)
    if kind == "knn":
        bre = native.EmbreeBre(s["ctx"])
        bre.build(s["photons"], radius_calculation=_abi.KNN_RADIUS, knn=s["knn"])
        beams = native.PhotonBeamsEvaluator(s["ctx"])
        beams.build(s["beams"], radius_calculation=_abi.KNN_RADIUS, knn=s["knn"])
        r = [bre.radii(), *beams.radii()]
        bre.destroy()
        beams.destroy()
        return r
    return native.eval_batch(s["ctx"], s["bre"], s["beams"], s["qv"])


def _iteration(s):
    ctx = s["ctx"]
    with torch.cuda.stream(s["stream"]):
        t = native.trace_light_paths(ctx, s["scene"], s["paths"], capacity=s["capacity"])
        f = {k: t[k].view(torch.int32 if k in ("beam_flags", "beam_medium") else torch.float32) for k in t
             if k.startswith("beam_")}
        lv = t["vertices"].view(torch.float32).view(-1, 28)
        in_medium = ((lv.view(torch.int32)[:, 10] & scenes.LV_IN_MEDIUM) != 0).to(torch.uint8)
        bre = native.EmbreeBre(ctx)
        bre.build(scenes.Photons(t["positions"].view(torch.float32).view(-1, 3), lv[:, 3:6].contiguous(),
                                 lv[:, 0:3].contiguous(), None, 0.005), in_medium=in_medium)
        beams = native.PhotonBeamsEvaluator(ctx)
        beams.build(scenes.Beams(f["beam_origin"].view(-1, 3), f["beam_direction"].view(-1, 3), f["beam_length"],
                                 f["beam_throughput"].view(-1, 3), f["beam_flags"], f["beam_medium"], 0.003))
        out = native.eval_batch(ctx, bre, beams, s["qv"])
        bre.destroy()
        beams.destroy()
    return out


def _hits(c):
    """Expected photon and beam hits of one pass (isotropic, uniform in the unit box)."""
    q = c["queries"] if "queries" in c else c["width"] * c["height"]
    cam = {"rays": 0.45, "stress": 1.02}.get(c["kind"], 0.85)  # mean length of a ray inside the box
    ph = c.get("photons", c.get("paths", 0) * 2.5) if c["kind"] != "stress" else 0
    r2 = 1e-4 if c["kind"] == "frame" and not c.get("sphere") else 3.4e-5
    length = {"stress": 0.25, "rays": 0.35}.get(c["kind"], 0.4)
    return q, q * cam * ph * math.pi * r2, q * cam * c.get("beams", 0) * length * 2 * 0.003 * math.pi / 4


def work(case):
    c, kind = case, case["kind"]
    if kind in ("pp3d", "surf"):
        v = 2.5 * c["paths"]
        found = c["queries"] * v * (4.19 * c["radius"] ** 3 if kind == "pp3d" else 3.14 * c["radius"] ** 2 / 3)
        return {"bytes": c["queries"] * ((48 if kind == "pp3d" else 128) + 3 * 64 + 12) + v * (112 + 12),
                "flops": found * (80 if kind == "pp3d" else 120)}
    if kind == "knn":
        n = c["photons"] + 2 * c["beams"]
        return {"bytes": c["photons"] * 44 + c["beams"] * 60, "flops": n * c["knn"] * 8 * 8}
    if kind == "batch":
        # the sizes are uneven; the means of their distributions
        q, n = c["instances"] * c["queries"] * 0.505, 1.6 * c["photons"]
        f = q * n * 1.02 * math.pi * 3.4e-5 * 30 + q * 1.02 * n / 5 * 0.3 * 0.0047 * 70
        return {"bytes": q * 100 + c["instances"] * n * 55, "flops": f}
    if kind == "iteration":
        q = c["width"] * c["height"]
        return {"bytes": c["paths"] * 1.5 * 124 + c["beam_paths"] * 1.6 * 80 + q * 150,
                "flops": c["paths"] * 300 + q * (c["paths"] * 1.2e-4 * 30 + c["beam_paths"] * 2.6e-3 * 70)}
    q, hp, hb = _hits(c)
    per_p, per_b, per_q = (30, 70, 152)
    if kind == "upbp":
        per_p, per_b, per_q = 150, 200, 400
    if kind == "adjoint":
        per_p, per_b, per_q = 80, 160, 330
    items = c.get("photons", 0) * 44 + c.get("beams", 0) * 48 + c.get("paths", 0) * 3.5 * 124
    return {"bytes": q * per_q + items, "flops": hp * per_p + hb * per_b}


# ---- the same in 64 bits --------------------------------------------------------------------
_PAIRS = 1 << 24  # ray-item pairs of one dense block


def _ray_chunks(x):
    """Ray index chunks; those of camera rays are compact in the image, so that few items are near each."""
    n = x.o.shape[0]
    if not x.common:
        return list(torch.arange(n, device=DEV).split(4096))
    u = x.d.double()[:, :2] / x.d.double()[:, 2:]
    lo, hi = u.amin(0), u.amax(0)
    cells = max(1, int(math.sqrt(n / 1024)))
    c = ((u - lo) / torch.clamp(hi - lo, min=1e-12) * cells).long().clamp(max=cells - 1)
    return list(torch.argsort(c[:, 1] * cells + c[:, 0]).split(1024))


def _nearby(x, rays, centre, reach):
    """Items (bounding spheres) that some ray of the chunk may touch."""
    if not x.common:
        return torch.arange(centre.shape[0], device=DEV)
    d = x.d[rays].double()
    m = d.mean(0)
    m = m / m.norm()
    half = torch.acos(torch.clamp((d @ m).min() / d.norm(dim=1).max(), -1, 1)) + 1e-6
    v = centre - x.o[rays[0]].double()
    dist = v.norm(dim=1)
    ang = torch.acos(torch.clamp(v @ m / dist, -1, 1))
    return ((dist <= reach) | (ang <= half + torch.asin(torch.clamp(reach / dist, max=1.0)))).nonzero()[:, 0]


def _segment_of(x, rays, t, tab):
    """The scattering segment holding t of each ray, or -1."""
    t0, t1, mid, ok = (a[rays] for a in x.pad)
    inside = ok & tab[5][mid] & (t[:, None] > t0.double()) & (t[:, None] < t1.double())
    return torch.where(inside.any(1), inside.int().argmax(1), torch.full_like(rays, -1))


def _photon_pairs(x, tab):
    p = x.photons.position.double()
    r = (x.photons.radius.double() if x.photons.radius is not None
         else torch.full((p.shape[0],), float(np.float32(x.photons.const_radius)), device=DEV, dtype=torch.float64))
    for rays in _ray_chunks(x):
        near = _nearby(x, rays, p, r)
        for items in near.split(max(1, _PAIRS // max(1, rays.shape[0]))):
            o, d, c = x.o[rays].double(), x.d[rays].double(), p[items]
            t = d @ c.T - (d * o).sum(1, keepdim=True)
            vv = (c * c).sum(1)[None] + (o * o).sum(1, keepdim=True) - 2.0 * (o @ c.T)
            s = vv + t * t * ((d * d).sum(1, keepdim=True) - 2.0)
            i, j = (s <= (r * r)[items][None]).nonzero(as_tuple=True)
            t, s = t[i, j], s[i, j]
            k = _segment_of(x, rays[i], t, tab)
            m = k >= 0
            yield rays[i][m], items[j][m], k[m], t[m], torch.clamp(s[m], min=0) / (r * r)[items[j][m]], r[items[j][m]]


def _beam_pairs(x, tab):
    b = x.beams
    bo, bd, bl, r = b.origin.double(), b.direction.double(), b.length.double(), float(np.float32(b.radius))
    step = 0.04
    n = torch.ceil(bl / step).long()
    owner = torch.repeat_interleave(torch.arange(bo.shape[0], device=DEV), n)
    at = (torch.arange(owner.shape[0], device=DEV) - (torch.cumsum(n, 0) - n)[owner] + 0.5) * step
    centre = bo[owner] + bd[owner] * at[:, None]
    reach = torch.full_like(at, step / 2 + r * 1.01)
    bm = b.medium_id.long()
    for rays in _ray_chunks(x):
        near = torch.unique(owner[_nearby(x, rays, centre, reach)])
        o, d = x.o[rays].double(), x.d[rays].double()
        od = torch.linalg.cross(o, d)
        for items in near.split(max(1, _PAIRS // max(1, rays.shape[0]))):
            o2, d2 = bo[items], bd[items]
            ad = d @ torch.linalg.cross(d2, o2).T - od @ d2.T
            q = d @ d2.T
            s2 = (d * d).sum(1, keepdim=True) * (d2 * d2).sum(1)[None] - q * q
            i, j = ((ad * ad < r * r * s2) & ((q * q - 1.0).abs() >= 1e-5)).nonzero(as_tuple=True)
            ad, q, s2 = ad[i, j], q[i, j], s2[i, j]
            w = o[i] - o2[j]
            d2w = (d2[j] * w).sum(1)
            t1 = ((d[i] * w).sum(1) - q * d2w) / (q * q - 1.0)
            t2 = d2w + t1 * q
            k = _segment_of(x, rays[i], t1, tab)
            med = x.pad[2][rays[i], torch.clamp(k, min=0)]
            m = (k >= 0) & (t2 > 0) & (t2 < bl[items[j]]) & (med == bm[items[j]])
            yield (rays[i][m], items[j][m], k[m], t1[m], t2[m], (ad.abs() / torch.sqrt(s2))[m] / r,
                   torch.sqrt(s2)[m], r)


def _phase(g, cos):
    dd = 1.0 + g * g - 2.0 * g * cos
    return torch.where(g.abs() < 1e-3, torch.ones_like(dd), (1.0 - g * g) / (dd * torch.sqrt(dd))) / (4.0 * math.pi)


def _plain(x, sigma=None, power=None):
    """Both estimates of every ray; with `sigma` = (sigma_s, sigma_a) differentiable in them and in `power`."""
    tab = list(_tables(x.media))
    if sigma is not None:
        tab[1], tab[0] = sigma
        tab[2] = sigma[0] + sigma[1]
    ss, st, kch, g = tab[1], tab[2], tab[4], tab[6]
    t0, t1, mid, ok = x.pad
    n = x.o.shape[0]
    ln = (t1 - t0).double()
    # prefix transmittance of the earlier segments
    if sigma is None:
        att = torch.ones((n, 4, 3), device=DEV, dtype=torch.float64)
        pdf = torch.ones((n, 4), device=DEV, dtype=torch.float64)
        att[ok], pdf[ok] = x.seg[:, 4:7].double(), x.seg[:, 2].double()
        if x.short:
            att = att / pdf[..., None]
    else:
        att = torch.where(ok[..., None], torch.exp(-st[mid] * ln[..., None]), torch.ones((), device=DEV, dtype=torch.float64))
    pre = torch.cat([torch.ones((n, 1, 3), device=DEV, dtype=torch.float64), torch.cumprod(att, 1)[:, :3]], 1)

    def normal(med, t):  # exponent of the SHORT normalisation by the smallest sigma_t's channel
        return st[med, kch[med]] * t

    lp = torch.zeros((n, 3), device=DEV, dtype=torch.float64)
    lb = torch.zeros((n, 3), device=DEV, dtype=torch.float64)
    if x.photons is not None:
        power = x.photons.power.double() if power is None else power
        for q, i, k, t, s, r in _photon_pairs(x, tab):
            med = mid[q, k]
            dt = t - t0[q, k].double()
            e = -st[med] * dt[:, None] + (normal(med, dt)[:, None] if x.short else 0.0)
            ph = _phase(g[med], (x.photons.inc_dir[i].double() * x.d[q].double()).sum(1))
            c = pre[q, k] * power[i] * ss[med] * torch.exp(e) * (ph * (1.0 - s) * 2.0 / (math.pi * r * r))[:, None]
            lp = lp.index_add(0, q, c)
    if x.beams is not None:
        b = x.beams
        for q, i, k, t, u, dist, sin, r in _beam_pairs(x, tab):
            med = mid[q, k]
            dt = t - t0[q, k].double()
            e = -st[med] * (dt + u)[:, None]
            if x.short:
                e = e + normal(med, dt)[:, None]
            e = e + torch.where(b.flags[i] == scenes.SHORT_BEAM, normal(med, u), torch.zeros_like(u))[:, None]
            ph = _phase(g[med], -(b.direction[i].double() * x.d[q].double()).sum(1))
            w = ph * (1.0 - dist * dist) * 0.75 / (r * sin)
            lb = lb.index_add(0, q, pre[q, k] * b.throughput[i].double() * ss[med] * torch.exp(e) * w[:, None])
    return lp, lb


def _kth(points, queries, k):
    """Distance of each query to its k-th nearest point (a query that is a point counts itself)."""
    out = []
    for q in queries.split(1024):
        d2 = (q * q).sum(1, keepdim=True) + (points * points).sum(1)[None] - 2.0 * (q @ points.T)
        near = torch.topk(d2, k, dim=1, largest=False).indices[:, k - 1]
        out.append((q - points[near]).norm(dim=1))
    return torch.cat(out)


def _leaf(a):
    return torch.tensor(a.astype(np.float64), device=DEV, requires_grad=True)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("upbp", "iteration", "pp3d", "surf"):
        return None  # weights over whole sub-paths, hashed buckets, the tracer's own random numbers
    if kind == "knn":
        _, ph, bm = _knn_inputs(case, seed)
        k = case["knn"]
        o = bm.origin.double()
        ends = (bm.origin + bm.direction * bm.length[:, None]).double()
        p = ph.position.double()
        beam = [torch.clamp(2.0 * _kth(o, q, k) * bm.radius, min=0.001).cpu().numpy() for q in (o, ends)]
        return [(ph.const_radius * 2.0 * _kth(p, p, k)).cpu().numpy(), *beam]
    if kind == "batch":
        return [_plain(x) for x in _batch_inputs(case, seed)]
    if kind == "stress" and case["queries"] * case["beams"] > 2e11:
        return None
    x = _frame_inputs(case, seed)
    if kind == "adjoint":
        target = x.gen.uni((x.o.shape[0], 3)).float().double()
        if case["width"] * case["height"] * (case["photons"] + 4 * case["beams"]) > 3e11:
            return {"photons": None, "beams": None, "grads": None}
        ss, sa = _leaf(x.media["scattering"]), _leaf(x.media["absorption"])
        power = x.photons.power.double().requires_grad_(True)
        lp, lb = _plain(x, (ss, sa), power)
        ((lp + lb - target) ** 2).sum().backward()
        return {"photons": lp.detach(), "beams": lb.detach(), "grads": [ss.grad, sa.grad, power.grad]}
    lp, lb = _plain(x)
    return (lp if x.photons is not None else None), (lb if x.beams is not None else None)
