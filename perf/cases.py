"""The work that users of this library have it do, as measurable cases.

A case is one call path through the public entry points (mnrt_amd.api, .adjoint, .inverse):

  build    triangle kd-tree of a scene (host-driven build, records attached)
  map      photon kd-tree plus records and query-time data: a photon map made ready to query
  trace    closest hits of camera rays (tile order) or of diffuse bounce rays (incoherent)
  shadow   shadow rays from camera hits to a point light or to samples of an area light
  photons  a photon map traced from the ceiling light (4 bounces, Russian roulette)
  knn      radiance estimate from the k nearest photons at camera or bounce hits
  adjoint  the same estimate under torch.autograd: radiance, dL/dpower, dL/dcolour
  frame    many scenes of uneven size: recorded tree rebuilds, traversal, compaction, kNN
  inverse  one step of batched inverse lighting: loss and gradients of emission and albedo

Scenes are the closed box with spheres, small random triangles and a ceiling light of
mnrt_amd.scene; sizes run from its smallest test scenes (1k triangles, 4k photons) to the
large benchmark scene (1.03M triangles, 1M photons, 1920x1080).  Inputs are made with torch
on the GPU from the seed: triangles by subdivision, and hit points and photons by tracing
the box and the spheres in closed form, so queries have the coherence of a camera's pixel
tiles and photons the uneven density of a lit room.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from mnrt_amd import adjoint, api, inverse
from mnrt_amd import native as N
from mnrt_amd import scene as S

DEV = "cuda"
EPS = 5e-5 * 2.0 * math.sqrt(3.0)  # the scenes' ray epsilon: 5e-5 of the box diagonal
R_MAX = 0.1 * 2.0 * math.sqrt(3.0)  # and their largest query radius: a tenth of it


# ---- the cases -------------------------------------------------------------------------


def listed():
    return [
        # a preview pass over a test scene: one small launch, latency counts
        dict(name="trace_small", kind="trace", tris=1294, width=96, height=64, rays="camera"),
        # the incoherent half of a full-HD frame over the large scene
        dict(name="trace_large", kind="trace", tris=1033054, width=1920, height=1080, rays="bounce"),
        # soft shadows of a mid-size scene at an odd window size
        dict(name="shadow_mid", kind="shadow", tris=205001, width=1023, height=767, light="area"),
        # rebuilding a small animated object's tree
        dict(name="build_small", kind="build", tris=3001),
        # the reference's own construction benchmark at the large scene's size
        dict(name="build_large", kind="build", tris=1033054),
        # a photon map of a million photons made ready to query
        dict(name="map_large", kind="map", photons=1000000),
        # a handful of probes against a small map
        dict(name="knn_small", kind="knn", photons=20001, k=50, width=83, height=49, rays="camera"),
        # the kNN stage of a full-HD frame's bounce hits, k as the reference's global map
        dict(name="knn_large", kind="knn", photons=1000000, k=100, width=1920, height=1080, rays="bounce"),
        # one differentiable render of a small window: forward and backward
        dict(name="adjoint_mid", kind="adjoint", photons=131072, k=50, width=321, height=241),
        # tracing the photon map of a mid-size scene
        dict(name="photons_mid", kind="photons", tris=51201, target=262144),
        # 32 uneven scenes rebuilt, traced and queried in one step
        dict(name="frame_batch", kind="frame", scenes=32, tris=20000, photons=65536, pixels=131072, k=50),
        # an inverse-lighting step over 8 scenes with 4 lights each
        dict(name="inverse_step", kind="inverse", scenes=8, tris=12000, photons=65536, pixels=65536, k=50),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _window(rng, lo, hi):
    """A window of lo..hi pixels, any width and height (odd ones among them)."""
    px = _log(rng, lo, hi)
    w = max(8, int(round(math.sqrt(px * rng.uniform(1.0, 1.8)))))
    return dict(width=w, height=max(8, px // w))


def draw(rng):
    kind = rng.choice(["build", "map", "trace", "trace", "shadow", "photons", "knn", "knn", "adjoint", "frame",
                       "inverse"])
    c = dict(kind=kind)
    if kind in ("build", "trace", "shadow"):
        c["tris"] = _log(rng, 1000, 1000000)
    if kind == "map":
        c["photons"] = _log(rng, 4000, 1000000)
    if kind in ("trace", "shadow"):
        c.update(_window(rng, 4000, 1900000))
    if kind == "trace":
        c["rays"] = rng.choice(["camera", "bounce"])
    if kind == "shadow":
        c["light"] = rng.choice(["point", "area"])
    if kind == "photons":
        c.update(tris=_log(rng, 1000, 200000), target=_log(rng, 4000, 500000))
    if kind == "knn":
        c.update(photons=_log(rng, 4000, 1000000), k=rng.choice([50, 100, 200]),
                 rays=rng.choice(["camera", "bounce"]), **_window(rng, 4000, 900000))
    if kind == "adjoint":
        c.update(photons=_log(rng, 4000, 500000), k=rng.choice([50, 100]), **_window(rng, 4000, 300000))
    if kind == "frame":
        c.update(scenes=rng.randint(2, 32), tris=_log(rng, 2000, 20000), photons=_log(rng, 8000, 65536),
                 pixels=_log(rng, 16000, 131072), k=rng.choice([50, 100]))
    if kind == "inverse":
        c.update(scenes=rng.randint(2, 8), tris=_log(rng, 2000, 12000), photons=_log(rng, 8000, 65536),
                 pixels=_log(rng, 8000, 65536), k=50)
    return c


# ---- inputs ----------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _rand(g, *shape):
    return torch.rand(shape, device=DEV, generator=g)


def _f4(a):
    out = torch.zeros((a.shape[0], 4), dtype=torch.float32, device=DEV)
    out[:, :3] = a
    return out


def _unit(a):
    return a / a.norm(dim=1, keepdim=True).clamp_min(1e-30)


def _sphere_faces(subdiv):
    """Faces (20 * 4**subdiv, 3, 3) of a subdivided icosahedron on the unit sphere."""
    f = torch.from_numpy(S.icosphere(0)).to(DEV)
    for _ in range(subdiv):
        a, b, c = f[:, 0], f[:, 1], f[:, 2]
        ab, bc, ca = _unit(a + b), _unit(b + c), _unit(c + a)
        f = torch.cat([torch.stack(t, 1) for t in ((a, ab, ca), (b, bc, ab), (c, ca, bc), (ab, bc, ca))])
    return f


def _spheres(count, g):
    """Centres and radii: one sphere near the middle, or many anywhere in the box."""
    u = _rand(g, count, 4)
    if count == 1:
        return (u[:, :3] - 0.5) * 0.6, 0.3 + 0.3 * u[:, 3]
    return u[:, :3] * 2 - 1, 0.05 + 0.25 * u[:, 3]


def _sphere_plan(tris):
    """How many spheres, and how finely divided, a scene of `tris` triangles has."""
    count = 1 if tris < 100000 else min(48, tris // 20480)
    sub = 0
    while count * 20 * 4 ** (sub + 1) <= (0.96 if count > 1 else 0.5) * tris and sub < 5:
        sub += 1
    return count, sub


def _ball(g, n):
    d = _unit(torch.randn((n, 3), device=DEV, generator=g))
    return d * _rand(g, n, 1) ** (1.0 / 3.0)


def _scene(tris, seed, lights=1):
    """(v0, v1, v2, albedo, lights, centres, radii) of a scene of exactly `tris` triangles."""
    g = _gen(seed)
    count, sub = _sphere_plan(tris)
    cen, rad = _spheres(count, g)
    parts = [torch.from_numpy(S.box_tris()).to(DEV)]
    unit = _sphere_faces(sub)
    parts.append((unit[None] * rad.double()[:, None, None, None] + cen.double()[:, None, None, :]).reshape(-1, 3, 3))
    rest = tris - 12 - parts[1].shape[0] - 2 * lights
    a = _rand(g, max(rest, 0), 3) * 2 - 1
    e = 0.05 * _rand(g, max(rest, 0), 2)
    t = torch.stack([a, a + _ball(g, a.shape[0]) * e[:, :1], a + _ball(g, a.shape[0]) * e[:, 1:]], 1).clamp(-1, 1)
    parts.append(t.double())
    recs = []
    spots = [(0.0, 0.0)] if lights == 1 else [(-0.5, -0.5), (0.5, 0.5), (0.5, -0.5), (-0.5, 0.5)][:lights]
    for xz in spots:
        q = S.light_quad(xz)
        parts.append(torch.from_numpy(q).to(DEV))
        recs.append([q[0][0], q[0][1] - q[0][0], q[0][2] - q[0][1], [10.0, 10.0, 10.0]])
    v = torch.cat(parts).float()
    alb = torch.tensor([0.7, 0.7, 0.7, 1.0], device=DEV).repeat(v.shape[0], 1)
    alb[-2 * lights:, :3] = 0.0
    return (_f4(v[:, 0]), _f4(v[:, 1]), _f4(v[:, 2]), alb, np.array(recs, np.float32), cen, rad)


def _camera(width, height):
    """Origins and directions of a pinhole camera at (0, 0, 0.9), 8x8 pixel tiles in order."""
    py, px = torch.meshgrid(torch.arange(height, device=DEV), torch.arange(width, device=DEV), indexing="ij")
    px, py = px.reshape(-1), py.reshape(-1)
    key = (((py // 8) * ((width + 7) // 8) + px // 8) * 8 + py % 8) * 8 + px % 8
    at = torch.argsort(key)
    px, py = px[at].double(), py[at].double()
    d = torch.stack([(2 * (px + 0.5) / width - 1) * (width / height), 1 - 2 * (py + 0.5) / height,
                     -torch.ones_like(px)], 1)
    o = torch.tensor([0.0, 0.0, 0.9], device=DEV).repeat(d.shape[0], 1)
    return o, _unit(d).float()


def _hit(o, d, cen, rad):
    """First hit of the box's inside and the spheres: (points, normals facing the ray)."""
    inv = 1.0 / torch.where(d.abs() < 1e-12, torch.full_like(d, 1e-12), d)
    far = torch.maximum((1 - o) * inv, (-1 - o) * inv)
    t, axis = far.min(dim=1)
    best = torch.full_like(t, -1.0)
    for s in range(cen.shape[0]):
        m = o - cen[s]
        b = (m * d).sum(1)
        disc = b * b - (m * m).sum(1) + rad[s] * rad[s]
        r = disc.clamp_min(0).sqrt()
        x = torch.where(-b - r > 1e-3, -b - r, -b + r)
        ok = (disc > 0) & (x > 1e-3) & (x < t)
        t = torch.where(ok, x, t)
        best = torch.where(ok, torch.full_like(best, float(s)), best)
    p = (o + d * t[:, None]).clamp(-1, 1)
    n = torch.zeros_like(p).scatter_(1, axis[:, None], 1.0)
    on = best >= 0
    n = torch.where(on[:, None], _unit(p - cen[best.clamp_min(0).long()]), n)
    return p, torch.where((n * d).sum(1, keepdim=True) > 0, -n, n)


def _scatter(n, g):
    """Cosine-distributed directions about unit normals."""
    return _unit(n + 0.9999 * _unit(torch.randn(n.shape, device=DEV, generator=g)))


def _photon_map(count, cen, rad, g):
    """(positions, powers, directions) of a photon map: paths from the ceiling light, five
    stored hits each, in path order as the photon tracer stores them."""
    m = (count + 4) // 5
    o = torch.stack([_rand(g, m) * 0.5 - 0.25, torch.full((m,), 0.999, device=DEV), _rand(g, m) * 0.5 - 0.25], 1)
    d = _scatter(torch.tensor([0.0, -1.0, 0.0], device=DEV).repeat(m, 1), g)
    w = torch.full((m, 3), 10.0 / m, device=DEV) * (0.5 + _rand(g, m, 3))
    pos, pw, dr = [], [], []
    for _ in range(5):
        p, n = _hit(o, d, cen, rad)
        pos.append(p), pw.append(w), dr.append(d)
        o, d, w = p, _scatter(n, g), w * (0.5 + 0.4 * _rand(g, m, 3))
    cut = lambda a: _f4(torch.stack(a, 1).reshape(-1, 3)[:count])  # noqa: E731
    return cut(pos), cut(pw), cut(dr)


def _rays(case, cen, rad, g):
    o, d = _camera(case["width"], case["height"])
    if case.get("rays") == "bounce":
        o, n = _hit(o, d, cen, rad)
        d = _scatter(n, g)
    return o, d


def _queries(case, cen, rad, g):
    """Shading points at the rays' hits: pos, nrm, dir, clr, infl (float4 arrays)."""
    o, d = _rays(case, cen, rad, g)
    p, n = _hit(o, d, cen, rad)
    clr = torch.cat([0.2 + 0.7 * _rand(g, p.shape[0], 3), torch.ones((p.shape[0], 1), device=DEV)], 1)
    infl = torch.ones((p.shape[0], 4), device=DEV)
    if case.get("rays") == "bounce":
        infl[:, :3] = 0.7
    infl[:, 3] = 0.0
    return dict(pos=_f4(p), nrm=_f4(n), dir=_f4(d), clr=clr.float(), infl=infl)


def _knn_inputs(case, seed):
    g = _gen(seed)
    cen, rad = _spheres(48 if case["photons"] >= 500000 else 1, g)
    ppos, ppow, pdir = _photon_map(case["photons"], cen, rad, g)
    return ppos, ppow, pdir, _queries(case, cen, rad, g), g


def _light_samples(n, g):
    """Points on the ceiling light of the scenes."""
    return _f4(torch.stack([_rand(g, n) * 0.5 - 0.25, torch.full((n,), 0.998, device=DEV), _rand(g, n) * 0.5 - 0.25],
                           1))


def _ray_inputs(case, seed):
    v0, v1, v2, _, _, cen, rad = _scene(case["tris"], seed)
    g = _gen(seed + 1)
    if case["kind"] == "trace":
        o, d = _rays(case, cen, rad, g)
        return v0, v1, v2, _f4(o), _f4(d)
    p, _ = _hit(*_camera(case["width"], case["height"]), cen, rad)
    return v0, v1, v2, _f4(p), _light_samples(p.shape[0], g)


BOX = np.array([-1, -1, -1, 1, 1, 1], np.float32)


def _spread(case, what):
    """Per-scene sizes of a batch: log-uniform in [top / 8, top], the same for every seed."""
    rng = np.random.default_rng(len(what))
    top = case[what]
    return np.exp(rng.uniform(math.log(top / 8), math.log(top), case["scenes"])).astype(int)


def _offsets(counts):
    off = np.zeros(len(counts) + 1, np.uint32)
    off[1:] = np.cumsum(np.asarray(counts, np.int64))
    return off


def _dims(pixels):
    w = 8 * max(1, int(round(math.sqrt(pixels) / 8)))
    return w, max(1, int(round(pixels / w)))


class _Words:
    """A tree's device array, for torch.as_tensor."""

    def __init__(self, address, shape, kind):
        self.__cuda_array_interface__ = dict(shape=shape, typestr=kind, data=(int(address), False), version=3)


def _room(elems, refs):
    """The caller's arrays for a tree of `elems` elements, larger than any such tree."""
    return dict(nodes=torch.zeros((4 * elems + 4096, 2), dtype=torch.int32, device=DEV),
                refs=torch.zeros(refs, dtype=torch.int32, device=DEV))


def _take(T, room):
    """Copies a tree out, as a program does that caches it or ships it to another device."""
    t = T.t
    room["nodes"][:t.num_nodes].copy_(torch.as_tensor(_Words(t.d_nodes, (t.num_nodes, 2), "<i4"), device=DEV))
    room["refs"][:t.num_refs].copy_(torch.as_tensor(_Words(t.d_refs, (t.num_refs,), "<i4"), device=DEV))
    return dict(room)


# ---- preparing and running --------------------------------------------------------------


def prepare(case, seed):
    k = case["kind"]
    st = dict(kind=k)
    if k == "build":
        st.update(v=_scene(case["tris"], seed)[:3], room=_room(case["tris"], 6 * case["tris"] + 4096))
    elif k == "map":
        g = _gen(seed)
        cen, rad = _spheres(48 if case["photons"] >= 500000 else 1, g)
        st["photons"] = _photon_map(case["photons"], cen, rad, g)
        st.update(params=api.default_params(N.KIND_POINT, BOX, R_MAX), room=_room(case["photons"], case["photons"]))
    elif k in ("trace", "shadow"):
        v0, v1, v2, a, b = _ray_inputs(case, seed)
        st.update(tree=api.build_tri(v0, v1, v2), a=a, b=b)
        if k == "shadow" and case["light"] == "point":
            st.update(light=api.make_light(N.LIGHT_POINT, (0.0, 0.99, 0.0)), b=None)
        elif k == "shadow":
            st["light"] = api.make_light(N.LIGHT_AREA_RECT, (-0.25, 0.998, -0.25), (0.0, -1.0, 0.0),
                                         v1=(0.5, 0.0, 0.0), v2=(0.0, 0.0, 0.5))
    elif k == "photons":
        v0, v1, v2, alb, lights, _, _ = _scene(case["tris"], seed)
        st.update(tree=api.build_tri(v0, v1, v2), v=(v0, v1, v2), albedo=alb, lights=lights, target=case["target"],
                  seed=seed & 0xFFFF)
    elif k in ("knn", "adjoint"):
        ppos, ppow, pdir, q, g = _knn_inputs(case, seed)
        pmap = api.build_points(ppos, api.default_params(N.KIND_POINT, BOX, R_MAX))
        api.attach_photon_records(pmap, ppos, ppow, pdir)
        st.update(map=pmap, q=q, k=case["k"])
        if k == "adjoint":
            st.update(ppos=ppos, pdir=pdir, power=ppow.requires_grad_(True), clr=q["clr"].requires_grad_(True),
                      target=_target(q, g))
    elif k == "frame":
        st.update(_prepare_frame(case, seed))
    elif k == "inverse":
        st.update(_prepare_inverse(case, seed))
    return st


def _target(q, g):
    """Radiance to match, of the magnitude the estimate has."""
    n = q["pos"].shape[0]
    return torch.cat([_rand(g, n, 3) * 2.0, torch.zeros((n, 1), device=DEV)], 1)


def _prepare_frame(case, seed):
    ns = case["scenes"]
    scenes = [_scene(int(n), seed * 131 + s) for s, n in enumerate(_spread(case, "tris"))]
    maps = [_photon_map(int(n), sc[5], sc[6], _gen(seed * 137 + s))
            for s, (n, sc) in enumerate(zip(_spread(case, "photons"), scenes))]
    cams = [_camera(*_dims(n)) for n in _spread(case, "pixels")]
    cat = lambda parts: torch.cat(parts).contiguous()  # noqa: E731
    v0, v1, v2, alb = (cat([sc[i] for sc in scenes]) for i in range(4))
    ppos, ppow, pdir = (cat([m[i] for m in maps]) for i in range(3))
    toff, poff = _offsets([sc[0].shape[0] for sc in scenes]), _offsets([m[0].shape[0] for m in maps])
    roff = _offsets([c[0].shape[0] for c in cams])
    eps, rmax = np.full(ns, EPS, np.float32), np.full(ns, R_MAX, np.float32)
    tri = api.BuildGraph(N.KIND_TRI, toff, v0, v1, v2)
    pts = api.BuildGraph(N.KIND_POINT, poff, ppos, power=ppow, dirs=pdir, root_boxes=np.tile(BOX, (ns, 1)),
                         max_query_radius=rmax)
    batch = api.QueryBatch(tri.trees, toff, roff, eps, pts.trees, rmax, case["k"])
    n = int(roff[-1])
    f4 = lambda: torch.zeros((n, 4), device=DEV)  # noqa: E731
    bufs = dict(orig4=_f4(cat([c[0] for c in cams])), dir4=_f4(cat([c[1] for c in cams])), v0=v0, v1=v1, v2=v2,
                albedo4=alb, hit_tri=torch.zeros(n, dtype=torch.int32, device=DEV),
                hit_t=torch.zeros(n, device=DEV), sp_pos4=f4(), sp_nrm4=f4(), sp_dir4=f4(), sp_clr4=f4(),
                sp_infl4=f4(), sp_count=torch.zeros(ns, dtype=torch.int32, device=DEV), io_rad4=f4())
    batch.make_io(**bufs)
    for phase in (N.PHASE_TRACE, N.PHASE_SHADE, N.PHASE_KNN):
        batch.capture(phase)
    return dict(tri=tri, pts=pts, batch=batch, bufs=bufs)


def _prepare_inverse(case, seed):
    scenes = []
    for s, n in enumerate(_spread(case, "tris")):
        v0, v1, v2, alb, lights, _, _ = _scene(int(n), seed * 131 + s, lights=4)
        scenes.append(S.Scene(*(a.cpu().numpy() for a in (v0, v1, v2, alb)), lights))
    fit = inverse.BatchedInverseLighting(scenes, _spread(case, "photons"),
                                         [_dims(n) for n in _spread(case, "pixels")], case["k"], seed & 0xFFFF)
    g = _gen(seed)
    truth = 0.5 + 1.5 * _rand(g, 4 * case["scenes"], 3)
    target = fit.full_target(fit.radiance(truth, fit.albedo0))
    e = 0.5 + 1.5 * _rand(g, 4 * case["scenes"], 3)
    a = (fit.albedo0 * (0.8 + 0.4 * _rand(g, *fit.albedo0.shape))).contiguous()
    return dict(fit=fit, target=target, emission=e, albedo=a)


def run(st):
    k = st["kind"]
    if k == "build":
        return _take(api.build_tri(*st["v"]), st["room"])
    if k == "map":
        T = api.build_points(st["photons"][0], st["params"])
        api.attach_photon_records(T, *st["photons"])
        return _take(T, st["room"])
    if k == "trace":
        tri, t, bary, _ = api.trace_closest(st["tree"], st["a"], st["b"], EPS)
        return dict(tri=tri, t=t, bary=bary)
    if k == "shadow":
        return dict(visible=api.trace_shadow(st["tree"], st["light"], st["a"], EPS, st["b"]))
    if k == "photons":
        return api.photons_generate(st["tree"], *st["v"], st["albedo"], st["lights"], st["target"], 4, st["seed"],
                                    EPS, want_meta=True)
    q = st.get("q")
    if k == "knn":
        return dict(rad=api.knn_gather(st["map"], st["k"], R_MAX, q["pos"], q["nrm"], q["dir"], q["infl"],
                                       q["clr"])["rad"])
    if k == "adjoint":
        power, clr = st["power"], st["clr"]
        power.grad = clr.grad = None
        rad = adjoint.knn_radiance(power, clr, st["map"], st["ppos"], st["pdir"], q, st["k"], R_MAX)
        torch.square(rad - st["target"])[:, :3].sum().backward()
        return dict(rad=rad.detach(), grad_power=power.grad, grad_clr=clr.grad)
    if k == "frame":
        b = st["bufs"]
        st["tri"].replay()
        st["pts"].replay()
        b["io_rad4"].zero_()
        for phase in (N.PHASE_TRACE, N.PHASE_SHADE, N.PHASE_KNN):
            st["batch"].replay(phase)
        return dict(tri=b["hit_tri"], t=b["hit_t"], count=b["sp_count"], rad=b["io_rad4"])
    loss, ge, ga = st["fit"].loss_and_grad(st["emission"], st["albedo"], st["target"])
    return dict(loss=loss, grad_emission=ge, grad_albedo=ga, rad=st["fit"].bufs["io_rad4"])


# ---- what a pass cannot do without ---------------------------------------------------


def work(case):
    """Bytes: inputs read once (float3 payloads as the 16-byte rows they come in), outputs
    written once.  Operations: one distance per kept neighbour (8), one ray-triangle test per
    ray (50), one bound update per element and tree level (20)."""
    k = case["kind"]
    levels = lambda n: max(1.0, math.log2(max(n, 2)))  # noqa: E731
    rays = case.get("width", 0) * case.get("height", 0)
    if k == "build":
        n = case["tris"]
        return dict(bytes=n * (48 + 8 + 4 + 48), flops=20 * n * levels(n))
    if k == "map":
        n = case["photons"]
        return dict(bytes=n * (48 + 2 + 4 + 32), flops=20 * n * levels(n))
    if k == "trace":
        return dict(bytes=rays * (32 + 16) + case["tris"] * 48, flops=50 * rays)
    if k == "shadow":
        return dict(bytes=rays * (36 if case["light"] == "area" else 20) + case["tris"] * 48, flops=50 * rays)
    if k == "photons":
        n = case["target"]
        return dict(bytes=n * (48 + 24) + case["tris"] * 64, flops=50 * n)
    if k == "knn":
        return dict(bytes=rays * (80 + 16) + case["photons"] * 32, flops=8 * rays * case["k"])
    if k == "adjoint":
        return dict(bytes=rays * (80 + 16 + 16 + 80 + 16 + 16) + case["photons"] * (48 + 32 + 32 + 16),
                    flops=8 * rays * case["k"] * 2)
    s, mean = case["scenes"], (1 - 1 / 8) / math.log(8)  # the mean of log-uniform sizes
    t, p, r = (s * mean * case[w] for w in ("tris", "photons", "pixels"))
    if k == "frame":
        return dict(bytes=t * 108 + p * 86 + r * (48 + 96 + 96), flops=r * (50 + 8 * case["k"]))
    return dict(bytes=p * (16 + 20 + 16 + 48 + 32 + 32 + 16) + r * (96 + 128) + t * 24, flops=16 * r * case["k"])


# ---- values in 64 bits ---------------------------------------------------------------


def exact(case, seed):
    k = case["kind"]
    if k == "trace":
        if case["width"] * case["height"] * case["tris"] > 4e9:
            return None
        v0, v1, v2, o, d = (a[:, :3].double() for a in _ray_inputs(case, seed))
        return dict(tri=None, t=_closest(v0, v1, v2, o, d), bary=None)
    if k in ("knn", "adjoint"):
        n = case["width"] * case["height"]
        if n * case["photons"] > 2e10:
            return None
        return _radiance(case, seed)
    return None


def _cross(a, b):
    return torch.linalg.cross(a, b)


def _closest(v0, v1, v2, o, d):
    """Distance to the first triangle beyond EPS along each ray; 0 where there is none."""
    e1, e2, out = v1 - v0, v2 - v0, []
    for lo in range(0, o.shape[0], max(1, 20000000 // v0.shape[0])):
        oo, dd = (a[lo:lo + max(1, 20000000 // v0.shape[0]), None] for a in (o, d))
        pv = _cross(dd.expand(-1, e2.shape[0], -1), e2[None].expand(dd.shape[0], -1, -1))
        inv = 1.0 / (pv * e1).sum(-1)
        tv = oo - v0
        u = (tv * pv).sum(-1) * inv
        qv = _cross(tv, e1[None].expand_as(tv))
        v = (qv * dd).sum(-1) * inv
        t = (qv * e2).sum(-1) * inv
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t > EPS)
        best = torch.where(ok, t, torch.full_like(t, math.inf)).min(1).values
        out.append(torch.where(best.isinf(), torch.zeros_like(best), best))
    return torch.cat(out)


def _stored_dirs(d):
    """Photon directions as the records hold them: two 16-bit octahedral coordinates."""
    d = d / d.abs().sum(1, keepdim=True)
    sign = lambda a: torch.where(a >= 0, torch.ones_like(a), -torch.ones_like(a))  # noqa: E731
    fold = lambda a: (1 - a.flip(1).abs()) * sign(a)  # noqa: E731
    uv = torch.where(d[:, 2:] < 0, fold(d[:, :2]), d[:, :2])
    uv = torch.round(uv * 32767) / 32767
    z = 1 - uv.abs().sum(1, keepdim=True)
    return torch.cat([torch.where(z < 0, fold(uv), uv), z], 1)


def _radiance(case, seed):
    """rad = alpha rho / pi * (front-facing power of the k nearest) / (pi r^2) * influence,
    and the gradients of the squared difference to the target."""
    ppos, ppow, pdir, q, g = _knn_inputs(case, seed)
    pos, power, pd = ppos[:, :3].double(), ppow[:, :3].double(), _stored_dirs(pdir[:, :3].double())
    n, k = q["pos"].shape[0], case["k"]
    clr, infl = q["clr"].double(), q["infl"][:, :3].double()
    target = _target(q, g).double()
    nq, rd = q["nrm"][:, :3].double(), q["dir"][:, :3].double()
    nq = torch.where((-(rd * nq).sum(1, keepdim=True)) < 0, -nq, nq)
    rad, gc = torch.zeros((n, 4), dtype=torch.float64, device=DEV), torch.zeros((n, 4), dtype=torch.float64, device=DEV)
    gp = torch.zeros((power.shape[0], 4), dtype=torch.float64, device=DEV)
    step = max(1, 100000000 // pos.shape[0])
    for lo in range(0, n, step):
        s = slice(lo, min(n, lo + step))
        x = q["pos"][s, :3].double()
        d2 = sum((x[:, None, c] - pos[None, :, c]).square() for c in range(3))
        near, at = d2.topk(k, dim=1, largest=False)
        inside = near < R_MAX * R_MAX
        r2 = torch.where(inside.all(1), near[:, -1], torch.full_like(near[:, -1], R_MAX * R_MAX))
        front = inside & ((pd[at] * nq[s, None]).sum(-1) < 0)
        irr = (power[at] * front[..., None]).sum(1) / (math.pi * r2)[:, None]
        irr = irr * (inside.sum(1) >= 8)[:, None]
        f = clr[s, 3:] / math.pi * infl[s]
        rad[s, :3] = clr[s, :3] * f * irr
        if case["kind"] == "adjoint":
            up = 2 * (rad[s, :3] - target[s, :3])
            gc[s, :3] = up * f * irr
            w = up * clr[s, :3] * f / (math.pi * r2)[:, None] * (inside.sum(1) >= 8)[:, None]
            w = w[:, None] * front[..., None]
            gp[:, :3].index_add_(0, at.reshape(-1), w.reshape(-1, 3))
    return dict(rad=rad) if case["kind"] == "knn" else dict(rad=rad, grad_power=gp, grad_clr=gc)
