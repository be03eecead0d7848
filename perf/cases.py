"""Performance cases of the renderer, through its public Python entry points.

listed() names twelve pieces of work a program has the library do: ray queries
on host and device arrays, path-traced frames from a small preview to the
1080p benchmark frame, the Phong and Whitted renderers, a batch of scenes in
one graph, the radiance cache's training gradient and a frame rendered with a
trained cache.  draw() gives more of the same ranges.  A case is a dict of
plain values; prepare() makes what a program has in hand before the call
(scene uploaded, film or arrays allocated), run() is one call and its results.

A scene's geometry and its BVH are an asset that is built once; the seed moves
the camera, the rays, the random streams, the cache's weights and its samples
(and picks the soup).
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import raycer_amd as ra
from raycer_amd import api

CACHE_FAN = [(81, 64), (64, 64), (64, 64), (64, 64), (64, 3)]


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # An editor's pick or a physics probe: a few hundred host rays into a
        # small room, one synchronous call.  Latency only.
        {"name": "query_host_box", "op": "closest_host", "scene": "box", "size": 0, "n": 1013},
        # A lightmapper's or simulator's bounce: device-resident rays leaving
        # the surface of a large terrain in random directions.
        {"name": "query_closest_terrain", "op": "closest_device", "scene": "terrain", "size": 1024, "n": 1 << 20},
        # Visibility of point pairs (occlusion baking): device-resident rays
        # with a finite range through a cloud of triangles, ragged count.
        {"name": "query_any_soup", "op": "any_device", "scene": "soup", "size": 200000, "n": 777777},
        # The Cornell-style box at its test size: a preview frame, launches and
        # latency count.
        {"name": "render_box_preview", "op": "render", "scene": "box", "size": 0, "width": 256, "height": 256,
         "spp": 16, "depth": 8, "sampler": "jittered", "filter": "box", "hit": "fp32"},
        # A ragged thumbnail with the exact (FP64) triangle decision, another
        # sampler and filter.
        {"name": "render_soup_thumbnail_fp64", "op": "render", "scene": "soup", "size": 100000, "width": 499,
         "height": 373, "spp": 9, "depth": 5, "sampler": "cmj", "filter": "bell", "hit": "fp64"},
        # The benchmark frame: 2,093,058 triangles, 1080p, 64 samples.
        {"name": "render_terrain_1080p", "op": "render", "scene": "terrain", "size": 1024, "width": 1920,
         "height": 1080, "spp": 64, "depth": 6, "sampler": "jittered", "filter": "tent", "hit": "fp32"},
        # Primary ray + shadow ray + Phong at 1080p into page-locked arrays
        # (1,179,648 triangles), as the benchmark runs it.
        {"name": "phong_1080p", "op": "phong", "scene": "sphere", "size": 7, "width": 1920, "height": 1080},
        # The Whitted tracer as the benchmark runs it: mirrors, three
        # reflection levels, one point light.
        {"name": "whitted_mirror_1080p", "op": "whitted", "scene": "sphere", "size": 7, "width": 1920,
         "height": 1080, "spp": 1, "glossy": 0, "ao": 0, "area": 0},
        # The Whitted tracer with what makes its ray trees wide: glossy
        # reflection, ambient occlusion, an area light, fog; odd height.
        {"name": "whitted_glossy", "op": "whitted", "scene": "sphere", "size": 5, "width": 640, "height": 361,
         "spp": 4, "glossy": 2, "ao": 2, "area": 2},
        # Several scenes of a dataset in one captured graph.
        {"name": "batch_8_scenes", "op": "batch", "count": 8, "spp": 16, "branches": 8},
        # One training batch of the radiance cache at its default size.
        {"name": "cache_gradient", "op": "gradient", "n": 65536},
        # A frame whose paths end into a trained cache after one bounce.
        {"name": "render_cached_terrain", "op": "cached", "scene": "terrain", "size": 512, "width": 960,
         "height": 540, "spp": 16, "depth": 6, "vertex": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ranges at other sizes, odd ones among them."""
    op = rng.choice(["closest_host", "closest_device", "any_device", "render", "render", "render", "phong",
                     "whitted", "batch", "gradient", "cached"])
    scene = rng.choice(["box", "terrain", "soup"])
    size = {"box": 0, "terrain": _log(rng, 33, 1024), "soup": _log(rng, 1000, 300000)}[scene]
    if op == "closest_host":
        return {"op": op, "scene": scene, "size": size, "n": _log(rng, 64, 200000)}
    if op in ("closest_device", "any_device"):
        return {"op": op, "scene": scene, "size": size, "n": _log(rng, 4096, 1 << 21)}
    if op == "phong":
        return {"op": op, "scene": "sphere", "size": rng.randint(3, 7), "width": _log(rng, 128, 1920),
                "height": _log(rng, 96, 1080)}
    if op == "whitted":
        glossy, ao, area = rng.choice([(0, 0, 0), (0, 2, 0), (2, 0, 2), (2, 2, 2), (0, 0, 3)])
        heavy = glossy or ao or area
        return {"op": op, "scene": "sphere", "size": rng.randint(3, 7), "width": _log(rng, 128, 640 if heavy else 1920),
                "height": _log(rng, 96, 400 if heavy else 1080), "spp": rng.choice([1, 1, 4]), "glossy": glossy,
                "ao": ao, "area": area}
    if op == "batch":
        return {"op": op, "count": rng.randint(2, 10), "spp": rng.randint(4, 16), "branches": rng.randint(1, 8)}
    if op == "gradient":
        return {"op": op, "n": _log(rng, 512, 65536)}
    case = {"op": op, "scene": scene, "size": size, "width": _log(rng, 96, 1280), "height": _log(rng, 64, 720),
            "spp": rng.choice([1, 4, 9, 16]), "depth": rng.randint(4, 8)}
    if op == "cached":
        return {**case, "vertex": rng.randint(1, 2)}
    return {**case, "sampler": rng.choice(["jittered", "random", "cmj"]),
            "filter": rng.choice(["box", "tent", "gaussian", "bell"]), "hit": rng.choice(["fp32", "fp32", "fp64"])}


# ------------------------------------------------------------------ scenes
@functools.lru_cache(maxsize=24)
def _asset(kind, size, seed):
    """Geometry and binned-SAH BVH of a scene."""
    p = {"box": ra.scene_params(api.RCH_SCENE_BOX),
         "terrain": ra.scene_params(api.RCH_SCENE_TERRAIN, seed=1, grid=size),
         "sphere": ra.scene_params(api.RCH_SCENE_SPHERE_GROUND, seed=1, level=size, grid=1 << (size + 2)),
         "soup": ra.scene_params(api.RCH_SCENE_SOUP, seed=seed, tri_count=size)}[kind]
    sd = ra.generate_scene(p)
    nodes, ordered, _, _ = ra.build_bvh(sd.vertices, method=api.RCH_BVH_BINNED)
    return sd, nodes, ordered


def _scene(kind, size, seed):
    return _asset(kind, size, 1 + seed % 3 if kind == "soup" else 0)


@functools.lru_cache(maxsize=2)
def _context(hit):
    """The program's contexts: one per triangle decision."""
    ctx = ra.Context(0)
    ctx.set_hit_decision(hit)
    return ctx


def _triangles(case):
    kind, size = case.get("scene"), case.get("size")
    if kind == "box":
        return 36
    if kind == "terrain":
        return 2 * (size - 1) ** 2
    if kind == "sphere":
        return 40 * 4 ** size + 2 * 4 ** (size + 2)
    return size


def _camera(sd, rng):
    """The scene's view, moved a little."""
    c = api.Camera.from_buffer_copy(sd.desc.camera)
    c.yaw += float(rng.uniform(-2.0, 2.0))
    c.pitch += float(rng.uniform(-1.0, 1.0))
    for k in range(3):
        c.position[k] += float(rng.uniform(-0.01, 0.01))
    return c


def _settings(sd, case, rng):
    cfg = api.RenderCfg.from_buffer_copy(sd.desc.cfg)
    cfg.width, cfg.height, cfg.spp = case["width"], case["height"], case["spp"]
    cfg.max_path_length = case.get("depth", cfg.max_path_length)
    cfg.frame, cfg.seed = 0, int(rng.integers(1 << 40))
    cfg.sampler = {"jittered": api.RC_SAMPLER_JITTERED, "random": api.RC_SAMPLER_RANDOM,
                   "cmj": api.RC_SAMPLER_CMJ}[case.get("sampler", "jittered")]
    cfg.filter, cfg.filter_radius = {"box": (api.RC_FILTER_BOX, 0.5), "tent": (api.RC_FILTER_TENT, 1.0),
                                     "gaussian": (api.RC_FILTER_GAUSSIAN, 0.5),
                                     "bell": (api.RC_FILTER_BELL, 1.5)}[case.get("filter", "box")]
    if cfg.filter == api.RC_FILTER_GAUSSIAN:
        cfg.filter_param[0] = 0.4
    return cfg


def _rays(sd, case, rng):
    """(n, 8) float32 rays as rc_ray: origin, tmin, direction, tmax."""
    n, v = case["n"], sd.vertices.reshape(-1, 3, 3)
    out = np.empty((n, 8), np.float32)
    if case["op"] == "any_device":  # point pairs within the scene's bounds
        lo, hi = v.min(axis=(0, 1)).astype(np.float64), v.max(axis=(0, 1)).astype(np.float64)
        a, b = (lo + rng.random((n, 3)) * (hi - lo) for _ in range(2))
        d = b - a
        dist = np.linalg.norm(d, axis=1)
        out[:, 0:3], out[:, 3], out[:, 4:7], out[:, 7] = a, 1e-4, d / dist[:, None], dist
        return out
    # leaving random points of the surface in random directions of the
    # hemisphere around the normal
    t = v[rng.integers(len(v), size=n)].astype(np.float64)
    r = np.sqrt(rng.random((n, 1)))
    s = rng.random((n, 1))
    p = (1 - r) * t[:, 0] + r * (1 - s) * t[:, 1] + r * s * t[:, 2]
    nrm = np.cross(t[:, 1] - t[:, 0], t[:, 2] - t[:, 0])
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    d = rng.normal(size=(n, 3))
    d = d / np.linalg.norm(d, axis=1, keepdims=True) + nrm
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    out[:, 0:3], out[:, 3], out[:, 4:7], out[:, 7] = p + 1e-4 * d, 0.0, d, np.inf
    return out


# ------------------------------------------------------------------ cache inputs
def _cache_inputs(n, seed):
    """Weights (FP32 masters), queries and target radiances of a cache over the unit box."""
    rng = np.random.default_rng(seed)
    p = []
    for l, (fi, fo) in enumerate(CACHE_FAN):
        lim = math.sqrt(6.0 / fi) * (0.5 if l == 4 else 1.0)
        p += [rng.uniform(-lim, lim, fi * fo), rng.uniform(-0.1, 0.1, fo)]
    q = np.empty((n, 12))
    q[:, :3] = rng.random((n, 3))
    for k in (3, 6):
        u = rng.normal(size=(n, 3))
        q[:, k:k + 3] = u / np.linalg.norm(u, axis=1, keepdims=True)
    q[:, 9:] = rng.uniform(0.2, 0.9, (n, 3))
    base = 0.3 + 0.25 * np.sin(2 * np.pi * q[:, 0]) * np.cos(np.pi * q[:, 2]) + 0.2 * q[:, 1]
    t = base[:, None] * (0.2 + q[:, 9:]) * np.exp(0.3 * rng.normal(size=(n, 3)))
    return np.concatenate(p).astype(np.float32), q.astype(np.float32), t.astype(np.float32)


# ------------------------------------------------------------------ prepare and run
class _State:
    """What the program holds; its handles are closed with it."""

    def __init__(self, **kw):
        self.handles = []
        self.__dict__.update(kw)

    def own(self, h):
        self.handles.append(h)
        return h

    def __del__(self):
        for h in reversed(self.handles):
            h.close()


def prepare(case, seed):
    op = case["op"]
    rng = np.random.default_rng([seed, 17])
    ctx = _context(case.get("hit", "fp32"))
    s = _State(op=op, ctx=ctx)
    if op == "gradient":
        p, s.queries, s.targets = _cache_inputs(case["n"], seed)
        s.cache = s.own(api.RadianceCache(ctx, (0.0, 0.0, 0.0), (1.0, 1.0, 1.0), max_batch=65536))
        s.cache.set_params(p)
        return s
    if op == "batch":
        s.scenes, s.films, s.cams, s.cfgs = [], [], [], []
        for k in range(case["count"]):
            tris = (2000, 20000, 60000, 200000)[k % 4]
            side = (128, 256, 384, 512)[(k + k // 4) % 4]
            sd, nodes, ordered = _asset("soup", tris, 11 + k)
            s.scenes.append(s.own(ctx.upload(sd, nodes, ordered)))
            s.films.append(s.own(ctx.film(side, side)))
            s.cams.append(_camera(sd, rng))
            s.cfgs.append(_settings(sd, {"width": side, "height": side, "spp": case["spp"], "sampler": "random"}, rng))
        s.plans = [api.BatchPlan(case["spp"], 256, 128, 0)] * case["count"]
        s.branches = case["branches"]
        return s
    sd, nodes, ordered = _scene(case["scene"], case["size"], seed)
    s.scene = s.own(ctx.upload(sd, nodes, ordered))
    if op == "closest_host":
        s.rays = _rays(sd, case, rng).view(api.RAY_DTYPE).reshape(-1)
    elif op in ("closest_device", "any_device"):
        s.rays = torch.from_numpy(_rays(sd, case, rng)).cuda()
        s.n = case["n"]
        s.out = (torch.empty((s.n, 4), dtype=torch.float32, device="cuda") if op == "closest_device"
                 else torch.empty(s.n, dtype=torch.uint8, device="cuda"))
        torch.cuda.synchronize()
    elif op == "phong":
        s.cam, s.w, s.h = _camera(sd, rng), case["width"], case["height"]
        s.seed, s.offset, s.light = int(rng.integers(1 << 40)), sd.desc.cfg.ray_start_offset, sd.desc.light
        n = s.w * s.h
        s.out = [torch.empty(shape, dtype=dt, pin_memory=True).numpy() for shape, dt in
                 (((n,), torch.int32), ((n,), torch.float32), ((n, 4), torch.float32))]
    else:
        s.cam, s.cfg = _camera(sd, rng), _settings(sd, case, rng)
        s.film = s.own(ctx.film(s.cfg.width, s.cfg.height))
        if op == "cached":
            s.cfg.cache_vertex = case["vertex"]
            v = sd.vertices.reshape(-1, 3)
            s.cache = s.own(api.RadianceCache(ctx, v.min(axis=0), v.max(axis=0), train_stride=1024))
            s.cache.set_params(_cache_inputs(1, seed)[0])
        elif op == "whitted":
            L = sd.desc.light
            area = dict(area_light=1, area_n=case["area"], area_radius=0.2) if case["area"] else {}
            s.lights = [api.light(api.RC_LIGHT_POINT, position=tuple(L.position), intensity=L.intensity,
                                  max_distance=L.max_distance, attenuation=L.attenuation, **area)]
            ao = dict(ao_enabled=1, ao_n=case["ao"], ao_max_distance=0.3) if case["ao"] else {}
            fog = dict(fog_enabled=1, fog_distance=8.0, fog_color=(0.6, 0.6, 0.7)) if case["glossy"] else {}
            s.settings = api.ray_settings(max_ray_iterations=2 if case["glossy"] else 3, ambient_intensity=0.1,
                                          **ao, **fog)
            g = dict(refl_n=case["glossy"], refl_glossiness=40.0) if case["glossy"] else {}
            s.materials = api.ray_materials(len(sd.materials), ray_reflectance=0.5, **g)
    return s


def run(s):
    op, ctx = s.op, s.ctx
    if op == "closest_host":
        h = ctx.trace_closest(s.scene, s.rays)
        return {"t": h["t"], "u": h["u"], "v": h["v"], "tri": h["tri"]}
    if op == "closest_device":
        api.check(api.lib().rc_trace_closest_device(ctx.h, s.scene.h, s.rays.data_ptr(), s.n, s.out.data_ptr()))
        ctx.synchronize()  # before another stream reads the hits
        return {"t": s.out[:, 0], "uv": s.out[:, 1:3], "tri": s.out.view(torch.int32)[:, 3]}
    if op == "any_device":
        api.check(api.lib().rc_trace_any_device(ctx.h, s.scene.h, s.rays.data_ptr(), s.n, s.out.data_ptr()))
        ctx.synchronize()
        return s.out
    if op == "phong":
        ids, t, rgba = ctx.raycast_phong(s.scene, s.cam, s.w, s.h, s.seed, s.offset, s.light, out=s.out)
        return {"ids": ids, "t": t, "rgba": rgba}
    if op == "gradient":
        g, loss = s.cache.gradient(s.queries, s.targets)
        return {"grad": g, "loss": np.float32(loss)}
    if op == "batch":
        for f in s.films:
            f.clear()
        ctx.render_batch_tuned(s.scenes, s.films, s.cams, s.cfgs, s.plans, s.branches)
        return [f.linear() for f in s.films]
    s.film.clear()
    if op == "whitted":
        ctx.raytrace(s.scene, s.film, s.cam, s.cfg, s.settings, s.materials, s.lights)
    elif op == "cached":
        s.cache.render(s.scene, s.film, s.cam, s.cfg, train=0, want_loss=False)
        return s.film.linear()
    else:
        ctx.render(s.scene, s.film, s.cam, s.cfg)
    return s.film.tonemap()[0]


# ------------------------------------------------------------------ work and exact results
def work(case):
    """The scene and inputs read once, the outputs written once; per ray a
    descent of a 4-wide tree (18 operations per child box) and two triangle
    tests (46 operations).  Rays per sample: the camera's and one more, each
    with a shadow ray where there is a light."""
    op = case["op"]
    if op == "gradient":
        return {"bytes": case["n"] * 60 + 2 * 17923 * 4, "flops": case["n"] * 95616}
    if op == "batch":
        w = [work({"op": "render", "scene": "soup", "size": (2000, 20000, 60000, 200000)[k % 4],
                   "width": (128, 256, 384, 512)[(k + k // 4) % 4], "height": (128, 256, 384, 512)[(k + k // 4) % 4],
                   "spp": case["spp"]}) for k in range(case["count"])]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    tris = _triangles(case)
    per_ray = 72 * max(1.0, math.log(tris / 2, 4)) + 92
    if op in ("closest_host", "closest_device", "any_device"):
        n = case["n"]
        return {"bytes": n * (32 + (1 if op == "any_device" else 16)) + min(tris, 8 * n) * 61, "flops": n * per_ray}
    pixels = case["width"] * case["height"]
    if op == "phong":
        return {"bytes": min(tris, 8 * pixels) * 77 + pixels * 24, "flops": pixels * 2 * per_ray}
    samples = pixels * case["spp"]
    if op == "whitted":
        nodes = 1 + max(1, case["glossy"] ** 2)
        rays = samples * nodes * (1 + max(1, case["area"] ** 2) + case["ao"] ** 2)
    else:
        rays = samples * (2 if case["scene"] == "box" else 4)
    flops = rays * per_ray
    if op == "cached":
        flops += samples * 0.3 * 35328
    return {"bytes": min(tris, 8 * samples) * 77 + pixels * 16, "flops": flops}


def _exact_hits(case, seed):
    """Closest hits by testing every triangle (Moeller-Trumbore) in 64 bits."""
    rng = np.random.default_rng([seed, 17])
    sd = _scene(case["scene"], case["size"], seed)[0]
    r = _rays(sd, case, rng).astype(np.float64)
    v = sd.vertices.astype(np.float64).reshape(-1, 3, 3)
    o, d = r[:, None, 0:3], r[:, None, 4:7]
    e1, e2 = (v[:, 1] - v[:, 0])[None], (v[:, 2] - v[:, 0])[None]
    with np.errstate(divide="ignore", invalid="ignore"):
        pv = np.cross(d, e2)
        det = (e1 * pv).sum(-1)
        tv = o - v[None, :, 0]
        u = (tv * pv).sum(-1) / det
        qv = np.cross(tv, e1)
        w = (d * qv).sum(-1) / det
        t = (e2 * qv).sum(-1) / det
        ok = (det != 0) & (u >= 0) & (w >= 0) & (u + w <= 1) & (t >= r[:, None, 3]) & (t <= r[:, None, 7])
    t = np.where(ok, t, np.inf)
    i = t.argmin(1)
    at = np.arange(len(i))
    hit = np.isfinite(t[at, i])
    return {"t": t[at, i], "u": np.where(hit, u[at, i], 0.0), "v": np.where(hit, w[at, i], 0.0), "tri": None}


def _exact_gradient(case, seed):
    """The cache's loss gradient in 64 bits (automatic differentiation)."""
    p, q, tgt = (torch.from_numpy(a).double().cuda() for a in _cache_inputs(case["n"], seed))
    p.requires_grad_(True)
    x = []
    for a in range(3):
        for f in range(12):
            arg = math.pi * 2.0 ** f * q[:, a]
            x += [torch.sin(arg), torch.cos(arg)]
    h = torch.cat([torch.stack(x, 1), q[:, 3:]], 1)
    at = 0
    for l, (fi, fo) in enumerate(CACHE_FAN):
        w, b = p[at:at + fi * fo].reshape(fo, fi), p[at + fi * fo:at + fi * fo + fo]
        at += fi * fo + fo
        h = h @ w.T + b
        h = torch.relu(h) if l < 4 else torch.exp(h)
    loss = ((h - tgt) ** 2 / (h.detach() ** 2 + 1e-2)).mean()
    loss.backward()
    return {"grad": p.grad, "loss": loss.detach()}


def exact(case, seed):
    if case["op"] == "gradient":
        return _exact_gradient(case, seed)
    if case["op"] == "closest_host" and case["n"] * _triangles(case) <= 1 << 22:
        return _exact_hits(case, seed)
    # A traced image or the hits of millions of rays among millions of
    # triangles take far longer than a pass in 64 bits.
    return None
