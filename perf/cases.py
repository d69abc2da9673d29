"""The work this path tracer is timed on, through its public entry points.

A case is a dict of plain values. `kind` says which entry points a pass takes:

    frame    WavefrontPathTracer.render of one image (or its tone-mapped
             readback): scenes "room" (34 triangles, Lambert), "field" (256
             triangles per Disney sphere), "sky" (the field under an image-based
             light), "media" (the room around a density grid), "fog" (the room
             with a homogeneous medium and volume primitives)
    views    several cameras of a textured two-level field in one wavefront
    cache    progressive 1 spp frames with the radiance cache trained from scratch
    animate  new vertices for the field's geometry, tree refitted, one frame
    rays     ray batches: hits into device memory, or closest hits and
             visibility of host arrays
    network  the cache's network by itself: inference and loss gradients

Sizes are those of the benchmark and of the GPU tests, and the odd ones
between them.
"""
import functools
import math
import random

import numpy as np
import torch

import btrc_amd
from btrc_amd import _abi, scenes

FIELD = 4096          # instances of the benchmark's field, in a box of 100^3
ROOM_TRIANGLES = 34
SPHERE_TRIANGLES = 256
RAY_RANGE = 1000.0    # tmax of ray batches: beyond every scene's far side
MAX_PATHS = 1920 * 1080 * 16   # a drawn frame's largest path count


def listed():
    return [
        # an interactive preview of a small scene: one sample per pixel,
        # tone-mapped for the screen; launches and read-backs count
        dict(name="preview_320x180", kind="frame", scene="room", width=320, height=180, spp=1, depth=8,
             states=1000000, sampler="halton", filter="box", readback="tonemap"),
        # the reference's smallest full render: room, 256^2, 16 spp
        dict(name="room_256_16spp", kind="frame", scene="room", width=256, height=256, spp=16, depth=8,
             states=1 << 20, sampler="halton", filter="box", readback="film"),
        # the headline frame's scene, size and pool, at half its samples
        dict(name="field_1080p_32spp", kind="frame", scene="field", instances=FIELD, width=1920, height=1080, spp=32,
             depth=8, states=1 << 25, sampler="halton", filter="box", readback="film"),
        # a still with every output: image-based light, the reference's own
        # sampler and default pool, Gaussian filter, albedo and normal
        # images, FP64 film, tile order, a size no tile divides
        dict(name="sky_1003x565_all_outputs", kind="frame", scene="sky", instances=1024, width=1003, height=565, spp=4,
             depth=10, states=1000000, sampler="independent", filter="gaussian", readback="all"),
        # the participating-media workload at a preview's samples: 128^3
        # density grid, delta and ratio tracking, depth 16
        dict(name="media_1080p_4spp", kind="frame", scene="media", grid=128, width=1920, height=1080, spp=4,
             depth=16, states=1 << 23, sampler="halton", filter="box", readback="film"),
        # homogeneous medium and overlapping volume primitives
        dict(name="fog_640x360_8spp", kind="frame", scene="fog", grid=32, width=640, height=360, spp=8, depth=10,
             states=1 << 20, sampler="halton", filter="box", readback="film"),
        # the batched workload: uneven views of a textured instanced scene in
        # one wavefront
        dict(name="views_4_textured_two_level", kind="views", instances=8192, texture=512, views=4, spp=2, depth=8,
             states=1 << 22),
        # the radiance cache from a new scene's first frame on
        dict(name="cache_256_8frames", kind="cache", width=256, height=256, frames=8, steps=4, train_depth=2,
             states=1 << 17),
        # an animated scene: vertices replaced, tree refitted, 1 spp frame
        dict(name="animate_720p", kind="animate", instances=FIELD, width=1280, height=720, spp=1, depth=8,
             states=1 << 20),
        # a device-resident batch of incoherent rays against a million triangles
        dict(name="rays_device_1m", kind="rays", instances=FIELD, rays=(1 << 20) + 77, memory="device"),
        # queries of a host program: closest hits and visibility, host arrays
        dict(name="rays_host_40k", kind="rays", instances=256, rays=40003, memory="host"),
        # the cache's network: 100,003 predictions, gradients of 16,384 samples
        dict(name="network_100k", kind="network", queries=100003, samples=16384),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_frame(rng, scene):
    w = _log_int(rng, 96, 1920)
    h = max(64, int(w * rng.choice([9 / 16, 2 / 3, 0.75, 1.0]) * rng.uniform(0.9, 1.0)))
    limit = {"room": MAX_PATHS // 2, "field": MAX_PATHS, "sky": MAX_PATHS // 4, "media": 1920 * 1080 * 2,
             "fog": 1920 * 1080 * 2}[scene]
    spp = max(1, min(_log_int(rng, 1, 64), limit // (w * h)))
    c = dict(kind="frame", scene=scene, width=w, height=h, spp=spp, depth=rng.randint(3, 16),
             states=rng.choice([1 << 18, 1000000, 1 << 20, 1 << 22, 1 << 23]),
             sampler="halton" if rng.random() < 0.75 else "independent",
             filter="box" if rng.random() < 0.75 else "gaussian", readback=rng.choice(["film", "film", "tonemap", "all"]))
    if scene in ("field", "sky"):
        c["instances"] = _log_int(rng, 64, FIELD)
    if scene in ("media", "fog"):
        c["grid"] = rng.choice([24, 32, 50, 64, 128])
    return c


def draw(rng):
    kind = rng.choice(["room", "room", "field", "field", "field", "sky", "media", "media", "fog", "views", "cache",
                       "animate", "rays", "rays", "network"])
    if kind in ("room", "field", "sky", "media", "fog"):
        return _draw_frame(rng, kind)
    if kind == "views":
        return dict(kind="views", instances=_log_int(rng, 512, 8192), texture=rng.choice([128, 256, 512]),
                    views=rng.randint(2, 6), spp=rng.randint(1, 2), depth=rng.randint(4, 10), states=1 << 22)
    if kind == "cache":
        w = _log_int(rng, 128, 512)
        return dict(kind="cache", width=w, height=max(64, int(w * rng.uniform(0.6, 1.0))), frames=rng.randint(2, 12),
                    steps=rng.randint(1, 4), train_depth=rng.choice([0, 2, 3]), states=1 << 18)
    if kind == "animate":
        w = _log_int(rng, 160, 1280)
        return dict(kind="animate", instances=_log_int(rng, 128, FIELD), width=w, height=max(90, w * 9 // 16),
                    spp=rng.randint(1, 2), depth=rng.randint(4, 10), states=1 << 20)
    if kind == "rays":
        memory = rng.choice(["device", "host"])
        return dict(kind="rays", instances=_log_int(rng, 16, FIELD), memory=memory,
                    rays=_log_int(rng, 100, (4 << 20) if memory == "device" else 400000))
    return dict(kind="network", queries=_log_int(rng, 500, 400000), samples=_log_int(rng, 500, 65536))


# ------------------------------------------------------------------ scenes


@functools.lru_cache(maxsize=None)
def _grid(n):
    return scenes.fbm_grid(n, seed=3, max_sigma=2.0)


@functools.lru_cache(maxsize=None)
def _noise(n, seed):
    return scenes.noise_texture(n, seed=seed)


def _extent(instances):
    return 100.0 * (instances / FIELD) ** (1.0 / 3.0)


def _field(instances, seed):
    return scenes.sphere_field(instances=instances, lights=max(4, instances // 64), seed=seed,
                               extent=_extent(instances))


def _textured_field(instances, texture, seed):
    """the textured two-level field of the batched workload at a smaller
    instance count and the same density, its textures made once"""
    s, _ = scenes.sphere_field(instances=instances, lights=64, seed=seed, extent=250.0 * (instances / 65536) ** (1 / 3))
    s.accel = _abi.ACCEL_TWO_LEVEL
    rng = scenes.PCG32(seed)
    uvs = scenes.uv_sphere_uvs()
    first = len(s.geometries)
    for _ in range(4):
        s.add_geometry(scenes.uv_sphere(rng, displacement=0.15), uvs=uvs)
    tex = [s.add_texture(_noise(texture, 200 + k), address_u="wrap") for k in range(8)]
    for k, inst in enumerate(s.instances):
        if inst["light"] is None:
            inst["geometry"] = first + k % 4
            m = s.materials[inst["material"]]
            m["color"], m["color_texture"] = (1.0, 1.0, 1.0), tex[k % 8]
    return s


def _fog(n):
    s, cam = scenes.cornell()
    haze = s.add_homogeneous(0.8, (0.9, 0.85, 0.8), g=0.3)
    box = np.concatenate(scenes.box_faces(0.8, 0.8, 0.8))
    s.add_instance(s.add_geometry(box), s.add_invisible(), scenes.translate(0.35, 1.2, 0.2), inner_medium=haze)
    s.add_volume((-0.9, 0.05, -0.9), (1.8, 0, 0), (0, 0.9, 0), (0, 0, 1.8), 0.5 * _grid(n), (0.9, 0.9, 0.9))
    s.add_volume((-0.5, 0.4, -0.5), (0.9, 0.2, 0), (-0.2, 0.9, 0), (0, 0, 0.9), 0.7, (0.8, 0.6, 0.4))
    return s, cam


def _scene(case, rng):
    """the case's scene and camera, the camera moved a little by the seed"""
    kind = case["scene"]
    if kind == "room":
        s, cam = scenes.cornell(seed=rng.randrange(1, 1 << 20))
    elif kind in ("field", "sky"):
        s, cam = _field(case["instances"], rng.randrange(1, 1 << 20))
        if kind == "sky":
            s.set_ibl(s.add_texture(scenes.sky_texture(512, 256, seed=rng.randrange(1 << 20)), address_u="wrap"),
                      up=(0.0, 1.0, 0.0))
    elif kind == "media":
        s, cam = scenes.cornell_media(grid=_grid(case["grid"]))
    else:
        s, cam = _fog(case["grid"])
    size = abs(cam.eye[2] - cam.dst[2])
    cam.eye = tuple(float(e) + 0.03 * size * rng.uniform(-1.0, 1.0) for e in cam.eye)
    return s, cam


# ------------------------------------------------------------------ states


def _params(case, **more):
    p = _abi.RenderParams()
    p.spp, p.min_depth, p.max_depth = case.get("spp", 1), 3, case.get("depth", 8)
    p.rr_threshold, p.rr_cont_prob = 0.1, 0.5
    p.state_count = case["states"]
    for k, v in more.items():
        setattr(p, k, v)
    return p


def _prepare_frame(case, rng):
    s, cam = _scene(case, rng)
    every = case["readback"] == "all"
    r = btrc_amd.WavefrontPathTracer(spp=case["spp"], min_depth=3, max_depth=case["depth"],
                                     state_count=case["states"], sampler=case["sampler"], tile=every, albedo=every,
                                     normal=every, film_fp64=every)
    r.set_scene(s)
    r.set_camera(cam)
    r.set_film(case["width"], case["height"])
    r.set_film_filter(case["filter"])
    r.commit()
    return dict(renderer=r)


def _run_frame(case, st):
    r = st["renderer"]
    if case["readback"] == "tonemap":
        stats = r.ctx.render(r.render_params())
        out = dict(image=r.ctx.tonemapped(r.width, r.height))
    else:
        res = r.render()
        stats = res.stats
        out = dict(image=res.color)
        if case["readback"] == "all":
            out.update(image64=res.color64, albedo=res.albedo, normal=res.normal)
    out.update(rays=stats.extension_rays, shadow_rays=stats.shadow_rays)
    return out


VIEW_SIZES = [(512, 512), (640, 480), (801, 600), (1280, 720), (333, 1024), (1600, 900)]


def _prepare_views(case, rng):
    ctx = btrc_amd.Context()
    s = _textured_field(case["instances"], case["texture"], rng.randrange(1, 1 << 20))
    ctx.upload_scene(s)
    e = 250.0 * (case["instances"] / 65536) ** (1 / 3)
    c, turn = e / 2, rng.uniform(0.0, 2.0 * math.pi)
    views = []
    for k, (w, h) in enumerate(VIEW_SIZES[:case["views"]]):
        a = turn + 2.0 * math.pi * k / case["views"]
        eye = (c + 0.8 * e * math.cos(a), c + 0.1 * e * (k % 3 - 1), c + 0.8 * e * math.sin(a))
        views.append((scenes.Camera(eye, (c, c, c), (0.0, 1.0, 0.0), 60.0), w, h))
    return dict(ctx=ctx, views=views, params=_params(case))


def _run_views(case, st):
    stats = st["ctx"].render_views(st["params"], st["views"])
    return dict(images=[st["ctx"].view_film(k, w, h) for k, (_, w, h) in enumerate(st["views"])],
                rays=stats.extension_rays, shadow_rays=stats.shadow_rays)


def _prepare_cache(case, rng):
    ctx = btrc_amd.Context()
    s, cam = _scene(dict(scene="room"), rng)
    ctx.upload_scene(s)
    ctx.set_camera(cam, case["width"], case["height"])
    ctx.nrc_configure(enabled=1, train=1, train_depth=case["train_depth"], steps=case["steps"], train_stride=16,
                      query_depth=2)
    return dict(ctx=ctx, seed=rng.randrange(1, 1 << 20))


def _run_cache(case, st):
    # a new scene on the screen: fresh weights, frames accumulated while the
    # cache learns, then the image
    ctx = st["ctx"]
    ctx.nrc_reset(st["seed"])
    rays = 0
    for f in range(case["frames"]):
        p = _params(case, width=case["width"], height=case["height"], sample_offset=f, accumulate=1 if f else 0)
        stats = ctx.render(p)
        rays += stats.extension_rays + stats.shadow_rays
    return dict(image=ctx.film(case["width"], case["height"])[0], weights=ctx.nrc_weights(), rays=rays)


def _prepare_animate(case, rng):
    ctx = btrc_amd.Context()
    s, cam = _field(case["instances"], rng.randrange(1, 1 << 20))
    s.accel = _abi.ACCEL_FLAT_GPU
    ctx.upload_scene(s)
    ctx.set_camera(cam, case["width"], case["height"])
    # the next animation frame's vertices: the sphere stretched and twisted
    p = s.geometries[0]["positions"].reshape(-1, 3).astype(np.float64)
    a = rng.uniform(0.2, 0.6) * p[:, 1]
    y = p[:, 1] * rng.uniform(0.8, 1.25)
    q = np.stack([p[:, 0] * np.cos(a) - p[:, 2] * np.sin(a), y, p[:, 0] * np.sin(a) + p[:, 2] * np.cos(a)], axis=1)
    s.geometries[0]["positions"][...] = q.reshape(-1, 9).astype(np.float32)
    return dict(ctx=ctx, scene=s, params=_params(case, width=case["width"], height=case["height"]))


def _run_animate(case, st):
    ctx = st["ctx"]
    ctx.update_geometry(st["scene"], 0)
    stats = ctx.render(st["params"])
    return dict(image=ctx.film(case["width"], case["height"])[0], rays=stats.extension_rays,
                shadow_rays=stats.shadow_rays)


def _make_rays(case, seed):
    """rays that start anywhere in the scene's box, in any direction"""
    rng = np.random.default_rng(seed)
    n, e = case["rays"], _extent(case["instances"])
    rays = np.zeros(n, dtype=_abi.ray_dtype())
    rays["o"] = rng.random((n, 3), dtype=np.float32) * np.float32(e)
    d = rng.standard_normal((n, 3), dtype=np.float32)
    rays["d"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays["tmax"] = RAY_RANGE
    return rays


def _rays_scene(case, seed):
    return _field(case["instances"], 2 + seed % 1000)[0]


def _prepare_rays(case, seed):
    ctx = btrc_amd.Context()
    ctx.upload_scene(_rays_scene(case, seed))
    rays = _make_rays(case, seed)
    st = dict(ctx=ctx, rays=rays)
    if case["memory"] == "device":
        st["rays"] = torch.from_numpy(rays.view(np.float32).reshape(-1, 8)).cuda()
        st["hits"] = torch.zeros((case["rays"], 5), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
    return st


def _run_rays(case, st):
    ctx = st["ctx"]
    if case["memory"] == "device":
        hits = st["hits"]
        ctx.trace_closest_noalloc(st["rays"].data_ptr(), case["rays"], hits.data_ptr())
        return dict(t=hits[:, 0], triangle=hits.view(torch.int32)[:, 1:3], uv=hits[:, 3:5])
    hits = ctx.trace_closest(st["rays"])
    occluded = ctx.trace_any(st["rays"])
    return dict(t=hits["t"], triangle=np.stack([hits["instance"], hits["prim"]], axis=1).view(np.int32),
                uv=np.stack([hits["u"], hits["v"]], axis=1), occluded=occluded)


def _network_inputs(case, seed):
    """weights (uniform He), vertex records over the room's box, targets"""
    rng = np.random.default_rng(seed)
    w = np.zeros(_abi.NRC_PARAMS, dtype=np.float32)
    w[:5 * 4096 + 3 * 64] = rng.uniform(-1.0, 1.0, 5 * 4096 + 3 * 64) * math.sqrt(6.0 / 64.0)

    def vertices(n):
        v = np.empty((n, 16), dtype=np.float32)
        v[:, 0:3] = rng.random((n, 3)) * 2.0 + np.array([-1.0, 0.0, -1.0])
        for a in (3, 6):
            d = rng.standard_normal((n, 3))
            v[:, a:a + 3] = d / np.linalg.norm(d, axis=1, keepdims=True)
        v[:, 9] = rng.uniform(0.05, 1.0, n)
        v[:, 10:16] = rng.random((n, 6))
        return v

    v, t = vertices(case["queries"]), vertices(case["samples"])
    return w, v, t, rng.uniform(0.0, 2.0, (case["samples"], 3)).astype(np.float32)


def _prepare_network(case, seed):
    ctx = btrc_amd.Context()
    ctx.upload_scene(scenes.cornell()[0])
    w, queries, samples, targets = _network_inputs(case, seed)
    ctx.nrc_set_weights(w)
    return dict(ctx=ctx, queries=queries, samples=samples, targets=targets)


def _run_network(case, st):
    ctx = st["ctx"]
    out = ctx.nrc_eval(st["queries"])
    grad, loss = ctx.nrc_gradients(st["samples"], st["targets"])
    return dict(radiance=out, gradients=grad, loss=loss)


PREPARE = {"frame": _prepare_frame, "views": _prepare_views, "cache": _prepare_cache, "animate": _prepare_animate}
RUN = {"frame": _run_frame, "views": _run_views, "cache": _run_cache, "animate": _run_animate, "rays": _run_rays,
       "network": _run_network}


def prepare(case, seed):
    if case["kind"] == "rays":
        st = _prepare_rays(case, seed)
    elif case["kind"] == "network":
        st = _prepare_network(case, seed)
    else:
        st = PREPARE[case["kind"]](case, random.Random(seed))
    st["case"] = case
    return st


def run(state):
    return RUN[state["case"]["kind"]](state["case"], state)


# ------------------------------------------------------------------ work


def _ray_work(rays, triangles):
    """a ray is read (32 B) and its hit written (20 B); it descends a tree of
    four-box nodes (4 x 14 operations) to one triangle (60 operations)"""
    levels = max(1.0, math.log(max(triangles, 4), 4))
    return rays * 52.0, rays * (levels * 56.0 + 60.0)


def work(case):
    kind = case["kind"]
    if kind == "network":
        # 20,672 weights; forward for the queries; forward, input gradients
        # and weight gradients for the samples
        return dict(bytes=76.0 * (case["queries"] + case["samples"]) + 2 * 4.0 * _abi.NRC_PARAMS,
                    flops=2.0 * 20672 * (case["queries"] + 3 * case["samples"]))
    triangles = case["instances"] * SPHERE_TRIANGLES if "instances" in case else ROOM_TRIANGLES
    if kind == "rays":
        passes = 1 if case["memory"] == "device" else 2
        b, f = _ray_work(case["rays"] * passes, triangles)
        return dict(bytes=b, flops=f)
    if kind == "views":
        pixels = sum(w * h for w, h in VIEW_SIZES[:case["views"]])
    else:
        pixels = case["width"] * case["height"]
    paths = pixels * (case["frames"] if kind == "cache" else case["spp"])
    # vertices per path and shadow rays per vertex: about what these scenes
    # show (paths leave an open field; a room keeps them until roulette; the
    # cache ends them at their third vertex)
    open_scene = kind in ("views", "animate") or case.get("scene") in ("field", "sky")
    depth = 3.0 if kind == "cache" else min(case["depth"] + 1, 3.0 if open_scene else 6.0)
    b, f = _ray_work(paths * depth * 2.0, triangles)
    f += paths * depth * 400.0          # a vertex: surface point, light sample, BSDF, continuation
    if case.get("scene") in ("media", "fog"):
        f += paths * depth * 1000.0     # tracking steps: random numbers, trilinear lookups
        b += 4.0 * case["grid"] ** 3
    if kind == "cache":
        f += 2.0 * 20672 * paths + 6.0 * 20672 * 65536 * case["frames"] * 0.25
    return dict(bytes=b + 16.0 * pixels + 144.0 * triangles, flops=f)


def tolerance(case):
    kind = case["kind"]
    if kind == "rays":
        return "exact"              # a hit is a function of the ray and the triangles alone, bit for bit
    if kind == "network":
        return dict(rel=5e-3)       # BF16 weights and activations, FP32 accumulation
    if kind == "cache":
        return dict(rel=1e-4)       # weights and images after the training steps
    # every number of a path is the same; only the order of the film's FP32
    # atomics differs (5e-9 in the norm, 3e-7 in a pixel between two passes)
    return dict(rel=1e-6, max=1e-5)


# ------------------------------------------------------------------ 64 bits


def _world_triangles(scene):
    tris, ids = [], []
    for k, inst in enumerate(scene.instances):
        p = scene.geometries[inst["geometry"]]["positions"].reshape(-1, 3).astype(np.float32)
        m = inst["mat"].astype(np.float32)
        w = ((m[:, 0] * p[:, :1] + m[:, 1] * p[:, 1:2]) + m[:, 2] * p[:, 2:3]) + m[:, 3]
        tris.append(w[:, :3].reshape(-1, 9))
        ids.append(np.stack([np.full(len(p) // 3, k), np.arange(len(p) // 3)], axis=1))
    return np.concatenate(tris).astype(np.float64), np.concatenate(ids)


def _exact_rays(case, seed):
    """closest hits by testing every triangle (Moeller-Trumbore) in float64"""
    tris, _ = _world_triangles(_rays_scene(case, seed))
    if case["rays"] * len(tris) > 6e9:
        return None
    rays = _make_rays(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    tri = torch.from_numpy(tris).to(dev)
    a, e1, e2 = tri[:, 0:3], tri[:, 3:6] - tri[:, 0:3], tri[:, 6:9] - tri[:, 0:3]
    o = torch.from_numpy(rays["o"].astype(np.float64)).to(dev)
    d = torch.from_numpy(rays["d"].astype(np.float64)).to(dev)
    n = torch.linalg.cross(e1, e2)
    n_a, a_e1, a_e2 = (n * a).sum(1), torch.linalg.cross(a, e1), torch.linalg.cross(a, e2)
    ts, uvs = [], []
    step = max(1, int(4e7 // len(tris)))
    for k in range(0, len(o), step):
        ok, dk = o[k:k + step], d[k:k + step]
        m = torch.linalg.cross(ok, dk)      # the ray as a Pluecker line
        inv = 1.0 / (dk @ n.T)
        t = (n_a - ok @ n.T) * inv
        # weights of vertices b and c
        u = -(m @ e2.T + dk @ a_e2.T) * inv
        v = (m @ e1.T + dk @ a_e1.T) * inv
        hit = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= 0) & (t <= RAY_RANGE)
        t = torch.where(hit, t, torch.full_like(t, math.inf))
        best, at = t.min(dim=1)
        miss = torch.isinf(best)
        row = torch.arange(len(ok), device=dev)
        uv = torch.stack([u[row, at], v[row, at]], dim=1)
        uv[miss] = 0.0
        ts.append(torch.where(miss, torch.full_like(best, RAY_RANGE), best))
        uvs.append(uv)
    t, uv = torch.cat(ts), torch.cat(uvs)
    if case["memory"] == "device":
        return dict(t=t, triangle=None, uv=uv)
    return dict(t=t, triangle=None, uv=uv, occluded=None)


def _encode(v, lo, inv_extent):
    """the network's 64 inputs: eight frequencies of sine and cosine of the
    normalised position, directions and material values, three ones, in the
    order 16 s + 8 h + j of (slice, half, element)"""
    q = (v[:, 0:3] - lo) * inv_extent
    x = torch.empty((len(v), 64), dtype=torch.float64, device=v.device)
    ones = torch.ones((len(v), 3), dtype=torch.float64, device=v.device)
    for h in range(2):
        e = []
        for f in range(4):
            w = 2.0 ** (4 * h + f) * math.pi * q
            e.append(torch.stack([torch.sin(w), torch.cos(w)], dim=2).reshape(len(v), 6))
        e.append(v[:, 3:11] if h == 0 else torch.cat([v[:, 11:16], ones], dim=1))
        e = torch.cat(e, dim=1)
        for s in range(4):
            x[:, 16 * s + 8 * h:16 * s + 8 * h + 8] = e[:, 8 * s:8 * s + 8]
    return x


def _exact_network(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    w, queries, samples, targets = (torch.from_numpy(a).to(dev).double() for a in _network_inputs(case, seed))
    box = torch.from_numpy(scenes.cornell()[0].world_box()).to(dev).double()
    layers = [w[l * 4096:(l + 1) * 4096].reshape(64, 64) for l in range(5)] + [w[5 * 4096:].reshape(32, 64)[:3]]

    def forward(v):
        acts = [_encode(v, box[:3], box[3:])]
        for m in layers[:5]:
            acts.append(torch.relu(acts[-1] @ m.T))
        return acts, acts[-1] @ layers[5].T

    radiance = torch.cat([forward(q)[1] for q in queries.split(1 << 16)])
    acts, y = forward(samples)
    den = y * y + 0.01
    loss = float(((y - targets) ** 2 / den).mean())
    dz = 2.0 * (y - targets) / den / y.numel()
    grad = torch.zeros_like(w)
    for l in range(5, -1, -1):
        g = dz.T @ acts[l]
        grad[l * 4096:l * 4096 + g.numel()] = g.reshape(-1)
        if l:
            dz = (dz @ layers[l]) * (acts[l] > 0)
    return dict(radiance=radiance, gradients=grad, loss=loss)


def exact(case, seed):
    """None for images: a path tracer's 64-bit image is another image, since
    each of its discrete choices follows the rounding"""
    if case["kind"] == "rays":
        return _exact_rays(case, seed)
    if case["kind"] == "network":
        return _exact_network(case, seed)
    return None
