"""Rays where a box test can go wrong, against the oracle's brute force (no
tree), bit for bit: directions with zero, negative-zero and denormal
components, origins on box planes and triangle planes, negative tmin, far
origins, rays along edges; on one-level trees (host and GPU built), on two
levels, and with tie-rich coplanar geometry. Batches around a wavefront's and
a grid's size, and trees deep enough for the overflow stack."""
import numpy as np
import pytest

from btrc_amd import _abi, scenes
from oracle import oracle

from util import assert_hits_equal, random_rays, render_params

pytestmark = pytest.mark.gpu


def lattice_scene(accel, scale=1.0):
    """axis-aligned quads on integer planes (flat boxes, shared edges,
    coplanar duplicates) and a displaced sphere, `scale` times as large"""
    tris = []
    for k in range(4):
        for i in range(3):
            for j in range(3):
                tris.append(scenes.quad((i, j, k), (i + 1, j, k), (i + 1, j + 1, k), (i, j + 1, k)))
                tris.append(scenes.quad((k, i, j), (k, i + 1, j), (k, i + 1, j + 1), (k, i, j + 1)))
                tris.append(scenes.quad((i, k, j), (i, k, j + 1), (i + 1, k, j + 1), (i + 1, k, j)))
    tris = np.concatenate(tris).reshape(-1, 9) * np.float32(scale)
    ball = scenes.uv_sphere(scenes.PCG32(4), displacement=0.2) * np.float32(scale)
    s = scenes.Scene()
    m = s.add_diffuse([0.5, 0.5, 0.5])
    s.add_instance(s.add_geometry(tris), m)
    s.add_instance(s.add_geometry(tris[::3].copy()), m)          # ties
    s.add_instance(s.add_geometry(ball), m, np.eye(4))
    s.accel = accel
    return s


def edge_rays(n, seed):
    rng = np.random.default_rng(seed)
    rays = np.zeros(n, dtype=_abi.ray_dtype())
    o = rng.integers(-2, 10, (n, 3)).astype(np.float32) * np.float32(0.5)
    o += rng.choice([0.0, 0.0, 1e-6, 0.25], (n, 3)).astype(np.float32)
    d = rng.choice([0.0, -0.0, 1.0, -1.0, 0.5, 1e-30, -1e-38, 1e-42, 3.0], (n, 3)).astype(np.float32)
    dead = (np.abs(d) < 1e-20).all(axis=1)
    d[dead, 0] = 1.0
    far = rng.random(n) < 0.1
    o[far] *= np.float32(1e5)
    aim = rng.random((n, 3)).astype(np.float32) * 3
    d[far] = aim[far] - o[far]
    rays["o"], rays["d"] = o, d
    rays["tmin"] = rng.choice([0.0, 0.0, -5.0, 0.5], n).astype(np.float32)
    rays["tmax"] = rng.choice([3.4028234663852886e38, 2.0, 1.0, 0.0], n).astype(np.float32)
    return rays


@pytest.mark.parametrize("accel", [_abi.ACCEL_FLAT, _abi.ACCEL_FLAT_GPU, _abi.ACCEL_TWO_LEVEL])
@pytest.mark.parametrize("mode", [_abi.TRI_WATERTIGHT, _abi.TRI_MOLLER_TRUMBORE])
def test_edge_rays_equal_brute_force(ctx, accel, mode):
    scene = lattice_scene(accel)
    ctx.upload_scene(scene)
    ref = oracle.OracleScene(scene)
    rays = edge_rays(20011, 5)
    got, want = ctx.trace_closest(rays, mode), ref.trace(rays, mode, use_bvh=False)
    if mode == _abi.TRI_WATERTIGHT:
        assert_hits_equal(got, want)
    else:
        # Moeller-Trumbore's barycentrics are off by a few 2^-24 of one, so a
        # ray along a shared edge may count as inside a triangle whose box it
        # misses by that much: the neighbour's hit. Both distances carry a few
        # roundings (2^-24 each) of the origin's distance to the vertices, here
        # up to 6
        assert np.array_equal(got["instance"] == 0xffffffff, want["instance"] == 0xffffffff)
        np.testing.assert_allclose(got["t"], want["t"], rtol=4 * 2.0 ** -24, atol=4 * 6 * 2.0 ** -24)
        same = (got["instance"] == want["instance"]) & (got["prim"] == want["prim"])
        assert same.mean() > 0.99
    assert np.array_equal(ctx.trace_any(rays, mode), ref.trace(rays, mode, any_hit=True, use_bvh=False))


@pytest.mark.parametrize("accel", [_abi.ACCEL_FLAT, _abi.ACCEL_TWO_LEVEL])
@pytest.mark.parametrize("scale,length", [(2.0 ** 20, 1.0), (2.0 ** 31, 1.0), (1.0, 2.0 ** -60), (1.0, 2.0 ** -97),
                                          (2.0 ** -20, 2.0 ** -110), (1.0, 2.0 ** 60)])
def test_any_magnitude_equals_brute_force(ctx, accel, scale, length):
    """scenes of large extent (origins beyond 2^32, rays that run inside a
    box's face for millions of units) and rays far from unit length; zero,
    negative-zero and very small components among the directions"""
    scene = lattice_scene(accel, scale)
    ctx.upload_scene(scene)
    rng = np.random.default_rng(17)
    n = 6000
    rays = np.zeros(n, dtype=_abi.ray_dtype())
    rays["o"] = rng.integers(-2, 10, (n, 3)).astype(np.float32) * np.float32(0.5 * scale)
    d = rng.choice([0.0, -0.0, 1.0, -1.0, 0.5, 2.0 ** -25, 3.0], (n, 3)).astype(np.float32)
    d[(d == 0).all(axis=1), 0] = 1.0
    rays["d"] = d * np.float32(length)
    rays["tmax"] = np.float32(3.4028234663852886e38)
    ref = oracle.OracleScene(scene)
    got, want = ctx.trace_closest(rays), ref.trace(rays, use_bvh=False)
    assert 0.1 < (want["instance"] != 0xffffffff).mean() < 0.95
    if length == 1.0:
        assert_hits_equal(got, want)
    else:
        # the culling margin is a distance along a ray of unit length: a
        # shorter ray may keep the other of two hits a few roundings (2^-24 of
        # a vertex' distance, up to 6 units) apart
        assert np.array_equal(got["instance"] == 0xffffffff, want["instance"] == 0xffffffff)
        np.testing.assert_allclose(got["t"].astype(np.float64) * length, want["t"].astype(np.float64) * length,
                                   rtol=4 * 2.0 ** -24, atol=4 * 6 * scale * 2.0 ** -24)
    assert np.array_equal(ctx.trace_any(rays), ref.trace(rays, any_hit=True, use_bvh=False))


# around a wavefront, and around the rays that are handed out by workgroup index:
# 20 (visibility) and 24 (closest hit) wavefronts on each of 256 CUs
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000] + [w * 256 * 64 + k for w in (20, 24) for k in (-1, 0, 1)])
def test_batch_sizes(ctx, n):
    assert ctx.get_tuning()["trace_waves_per_cu"] == 24
    scene = scenes.sphere_field(instances=64, lights=2, seed=9, extent=12.0)[0]
    ctx.upload_scene(scene)
    rays = random_rays(n, 0.0, 12.0, n)
    want = oracle.OracleScene(scene).trace(rays)
    assert_hits_equal(ctx.trace_closest(rays), want)
    assert np.array_equal(ctx.trace_any(rays), want["instance"] != 0xffffffff)


def slab_scene():
    """a fan of nested, overlapping slabs: every box holds every ray, so the
    stack grows past its LDS part in every lane"""
    rng = np.random.default_rng(3)
    n = 6000
    c = rng.uniform(-1, 1, (n, 1, 3)) * np.array([40.0, 0.01, 40.0])
    tris = (c + rng.uniform(-1, 1, (n, 3, 3)) * np.array([30.0, 0.5, 30.0])).astype(np.float32).reshape(n, 9)
    s = scenes.Scene()
    s.add_instance(s.add_geometry(tris), s.add_diffuse([0.5, 0.5, 0.5]))
    return s


def test_deep_stacks(ctx):
    s = slab_scene()
    ctx.upload_scene(s)
    assert ctx.scene_info()["stack"] > 16
    rays = random_rays(3000, [-40, -1, -40], [40, 1, 40], 8)
    rays["d"][:, 1] *= np.float32(0.01)
    want = oracle.OracleScene(s).trace(rays, use_bvh=False)
    assert_hits_equal(ctx.trace_closest(rays), want)
    assert np.array_equal(ctx.trace_any(rays), want["instance"] != 0xffffffff)


@pytest.mark.parametrize("w,h", [(1024, 1024), (250, 131)])  # on two streams, in one launch
def test_shadow_and_extension_rays_keep_their_deep_stacks_apart(ctx, w, h):
    """a bounce's shadow rays are traced beside the next bounce's extension
    rays: with both past the LDS part of their stacks, the frame equals the
    one whose launches run one by one"""
    s = slab_scene()
    s.add_instance(0, 0, scenes.translate(0.0, 4.0, 0.0))   # bounces go on between the two
    s.set_gradient_sky((0.0, 1.0, 0.0), (0.1, 0.2, 0.3), (0.6, 0.5, 0.4))
    ctx.upload_scene(s)
    assert ctx.scene_info()["stack"] > 16
    ctx.set_camera(scenes.Camera((30.0, 2.0, 0.0), (0.0, 2.0, 5.0), (0.0, 1.0, 0.0), 60.0), w, h)
    got = []
    for graph in (1, 0):
        ctx.set_tuning(launch_graph=graph)
        st = ctx.render(render_params(w, h, 1, max_depth=6, state_count=1 << 20, film_fp64=1))
        got.append((st.extension_rays, st.shadow_rays, ctx.film(w, h, fp64=True)[1]))
    (ea, sa, a), (eb, sb, b) = got
    assert ea == eb > 1.5 * w * h and sa == sb > 0.3 * w * h
    assert np.abs(a - b).max() <= 1e-12 * max(1.0, np.abs(b).max())
