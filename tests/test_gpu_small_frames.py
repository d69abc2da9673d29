"""Frames whose launches do not fill the GPU: one captured block when every
path fits the pool (odd and even numbers of bounces, the longest block and the
first frame past it), blocks of four otherwise, extension and shadow rays in
one launch. Films (FP64) and ray counts equal the direct launches', whose
stages run one by one; pools equal to the paths, one smaller, and tiny ones;
one level, two levels, media, and the cache's early ends."""
import numpy as np
import pytest

from btrc_amd import _abi, scenes

from util import render_params

pytestmark = pytest.mark.gpu

W, H, SPP = 60, 41, 2
PATHS = W * H * SPP


def scene_of(kind):
    if kind == "media":
        return scenes.cornell_media(grid=scenes.fbm_grid(12, octaves=3, seed=3, max_sigma=0.3))
    scene, cam = scenes.cornell() if kind == "room" else scenes.sphere_field(instances=60, lights=4, seed=6, extent=14.0)
    if kind == "two_level":
        scene.accel = _abi.ACCEL_TWO_LEVEL
    return scene, cam


def frame(ctx, graph, depth, pool, frames=2):
    ctx.set_tuning(launch_graph=graph)
    out = []
    for f in range(frames):
        p = render_params(W, H, SPP, min_depth=min(2, depth), max_depth=depth, state_count=pool, film_fp64=1)
        p.sample_offset = SPP * f
        st = ctx.render(p)
        out.append((ctx.film(W, H, fp64=True)[1], st.extension_rays, st.shadow_rays, st.paths))
    ctx.set_tuning(launch_graph=1)
    return out


@pytest.mark.parametrize("kind", ["room", "field", "two_level", "media"])
@pytest.mark.parametrize("depth,pool", [(0, PATHS), (1, PATHS), (2, PATHS + 1), (9, PATHS), (10, PATHS),
                                        (8, PATHS - 1), (5, 1000), (3, 64)])
def test_graph_equals_direct_launches(ctx, kind, depth, pool):
    scene, cam = scene_of(kind)
    ctx.upload_scene(scene)
    ctx.set_camera(cam, W, H)
    for a, b in zip(frame(ctx, 1, depth, pool), frame(ctx, 0, depth, pool)):
        assert a[1:] == b[1:] and a[3] == PATHS
        assert np.abs(a[0] - b[0]).max() <= 1e-12 * max(1.0, np.abs(b[0]).max())


@pytest.mark.parametrize("train,train_depth,query_depth", [(1, 0, 2), (1, 2, 2), (1, 4, 2), (0, 0, 2), (0, 0, 12)])
def test_cache_frames(ctx, train, train_depth, query_depth):
    scene, cam = scene_of("room")
    ctx.upload_scene(scene)
    ctx.set_camera(cam, W, H)
    counts = []
    for graph in (1, 0):
        ctx.set_tuning(launch_graph=graph)
        ctx.nrc_configure(enabled=1, train=train, train_depth=train_depth, query_depth=query_depth, steps=1)
        ctx.nrc_reset(4)
        out = []
        for f in range(3):
            p = render_params(W, H, 1, max_depth=8, state_count=1 << 13)
            p.sample_offset, p.accumulate = f, 1 if f else 0
            st = ctx.render(p)
            ns = ctx.nrc_stats()
            out.append((st.extension_rays, st.shadow_rays, ns.queries, ns.records))
        counts.append((out, ctx.film(W, H)[0], ctx.nrc_weights()))
    ctx.set_tuning(launch_graph=1)
    ctx.nrc_configure(enabled=0, train=1, train_depth=0, query_depth=2, steps=4)
    assert counts[0][0] == counts[1][0]
    np.testing.assert_allclose(counts[0][1], counts[1][1], rtol=1e-5, atol=1e-6)
    np.testing.assert_allclose(counts[0][2], counts[1][2], rtol=1e-5, atol=1e-6)
