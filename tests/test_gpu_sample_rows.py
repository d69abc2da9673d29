"""Frames large enough to read their Halton numbers from sample rows: per
pixel against the oracle at the smallest such film, with depths that draw the
most (a minimum depth above the maximum included) and both filters; films that share too few pixels or are narrower than 128 keep the
digit loop; frames in several windows of samples equal the same samples
rendered separately, at a sample offset; tile order equals uniform order."""
import numpy as np
import pytest

from btrc_amd import _abi, scenes
from oracle import oracle

from util import render_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,spp,min_depth,max_depth,filt", [
    (512, 384, 2, 3, 8, "box"),          # 12 pixels a row: the first size with rows
    (512, 383, 2, 3, 8, "box"),          # just below
    (2048, 128, 1, 0, 3, "gaussian"),
    (4096, 127, 1, 3, 5, "box"),         # rows of 128 x 127 pixels, another stride
    (100, 64, 3, 3, 8, "box"), (129, 33, 1, 2, 6, "gaussian"), (1, 30, 2, 3, 4, "box"),
    (640, 400, 1, 9, 2, "gaussian"),     # nine vertices without roulette, then the end
])
def test_rows_match_oracle(ctx, w, h, spp, min_depth, max_depth, filt):
    scene, cam = scenes.cornell()
    ctx.upload_scene(scene)
    ctx.set_camera(cam, w, h)
    ctx.set_filter(filt)
    p = render_params(w, h, spp, min_depth=min_depth, max_depth=max_depth, state_count=1 << 18)
    st = ctx.render(p)
    got = ctx.film(w, h)[0][..., :3].astype(np.float64)
    ctx.set_filter("box")
    r0, r1 = h // 2, min(h, h // 2 + 24)
    o = oracle.OracleScene(scene)
    ref = sum(o.render(cam, p, first=(s * h + r0) * w, count=(r1 - r0) * w,
                       filt=None if filt == "box" else ("gaussian", 1.3, 1.6))[0][r0:r1] for s in range(spp)) / spp
    rel = np.abs(got[r0:r1] - ref) / np.maximum(np.abs(ref), 1e-2)
    assert rel.max() <= 1e-4 and ref.max() > 0
    assert st.paths == w * h * spp


def fp64_film(ctx, w, h, spp, offset=0, accumulate=0, tile=0, state_count=1 << 20):
    p = render_params(w, h, spp, min_depth=3, max_depth=6, state_count=state_count, film_fp64=1)
    p.sample_offset, p.accumulate, p.tile = offset, accumulate, tile
    st = ctx.render(p)
    return ctx.film(w, h, fp64=True)[1], st.extension_rays


@pytest.mark.parametrize("graph", [1, 0])
def test_windows_of_samples(ctx, graph):
    # media rows hold 998 dimensions: 32 samples fill the rows' memory, so 40
    # samples take two windows
    scene, cam = scenes.cornell_media(grid=scenes.fbm_grid(16, octaves=3, seed=3, max_sigma=0.2))
    ctx.upload_scene(scene)
    w, h = 512, 400
    ctx.set_camera(cam, w, h)
    ctx.set_tuning(launch_graph=graph)
    whole, rays = fp64_film(ctx, w, h, 40)
    _, first = fp64_film(ctx, w, h, 20)
    parts, second = fp64_film(ctx, w, h, 20, offset=20, accumulate=1)
    ctx.set_tuning(launch_graph=1)
    assert rays == first + second
    assert np.abs(whole - parts).max() <= 1e-12 * max(1.0, np.abs(parts).max())


def test_tile_order_equals_uniform(ctx):
    scene, cam = scenes.cornell()
    ctx.upload_scene(scene)
    ctx.set_camera(cam, 600, 400)
    a, ra = fp64_film(ctx, 600, 400, 3)
    b, rb = fp64_film(ctx, 600, 400, 3, tile=1, state_count=100000)
    assert ra == rb
    assert np.abs(a - b).max() <= 1e-12 * max(1.0, np.abs(a).max())


def test_draws_past_the_last_dimension(ctx):
    """paths that draw more numbers than the 998 dimensions of a row start over
    at the first: a frame that tracks from rows (staged in chunks) equals the
    same camera as one of two views, where the small one keeps the digit loop"""
    grid = scenes.fbm_grid(10, octaves=3, seed=5, max_sigma=0.02).copy()
    grid[0, 0, 0] = 30.0   # 30 steps a unit, 40 units across, few of them real
    scene, cam = scenes.cornell_media(grid=grid)
    ctx.upload_scene(scene)
    w, h = 512, 384
    p = render_params(w, h, 1, max_depth=3, state_count=1 << 18)
    ctx.set_camera(cam, w, h)
    ctx.render(p)
    rows = ctx.film(w, h)[0]
    ctx.render_views(p, [(cam, w, h), (cam, 8, 8)])
    digits = ctx.view_film(0, w, h)
    np.testing.assert_allclose(rows, digits, rtol=1e-5, atol=1e-6)
    oracle.tracking_stats()
    ref = oracle.OracleScene(scene).render(cam, p, first=(h // 2) * w, count=w)[0][h // 2]
    segments, lookups = oracle.tracking_stats()
    assert lookups > 998 * segments / 2   # two draws a lookup
    assert (np.abs(rows[h // 2, :, :3] - ref) / np.maximum(np.abs(ref), 1e-2)).max() <= 1e-4 and ref.max() > 0


def test_rows_give_their_memory_back(ctx):
    """rows of two gigabytes are released by the next frame that needs none or
    far fewer and by a new scene, kept by frames that use them, and taken again
    beside another pool"""
    import ctypes as C
    hip = C.CDLL("libamdhip64.so.7")   # the runtime the library itself links
    free, total = C.c_size_t(), C.c_size_t()

    def used():
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return (total.value - free.value) / 2.0 ** 20

    def large():
        p = render_params(512, 384, 32, max_depth=2, state_count=1 << 16)
        ctx.render(p)     # media rows: 16,384 x 1,000 floats a sample
        return used()

    scene, cam = scenes.cornell_media(grid=scenes.fbm_grid(8, octaves=3, seed=3, max_sigma=0.2))
    ctx.upload_scene(scene)
    ctx.set_camera(cam, 512, 384)
    one = render_params(512, 384, 1, max_depth=2, state_count=1 << 16)
    independent = render_params(512, 384, 1, max_depth=2, state_count=1 << 16)
    independent.sampler = _abi.SAMPLER_INDEPENDENT
    ctx.render(independent)
    before = used()
    for change in (lambda: ctx.render(independent), lambda: ctx.render(one), lambda: ctx.upload_scene(scene)):
        assert large() > before + 1900
        assert large() > before + 1900
        change()
        assert used() < before + 100
    assert large() > before + 1900
    ctx.render(render_params(512, 384, 32, max_depth=2, state_count=1 << 17))
    assert used() > before + 1900
