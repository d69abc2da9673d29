"""Reporter callbacks during a render (Reporter, core/reporter.h:7-36, as
WavefrontPathTracer::render calls it, wavefront.cpp:221,287,314): one new
stage, progress rising to 100 % of the frame's paths, one completed stage,
also when the render is stopped from inside a progress callback."""
import threading
import time

import pytest

import btrc_amd
from btrc_amd import _abi, scenes

from util import render_params

pytestmark = pytest.mark.gpu


class Recorder:
    def __init__(self, stop_ctx=None):
        self.calls = []
        self.stop_ctx = stop_ctx

    def new_stage(self, name):
        self.calls.append(("new_stage", name))

    def complete_stage(self):
        self.calls.append(("complete_stage",))

    def progress(self, pct):
        self.calls.append(("progress", pct))
        if self.stop_ctx is not None:
            self.stop_ctx.lib.btrc_hip_request_stop(self.stop_ctx.h)


@pytest.mark.parametrize("graph", [1, 0])
def test_reporter_sees_the_whole_frame(ctx, graph):
    scene, cam = scenes.cornell()
    ctx.upload_scene(scene)
    ctx.set_camera(cam, 64, 64)
    ctx.set_tuning(launch_graph=graph)
    rec = Recorder()
    ctx.set_reporter(rec)
    try:
        ctx.render(render_params(64, 64, 16, state_count=1 << 14))
    finally:
        ctx.set_reporter(None)
    assert rec.calls[0] == ("new_stage", "") and rec.calls[-1] == ("complete_stage",)
    pct = [c[1] for c in rec.calls if c[0] == "progress"]
    assert len(pct) >= 2 and len(rec.calls) == len(pct) + 2
    assert all(0.0 <= a <= b for a, b in zip(pct, pct[1:]))
    assert pct[-1] == 100.0
    # removed: later renders report nothing
    ctx.render(render_params(64, 64, 1, state_count=1 << 14))
    assert rec.calls[-1] == ("complete_stage",) and len(rec.calls) == len(pct) + 2


def test_reporter_stage_completes_when_stopped(ctx):
    scene, cam = scenes.cornell()
    ctx.upload_scene(scene)
    ctx.set_camera(cam, 64, 64)
    rec = Recorder(stop_ctx=ctx)
    ctx.set_reporter(rec)
    try:
        with pytest.raises(btrc_amd.BtrcException) as e:
            ctx.render(render_params(64, 64, 64, state_count=1 << 12))
        assert e.value.status == _abi.BTRC_ERR_STOPPED
    finally:
        ctx.set_reporter(None)
    assert rec.calls[0][0] == "new_stage" and rec.calls[-1] == ("complete_stage",)
    assert sum(1 for c in rec.calls if c[0] == "progress") == 1


@pytest.mark.parametrize("stop", [False, True])
def test_progress_and_stop_within_a_frame_that_fits_the_pool(ctx, stop):
    """nine bounces, every path in flight at once: progress comes after each
    four, and a stop request from the first one ends the render"""
    scene, cam = scenes.cornell()
    ctx.upload_scene(scene)
    ctx.set_camera(cam, 64, 64)
    p = render_params(64, 64, 4, min_depth=8, max_depth=8, state_count=1 << 14)
    plain = ctx.render(p)
    rec = Recorder(stop_ctx=ctx if stop else None)
    ctx.set_reporter(rec)
    try:
        if stop:
            with pytest.raises(btrc_amd.BtrcException) as e:
                ctx.render(p)
            assert e.value.status == _abi.BTRC_ERR_STOPPED
        else:
            st = ctx.render(p)
            assert (st.extension_rays, st.shadow_rays) == (plain.extension_rays, plain.shadow_rays)
    finally:
        ctx.set_reporter(None)
    pct = [c[1] for c in rec.calls if c[0] == "progress"]
    assert len(pct) == (1 if stop else 3)
    assert all(0.0 <= a <= b for a, b in zip(pct, pct[1:])) and (stop or pct[-1] == 100.0)
    # the context renders on as before
    st = ctx.render(p)
    assert (st.extension_rays, st.shadow_rays) == (plain.extension_rays, plain.shadow_rays)


def test_stop_request_while_a_frame_that_fits_the_pool_runs(ctx):
    """without a progress callback such a frame has one read-back; a request
    from another thread meanwhile still ends it as stopped"""
    scene, cam = scenes.cornell()
    ctx.upload_scene(scene)
    ctx.set_camera(cam, 2048, 2048)
    p = render_params(2048, 2048, 4, min_depth=8, max_depth=8, state_count=1 << 24)
    ctx.render(p)
    t = time.perf_counter()
    plain = ctx.render(p)
    seconds = time.perf_counter() - t
    assert seconds > 0.005

    def stop():
        time.sleep(0.3 * seconds)
        ctx.lib.btrc_hip_request_stop(ctx.h)

    th = threading.Thread(target=stop)
    th.start()
    try:
        with pytest.raises(btrc_amd.BtrcException) as e:
            ctx.render(p)
        assert e.value.status == _abi.BTRC_ERR_STOPPED
    finally:
        th.join()
    assert ctx.render(p).extension_rays == plain.extension_rays
