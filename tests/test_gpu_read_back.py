"""Large results come back in chunks through pinned slots, emptied by two
threads: one chunk exactly, a ragged second one, every slot in use, slots used
again. The bytes in a numpy array (pageable) equal those that the direct copy
leaves in pinned memory; FP64 films are scaled by 1 / spp on the way. Two
contexts read at once from two threads."""
import threading

import numpy as np
import pytest
import torch

import btrc_amd
from btrc_amd import scenes

from util import render_params

pytestmark = pytest.mark.gpu

CHUNK = (2 << 20) // 16     # pixels of four floats per chunk


def rendered(ctx, width, height):
    scene, cam = scenes.cornell()
    ctx.upload_scene(scene)
    ctx.set_camera(cam, width, height)
    ctx.render(render_params(width, height, 3, min_depth=0, max_depth=1, film_fp64=1))


def check(ctx, width, height):
    rgba, rgb64 = ctx.film(width, height, fp64=True)
    a = torch.full((height, width, 4), -1.0, dtype=torch.float32, pin_memory=True)
    b = torch.full((height, width, 3), -1.0, dtype=torch.float64, pin_memory=True)
    ctx._check(ctx.lib.btrc_hip_film_readback(ctx.h, a.data_ptr(), b.data_ptr()))
    assert rgba.max() > 0 and rgba.tobytes() == a.numpy().tobytes()
    assert rgb64.tobytes() == b.numpy().tobytes()
    # FP32 atomics: three samples' sums and one product against FP64's
    assert np.allclose(rgb64, rgba[..., :3], rtol=8 * 2.0 ** -24, atol=0)


@pytest.mark.parametrize("width,height", [(CHUNK, 1), (CHUNK + 1, 1), (1, 2 * CHUNK // 3 + 1), (CHUNK, 8),
                                          (1003, 1309), (251, 8801)])
def test_pageable_equals_pinned(ctx, width, height):
    rendered(ctx, width, height)
    check(ctx, width, height)


def test_two_contexts_read_at_once():
    contexts = [btrc_amd.Context() for _ in range(2)]
    sizes = [(1003, 1309), (640, 2100)]
    for c, size in zip(contexts, sizes):
        rendered(c, *size)
    failures = []

    def work(c, size):
        try:
            for _ in range(4):
                check(c, *size)
        except BaseException as e:      # reported by the main thread
            failures.append(e)

    threads = [threading.Thread(target=work, args=a) for a in zip(contexts, sizes)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures[0]
