"""Density grids read from bricks: delta and ratio tracking bit for bit
against the oracle's plain grids at the sizes where the bricks end (one to a
few voxels along an axis, odd and even), inside, outside and across the
borders; several grids in one scene, beside albedo grids."""
import numpy as np
import pytest

from btrc_amd import _abi, scenes
from oracle import oracle

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (1, 2, 3), (2, 1, 4), (3, 3, 3), (4, 5, 2), (7, 1, 6), (5, 4, 9), (16, 15, 17)]  # z, y, x


def grids(seed):
    rng = np.random.default_rng(seed)
    return [rng.uniform(0.1, 3.0, s).astype(np.float32) for s in SHAPES]


def segments(n, seed, lo, hi):
    rng = np.random.default_rng(seed)
    seg = np.zeros(n, dtype=_abi.ray_dtype())
    a = rng.uniform(lo, hi, (n, 3)).astype(np.float32)
    seg["o"], seg["d"], seg["tmax"] = a, rng.uniform(lo, hi, (n, 3)).astype(np.float32) - a, 1.0
    return seg, rng.integers(0, 2 ** 63, n, dtype=np.uint64)


def test_media(ctx):
    s = scenes.Scene()
    for k, g in enumerate(grids(1)):
        alb = np.random.default_rng(k).uniform(0.2, 0.9, g.shape + (3,)).astype(np.float32) if k % 2 else None
        s.add_heterogeneous(g, (0.7, 0.8, 0.9), g=0.3, priority=float(-k), albedo_grid=alb)
    box = np.concatenate(scenes.box_faces(1, 1, 1))
    s.add_instance(s.add_geometry(box), s.add_invisible(), inner_medium=0)
    ctx.upload_scene(s)
    ref = oracle.OracleScene(s)
    seg, seeds = segments(4000, 2, -1.6, 1.6)   # the grids span [-1, 1]^3
    for m in range(len(SHAPES)):
        got, want = ctx.eval_medium(m, seg, seeds), ref.medium_eval(m, seg, seeds)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), SHAPES[m]
        assert 0.02 < got[:, 0].mean() < 0.98


@pytest.mark.parametrize("shape", SHAPES)
def test_volumes(ctx, shape):
    s = scenes.Scene()
    g = np.random.default_rng(9).uniform(0.1, 3.0, shape).astype(np.float32)
    s.add_volume((-0.5, -0.5, -0.5), (1, 0, 0), (0, 1, 0), (0, 0, 1), g, (0.9, 0.8, 0.7))
    ctx.upload_scene(s)
    seg, seeds = segments(4000, 3, -0.8, 0.8)
    got, want = ctx.eval_volumes(seg, seeds), oracle.OracleScene(s).volume_eval(seg, seeds)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
