"""The traversal's slab test (csrc/core/traverse.h) never loses a box that
holds a hit, at any magnitude of origins and directions: a triangle the
watertight test hits must be entered through its own box, up to the culling
distance of that very hit. Rays inside a box's face, origins beyond 2^32 with
zero direction components, directions far below and above unit length, mixed
magnitudes; and boxes that a ray clearly misses stay missed (an axis may not
be given up for rays of ordinary magnitude)."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT

MAX_FLOAT = np.float32(3.4028234663852886e38)


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("ray_box") / "ray_box.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-ffp-contract=off", "-Wno-unknown-pragmas",
                    os.path.join(ROOT, "tests", "cpp", "ray_box.cpp"), "-o", so], check=True)
    lib = C.CDLL(so)

    def go(o, d, tris, tmin=0.0, tmax=MAX_FLOAT, boxes=None):
        n = len(o)
        rays = np.zeros((n, 8), np.float32)
        rays[:, :3], rays[:, 3], rays[:, 4:7], rays[:, 7] = o, tmin, d, tmax
        tris = np.ascontiguousarray(np.broadcast_to(tris, (n, 9)), np.float32)
        boxes = np.zeros((n, 6), np.float32) if boxes is None else np.ascontiguousarray(boxes, np.float32)
        out = np.zeros(n, np.uint8)
        lib.ray_box(*(a.ctypes.data_as(C.c_void_p) for a in (rays, tris, boxes)), C.c_int(n),
                    out.ctypes.data_as(C.c_void_p))
        return out
    return go


WALL = np.array([-1, -1, 0, 3, -1, 0, -1, 3, 0], np.float32)  # across z, at z = 0


@pytest.mark.parametrize("o,d,tri", [
    # beyond 2^32 along an axis the ray does not move on
    ([5e9, 0, 0], [0, 0, 1], [4e9, -1e9, 1e9, 9e9, -1e9, 1e9, 5e9, 3e9, 1e9]),
    ([0, -3e12, 0], [1, 0, -0.0], [1, -1e13, -1e3, 1, 1e13, -1e3, 1, 0, 3e3]),
    # every component tiny
    ([0, 0, 0], [1e-30, 1e-29, 0], [1, 5, -1, 1, 15, -1, 1, 10, 3]),
    ([0, 0, 0], [1e-30, 2e-30, 1e-31], [1, 1, -1, 1, 4, -1, 1, 2, 3]),
    ([0, 0, 0], [0, 0, 1e-36], [-1, -1, 1, 3, -1, 1, -1, 3, 1]),
    # inside the plane x = 0 of the box's face, far from it
    ([0, 0, -1e5], [0, 0, 1], [0, -1, 0, -2, -1, 0, 0, 2, 0]),
    ([0, 0, -3], [0, 0, 1e-6], [0, -1, 0, -2, -1, 0, 0, 2, 0]),
    # directions near the largest float
    ([-3, -0.5, 0], [3e38, 5e37, 0], [0, -1, -1, 0, 1, -1, 0, 0, 2]),
])
def test_extreme_rays_keep_their_box(run, o, d, tri):
    got = run(np.float32([o]), np.float32([d]), np.float32(tri))
    assert got[0] & 1, "the triangle test itself must hit"
    assert got[0] & 2


def test_mixed_magnitudes_keep_their_box(run):
    """triangles of many sizes and places, rays through a point of each (its
    corners and edges too), directions with zero, tiny and ordinary
    components at every overall length"""
    rng = np.random.default_rng(11)
    n = 400000
    size = 10.0 ** rng.uniform(-6, 6, (n, 1, 1))
    centre = rng.uniform(-1, 1, (n, 1, 3)) * 10.0 ** rng.uniform(-6, 9, (n, 1, 1)) * rng.choice([0, 1], (n, 1, 3))
    flat = np.ones((n, 1, 3))
    flat[np.arange(n), 0, rng.integers(0, 3, n)] = rng.choice([0.0, 1.0], n)  # half of the boxes flat along one axis
    tris = np.float32(centre + rng.uniform(-1, 1, (n, 3, 3)) * size * flat)
    w = rng.dirichlet([0.3] * 3, n)
    w[rng.random(n) < 0.1] = [1, 0, 0]
    w[rng.random(n) < 0.1] = [0.5, 0.5, 0]
    p = (w[:, :, None] * tris.astype(np.float64)).sum(1)
    d = rng.normal(size=(n, 3)) * rng.choice([1.0, 1.0, 0.0, -0.0, 1e-10, 1e-25], (n, 3))
    d *= 10.0 ** rng.choice([0, 0, -5, -12, -20, -28, -33, 10, 30], (n, 1))
    d = np.float32(d)
    length = np.abs(d).max(1, keepdims=True).astype(np.float64)
    keep = length[:, 0] > 0
    far = size[:, 0] * 10.0 ** rng.uniform(-2, 4, (n, 1))
    o = np.float32(p - d / np.where(length > 0, length, 1) * far)
    got = run(o[keep], d[keep], tris[keep].reshape(-1, 9))
    hits = got & 1 != 0
    assert hits.sum() > n // 10
    lost = np.flatnonzero(hits & (got & 2 == 0))
    assert len(lost) == 0, (o[keep][lost[:3]], d[keep][lost[:3]], tris[keep][lost[:3]])


def test_clear_misses_stay_missed(run):
    """unit directions with one or two zero components past unit boxes: a
    hundredth of the box's size off on an axis the ray does not move on"""
    rng = np.random.default_rng(4)
    n = 50000
    scale = 10.0 ** rng.uniform(-3, 6, (n, 1))
    axis = rng.integers(0, 3, n)
    d = rng.normal(size=(n, 3))
    d[rng.random((n, 3)) < 0.3] = 0.0
    d[np.arange(n), axis] = 0.0
    d[np.abs(d).max(1) == 0, :] = np.eye(3)[(axis[np.abs(d).max(1) == 0] + 1) % 3]
    lo = rng.uniform(-1, 0, (n, 3)) * scale
    hi = lo + rng.uniform(0.5, 1, (n, 3)) * scale
    o = rng.uniform(lo, hi)
    side = rng.random(n) < 0.5
    off = 0.01 * scale[:, 0]
    o[np.arange(n), axis] = np.where(side, hi[np.arange(n), axis] + off, lo[np.arange(n), axis] - off)
    got = run(np.float32(o), np.float32(d), WALL, boxes=np.concatenate([lo, hi], 1))
    assert not (got & 4).any()
