"""Batches that a caller loads into the cache: the smallest, those around a
wavefront's samples, the largest, and small ones after the largest (whose
records must be gone); queries that fit the scratch and more that do not."""
import numpy as np
import pytest

from btrc_amd import scenes
from oracle import oracle

pytestmark = pytest.mark.gpu

RECORDS = 1 << 16
SCRATCH_QUERIES = 6 * 64 * RECORDS * 2 // 76


def vertices(n, box, seed):
    rng = np.random.default_rng(seed)
    v = np.empty((n, 16), dtype=np.float32)
    v[:, 0:3] = box[:3] + rng.uniform(0, 1, (n, 3)) / box[3:]
    for a in (3, 6):
        d = rng.standard_normal((n, 3))
        v[:, a:a + 3] = d / np.linalg.norm(d, axis=1, keepdims=True)
    v[:, 9] = rng.uniform(0.05, 1.0, n)
    v[:, 10:16] = rng.uniform(0, 1, (n, 6))
    return v, rng.uniform(0, 2, (n, 3)).astype(np.float32)


@pytest.fixture()
def cache(ctx):
    scene, cam = scenes.cornell()
    ctx.upload_scene(scene)
    ctx.set_camera(cam, 64, 64)
    ctx.nrc_reset(6)
    yield ctx
    ctx.nrc_configure(enabled=0)


@pytest.mark.parametrize("n", [1, 31, 32, 33, 1000, RECORDS - 1, RECORDS])
def test_gradients(cache, n):
    box, w = cache.scene_box(), cache.nrc_weights()
    cache.nrc_gradients(*vertices(RECORDS, box, 1))
    v, t = vertices(n, box, 2 + n)
    g, loss = cache.nrc_gradients(v, t)
    if n <= 1000:
        # one sample's relative gradients differ by the BF16 roundings of six
        # layers (about 6 * 2^-8 of the norm)
        ref, ref_loss = oracle.nrc_gradients(w, box, v, t, bf16=True)
        assert abs(loss - ref_loss) <= 6 * 2.0 ** -8 * ref_loss + 1e-6
        assert np.linalg.norm(g - ref) <= 6 * 2.0 ** -8 * 3 * np.linalg.norm(ref)
    else:
        # the sum over a batch is the sum over its parts, up to the order of
        # FP32 additions of 2^16 terms
        half = n // 2
        a, la = cache.nrc_gradients(v[:half], t[:half])
        b, lb = cache.nrc_gradients(v[half:], t[half:])
        parts = (a.astype(np.float64) * half + b.astype(np.float64) * (n - half)) / n
        assert np.linalg.norm(g - parts) <= 2.0 ** -16 * np.linalg.norm(parts)
        assert abs(loss - (la * half + lb * (n - half)) / n) <= 1e-12 * loss
    again, loss2 = cache.nrc_gradients(v, t)
    assert np.array_equal(g, again) and loss == loss2


@pytest.mark.parametrize("n", [1, 127, 129, SCRATCH_QUERIES, SCRATCH_QUERIES + 1])
def test_queries(cache, n):
    v, _ = vertices(n, cache.scene_box(), 3)
    out = cache.nrc_eval(v)
    assert np.isfinite(out).all()
    # an answer does not depend on the queries beside it
    parts = [cache.nrc_eval(p) for p in np.array_split(v, 3) if len(p)]
    assert np.array_equal(out, np.concatenate(parts))
