"""The Halton sampler as the tracer's stages evaluate it (even samples:
first-digit tables and the 24-bit digit loop after them; odd samples: the
digit loop from the first digit, as the tracking kernel runs it) against the
oracle's digit loop, bit for bit, where it can go wrong: the last dimension
and the wrap past it, films smaller than a stratum, the largest index a render
reaches, and indices beyond 32 bits (the general loop)."""
import numpy as np
import pytest

from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,lo,hi", [
    (1920, 1080, 0, 64), (1, 1, 0, 100000), (37, 500, 0, 3000),
    (640, 480, 2 ** 31 // 31104 - 50, 2 ** 31 // 31104 - 1),      # indices up to 2^31
    (640, 480, 2 ** 31 // 31104 + 1, 2 ** 31 // 31104 + 100)])    # the offset overflows: 64-bit indices
def test_every_dimension_equals_the_oracle(ctx, w, h, lo, hi):
    rng = np.random.default_rng(w + hi)
    n = 700
    px, py = rng.integers(0, w, n), rng.integers(0, h, n)
    px[1], py[1], si = px[0], py[0], rng.integers(lo, hi, n)
    si[:2] = hi - 1, hi - 1   # the largest index by both forms
    gpu = ctx.eval_halton(w, h, px, py, si, 1010)   # dimensions 2..999, then 2 again
    cpu = oracle.halton(w, h, px, py, si, 1010)
    assert np.array_equal(gpu.view(np.uint32), cpu.view(np.uint32))
