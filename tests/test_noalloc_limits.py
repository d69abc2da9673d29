"""How many wavefronts the no-allocation traversal launches, and which trees
it refuses (csrc/host/noalloc.h), without a GPU: the deepest tree accepted is
the one its first, 8 MiB scratch held (one wavefront, 16 entries per lane in
LDS), the entries always fit the scratch, and shallow trees keep their grid."""
import ctypes as C
import os
import subprocess

import pytest

from conftest import ROOT

SCRATCH, COUNTERS = 64 << 20, 2048


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("noalloc")
    src = d / "noalloc.cpp"
    src.write_text(f'#include "{ROOT}/btrc_amd/csrc/host/noalloc.h"\n'
                   'extern "C" int waves(int s, int l, int g) { return btrc::noalloc_waves(s, l, g); }\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", str(src), "-o", str(d / "noalloc.so")], check=True)
    return C.CDLL(str(d / "noalloc.so"))


@pytest.mark.parametrize("short_stack", [12, 16])
def test_limits(lib, short_stack):
    grid = 24 * 256
    deepest = 16 + ((8 << 20) - COUNTERS) // 512
    assert lib.waves(1, short_stack, grid) == lib.waves(short_stack, short_stack, grid) == grid
    assert lib.waves(deepest, short_stack, grid) >= 1
    assert lib.waves(deepest + 1, short_stack, grid) == 0
    for stack in (short_stack + 1, 34, 35, 43, 200, 5000, deepest):
        w = lib.waves(stack, short_stack, grid)
        bytes_per_wave = (stack - short_stack) * 512
        assert 1 <= w <= grid and w * bytes_per_wave <= SCRATCH - COUNTERS
        assert w == grid or (w + 1) * bytes_per_wave > SCRATCH - COUNTERS
