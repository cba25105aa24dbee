"""The cut of an expert's picks into tiles (csrc/moe_tiles.h), compiled for the CPU: the arithmetic at the
largest batches, where a GPU run would need every pick's buffers."""
import ctypes
import subprocess

import pytest

from conftest import PKG

SRC = """#include "moe_tiles.h"
extern "C" int tile_begin(int c, int j, int n) { return aegist::tile_begin(c, j, n); }
"""


@pytest.fixture(scope="module")
def tiles(tmp_path_factory):
    so = tmp_path_factory.mktemp("moe_tiles") / "moe_tiles.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-x", "c++", "-", "-I",
                    str(PKG / "csrc"), "-o", str(so)], input=SRC, text=True, check=True)
    return ctypes.CDLL(str(so))


@pytest.mark.parametrize("c", [1, 63, 64, 65, 129, 4097, 370703, 370704, 400000, 5_000_000, 2 ** 30 - 1])
def test_tiles_cover_the_picks_in_order(tiles, c):
    n = (c + 63) // 64
    # all boundaries of a small count, a spread of a large one's and both of its ends
    js = range(n) if n < 20000 else [*range(100), *range(100, n - 100, n // 5000), *range(n - 100, n)]
    assert tiles.tile_begin(c, 0, n) == 0 and tiles.tile_begin(c, n, n) == c
    for j in js:
        a, b = tiles.tile_begin(c, j, n), tiles.tile_begin(c, j + 1, n)
        assert c // n <= b - a <= min(64, c // n + 1), (j, a, b)
