"""The cut of a batch's picks into tiles (csrc/moe_tiles.h), compiled for the CPU: the rule, and the arithmetic at the
largest batches, where a GPU run would need every pick's buffers."""
import ctypes
import subprocess

import pytest

from conftest import PKG

SRC = """#include "moe_tiles.h"
extern "C" int tile_begin(int c, int j, int n) { return aegist::tile_begin(c, j, n); }
extern "C" int tile_picks(int T, int K, int E, int D, int I) { return aegist::moe_tile_picks(T, K, E, D, I); }
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


@pytest.mark.parametrize("T,K,E,I,picks", [
    # too few workgroups of 256 units: few experts, one token's picks at widths the decode kernel does not take
    (9, 2, 8, 512, 0), (32, 2, 8, 512, 0), (1, 8, 256, 768, 0), (4, 8, 256, 256, 0), (1, 2, 8, 1408, 0), (16, 4, 16, 128, 0),
    # the second round of workgroups nearly empty; padded units
    (16, 8, 256, 768, 0), (24, 8, 128, 768, 0), (64, 8, 256, 1408, 0),
    # experts of 17 to 32 picks, few workgroups
    (192, 2, 16, 768, 0), (96, 4, 16, 256, 0),
    # full rounds
    (65, 8, 256, 512, 64), (96, 8, 256, 512, 64), (128, 8, 256, 512, 64), (512, 8, 256, 512, 64), (1000, 8, 256, 512, 64),
    (2048, 8, 256, 512, 64), (64, 8, 256, 256, 64), (128, 8, 256, 768, 64),
    # experts past 16 picks that leave room for smaller tiles
    (128, 2, 8, 512, 16), (512, 2, 8, 1408, 32), (400_000, 1, 1, 128, 64), (2048, 2, 4, 256, 32)])
def test_tile_rule(tiles, T, K, E, I, picks):
    assert tiles.tile_picks(T, K, E, 2048, I) == picks


def test_tile_rule_takes_any_batch(tiles):
    for E in (1, 2, 5, 16, 255, 1024):
        for K in (1, 2, 8, 16):
            for T in (1, 2, 17, 333, 70_000, 2 ** 30 // K - 1):
                for I in (128, 640, 2048):
                    assert tiles.tile_picks(T, K, E, 640, I) in (0, 16, 32, 48, 64)


def test_tile_rule_counts_the_longer_rows_workgroups(tiles):
    """Wide experts of a narrow model: the down projection's few outputs decide."""
    assert tiles.tile_picks(24, 4, 32, 256, 2048) == 0 and tiles.tile_picks(96, 8, 256, 512, 2048) == 64


# the batches of test_moe_decode_gpu.py's sizes of tiles
@pytest.mark.parametrize("T,D,I,E,K,picks", [(70, 384, 256, 256, 8, 64), (96, 256, 256, 8, 2, 0), (128, 384, 256, 8, 2, 16),
                                             (1024, 256, 256, 4, 2, 16), (2048, 256, 256, 4, 2, 32),
                                             (5000, 256, 256, 8, 2, 48), (8000, 256, 256, 8, 2, 64),
                                             (1, 256, 768, 64, 8, 0), (9, 512, 512, 8, 2, 0)])
def test_tile_rule_of_the_gpu_test(tiles, T, D, I, E, K, picks):
    assert tiles.tile_picks(T, K, E, D, I) == picks


@pytest.mark.parametrize("K,D,I,E", [(8, 2048, 512, 256), (2, 512, 1408, 8), (1, 128, 128, 1), (4, 256, 256, 16), (8, 64, 192, 64)])
def test_workspace_of_more_tokens_serves_fewer(K, D, I, E):
    """The workspace is asked for once, for up to T tokens: its size may not fall with T, whatever tiles a
    smaller batch takes."""
    from aegist_mixer._lib import lib
    size = lib().aegist_moe_workspace_bytes
    ts = sorted({*range(1, 3000), *range(3000, 1_000_000, 997), *(int(2 ** 32 / (2 * n)) + d for n in (D, K * I) for d in (-1, 0, 1))})
    sizes = [size(t, K, D, I, E) for t in ts]
    for t, a, b in zip(ts, sizes, sizes[1:]):
        assert a <= b, (t, a, b)


def test_tile_rule_does_not_open_a_round_for_a_few_workgroups(tiles):
    """272 workgroups of 64 picks are two rounds of 256, which 48 picks fill better."""
    assert tiles.tile_picks(2048, 2, 8, 896, 896) == 48
