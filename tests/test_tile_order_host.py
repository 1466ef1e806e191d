"""The order of a large frame's tiles and the arithmetic by which a small one's are ranked and shared out (flashgs_amd/csrc/tile_order.h), compiled for the CPU."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "tile_order.h"
extern "C" void least_of(const uint64_t* each, int n, int* out) { for (int i = 0; i < n; i++) out[i] = fgs::least_shared_of(each[i]); }
extern "C" void bin_of(const int* length, int n, int* out) { for (int i = 0; i < n; i++) out[i] = fgs::order_bin(length[i]); }
extern "C" int first_bin(int least) { return fgs::first_bin_below(least); }
extern "C" long long positions(int tiles_x, int tiles_y) { return fgs::positions_of(tiles_x, tiles_y); }
extern "C" int block_size(int tiles_x, int tiles_y) { return 1 << fgs::block_log2_of(tiles_x, tiles_y); }
extern "C" void tiles_of(int tiles_x, int tiles_y, int n, int* out)
{
    for (int g = 0; g < n; g++) {
        int x = 0, y = 0;
        out[g] = fgs::tile_of_position(g, tiles_x, tiles_y, &x, &y) ? y * tiles_x + x : -1;
    }
}
extern "C" int bins(void) { return fgs::kOrderBins; }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    where = tmp_path_factory.mktemp("tile_order")
    (where / "order.cpp").write_text(PROGRAM)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "flashgs_amd", "csrc"),
                           str(where / "order.cpp"), "-o", str(where / "order.so")])
    return C.CDLL(str(where / "order.so"))


def of(function, dtype, values):
    values = np.asarray(values, dtype)
    out = np.empty(len(values), np.int32)
    function(values.ctypes.data_as(C.c_void_p), len(values), out.ctypes.data_as(C.c_void_p))
    return out


def test_the_ranking_counts_every_list_that_is_shared_out(lib):
    """A ranked tile whose list reaches the length has a workgroup with all its teams, and only such a tile has: so the bins
    in front of first_bin_below hold the lists of that length and more and no others, however many entries a
    SIMD walks of the frame."""
    each = np.array(sorted({*range(0, 30000, 7), *(1 << b for b in range(64)), 21845, 21846, 21888, 2 ** 64 - 1}), np.uint64)
    lengths = np.array([-(2 ** 31), -1, *range(20000), 2 ** 30 - 1, 2 ** 30, 2 ** 30 + 1, 2 ** 31 - 2, 2 ** 31 - 1])
    bins = of(lib.bin_of, np.int32, lengths)
    assert bins.min() == 0 and bins.max() == lib.bins() - 1
    assert (np.diff(bins[1:]) <= 0).all()                 # the longest lists come first
    least = of(lib.least_of, np.uint64, each)
    assert (np.diff(least) >= 0).all() and least[0] >= 128
    for l in np.unique(least):
        first = lib.first_bin(int(l))
        assert 0 < first < lib.bins()
        assert np.array_equal(bins < first, lengths >= l), l


@pytest.mark.parametrize("tiles_x, tiles_y", [(1, 1), (1, 9000), (9000, 1), (7, 1200), (8, 1025), (85, 107), (91, 91), (170, 107), (188, 138), (240, 135),
                                              (320, 180), (300, 225), (224, 127), (224, 128), (224, 129), (341, 513), (415, 254), (480, 270), (513, 513), (856, 12)])
def test_every_tile_of_a_large_frame_has_one_position(lib, tiles_x, tiles_y):
    """Every tile once, a block of tiles on one XCD, and blocks below each other on XCDs five apart, or five and
    the blocks of a row where the rotation of the row wraps (never, where these are a multiple of 8)."""
    lib.positions.restype = C.c_longlong
    n, size = lib.positions(tiles_x, tiles_y), lib.block_size(tiles_x, tiles_y)
    tiles = np.empty(n, np.int32)
    lib.tiles_of(tiles_x, tiles_y, n, tiles.ctypes.data_as(C.c_void_p))
    found = tiles[tiles >= 0]
    assert np.array_equal(np.sort(found), np.arange(tiles_x * tiles_y))
    xcd = np.full((tiles_y + size, tiles_x), -1)
    xcd[tiles[tiles >= 0] // tiles_x, tiles[tiles >= 0] % tiles_x] = np.flatnonzero(tiles >= 0) % 8
    xcd = xcd[:tiles_y]
    blocks = xcd[::size, ::size]
    assert np.array_equal(np.kron(blocks, np.ones((size, size), int))[:tiles_y, :tiles_x], xcd)
    apart = (blocks[1:] - blocks[:-1]) % 8
    width = blocks.shape[1]
    wrapped = {(5 + k * width) % 8 for k in range(-8, 9)} if width < 8 else {5, (5 + width) % 8}
    assert set(np.unique(apart)) <= wrapped
    if width % 8 == 0:
        assert (apart == 5).all()
