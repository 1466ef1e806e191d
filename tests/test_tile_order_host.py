"""The arithmetic by which a blend's tiles are ranked and shared out (flashgs_amd/csrc/tile_order.h), compiled for the CPU."""
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
