// The arithmetic of the tile ranking: which bin of list lengths a tile is counted in and from which length on a list is
// shared out.  Plain C++, the same on the host and in the kernels.
#pragma once

#include <stdint.h>

namespace fgs {

constexpr int kOrderBins = 256, kOrderStep = 32;       // bins of so many entries; everything from 8160 up shares the first one
constexpr int kLeastShared = 128;          // entries of the shortest list that is ever shared out (see blend_kernel_shared)
// The longest length from which lists can be shared out: the ranking tells lists apart by their bins, and lists of the first bin
// not at all.
constexpr int kMostShared = (kOrderBins - 1) * kOrderStep;

// Bin of a list, the longest first.  (A length below zero, of a range that no ranges launch wrote, counts as empty.)
constexpr int order_bin(int length)
{
    const int step = length / kOrderStep;
    return kOrderBins - 1 - (step < 0 ? 0 : step < kOrderBins - 1 ? step : kOrderBins - 1);
}

// From which length on a list is shared out in a frame of which a SIMD walks `each` entries: three eighths of them, a multiple of
// kOrderStep between kLeastShared and kMostShared.
constexpr int least_shared_of(uint64_t each)
{
    const uint64_t least = each / 8 * 3 / kOrderStep * kOrderStep;
    return least < kLeastShared ? kLeastShared : least > kMostShared ? kMostShared : (int)least;
}

// The lists of `least` entries and more are those in the bins in front of this one.
constexpr int first_bin_below(int least) { return kOrderBins - least / kOrderStep; }

} // namespace fgs
