// The order in which the tiles of a large frame start, and the arithmetic of the ranking of a small one's: which bin of list lengths a
// tile is counted in and from which length on a list is shared out.  Plain C++, the same on the host and in the kernels.
#pragma once

#include <stdint.h>

namespace fgs {

// Position in the launch of a frame that is not ranked -> tile.  The hardware deals consecutive workgroups out to the 8 XCDs in
// turn, and every XCD has its own L2.  Neighbouring tiles share most of their Gaussians, so each
// XCD is given whole blocks of tiles (of 8x8: its positions g = 8*slot + xcd walk blocks xcd, xcd+8,
// ... 64 tiles at a time): a Gaussian's attribute lines are then fetched into one L2 once instead
// of into several L2s once per tile.  Every row of blocks begins further right, so that a block's XCD is five behind that of the one above
// it or, in rows of other than a multiple of 8 blocks, where the rotation wraps, 5 + blocks_x: row after row from the left, an XCD would
// have the same columns of blocks in every second row of a frame of 60 blocks, in every row of one of 24, and 2 to 14 % more to blend
// than the average, and the launch ends when the last XCD does.  Blocks are of 4x4 tiles where of 8x8 an XCD would have some 55 or fewer,
// which no order deals evenly, and of 8x8 above, where smaller ones cost more in bytes (8 to 21 %) than they even out.  Behind the
// sort, in us (8x8 row after row; 8x8 and 4x4 five apart): 3000x2200 / 2M (25 944 tiles) 207; 199, 192; 3047x1725 / 1.1M clusters 180; 172, 164;
// 2720x1700 / 3M 261; 260, 264; orbit at 4K (32 400) 89.3; 89.3, 91.8; 4K / 3M 265; 260, 261; 5120x2880 / 5M 383; 370, 373; orbit at 4961x3641 178;
// 180, 183; 8K / 8M 650; 652, 644; 110M pairs 596; 598, 600.  Over 28 frames of 14 000 to 105 000 tiles the three are within 1 % of
// each other on average, single ones within 7 %.
// False for the padding positions.
constexpr int kFineTiles = 28 << 10;
constexpr int block_log2_of(int tiles_x, int tiles_y) { return (long long)tiles_x * tiles_y < kFineTiles ? 2 : 3; }

constexpr long long positions_of(int tiles_x, int tiles_y)
{
    const int block_log2 = block_log2_of(tiles_x, tiles_y), size = 1 << block_log2;
    const long long blocks = (long long)((tiles_x + size - 1) / size) * ((tiles_y + size - 1) / size);
    return (blocks + 7) / 8 * 8 * (size * size);
}

constexpr bool tile_of_position(int group, int tiles_x, int tiles_y, int* tile_x, int* tile_y)
{
    const int block_log2 = block_log2_of(tiles_x, tiles_y), size = 1 << block_log2;
    const int xcd = group & 7, slot = group >> 3;
    const int blocks_x = (tiles_x + size - 1) >> block_log2;
    const int block = (slot >> (2 * block_log2)) * 8 + xcd, inner = slot & (size * size - 1);
    const int row = block / blocks_x;
    const int column = (block - row * blocks_x + ((blocks_x - 5) & 7) * row) % blocks_x;
    *tile_x = (column << block_log2) + (inner & (size - 1));
    *tile_y = (row << block_log2) + (inner >> block_log2);
    return *tile_x < tiles_x && *tile_y < tiles_y;
}

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
