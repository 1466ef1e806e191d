// What is known of a frame's tiles in front of its blend: their ranges, the ranking of a small frame's by the length of their lists, and the
// long lists of a large one.  The launches of render.hip find it in the sorted keys; a sort that is followed by the blend in the same call
// (fgs_sort_render) writes it from its own table of segments.
#pragma once

#include "fgs_internal.h"
#include "tile_order.h"

namespace fgs {

// The lists of a large frame that are long for it (see long_table) start first: one that starts late ends late, and the launch with
// it (8K / 8M: lists of 2400 entries that start after a third of the launch end 50 us behind everything else: blend 695 -> 639 us).  The launch that marks the
// ranges lists them, the first workgroups of the blend take them from there, and a tile that finds itself listed leaves itself to
// them.  A tile is looked for where it would be listed, so whatever the table holds every tile is blended, and what is no such
// tile is passed over: the table needs no initial value, a list it has no room for starts where it would otherwise.
// There are two tables: a launch that reads one clears the counts of the other one for the frame that follows.
constexpr int kLongShards = 32, kLongPerShard = 32;        // (of the places in a shard behind tile_ranges_sampled_kernel the first half is used)
struct LongLists {
    uint32_t count[kLongShards], tiles[kLongShards][kLongPerShard];
};
__device__ __forceinline__ uint32_t long_shard(uint32_t tile) { return (tile ^ (tile >> 5) ^ (tile >> 10)) % kLongShards; }

constexpr int kOrderCap = 8192;            // tiles that are ranked at most

// Where the launches of a sort write what they know of the tiles: pointers on the device, null where nothing is wanted.
struct TileNotes {
    int2* ranges;
    LongLists* longer;
    uint32_t num_tiles;
    int long_list;              // entries of the shortest list that is listed
};
struct TileRanking {
    uint32_t* order;            // kOrderCap ranks, then how many lists are shared out and from which length on
    int num_tiles, squares, simds;
};
struct FrameTables {
    TileNotes notes;
    TileRanking ranking;
};

// The range of a tile, as fgs_tile_ranges has it.
__device__ __forceinline__ int2 range_of(int lo, int hi) { return hi > lo ? make_int2(lo, hi) : make_int2(0, 0); }

// What one thread writes of a tile whose pairs are [lo, hi).
__device__ __forceinline__ void note_tile(const TileNotes& t, uint32_t tile, int lo, int hi)
{
    if (!t.ranges || tile >= t.num_tiles) return;
    t.ranges[tile] = range_of(lo, hi);
    if (t.longer && hi - lo >= t.long_list) {
        const uint32_t shard = long_shard(tile), at = atomicAdd(&t.longer->count[shard], 1u);
        if (at < (uint32_t)kLongPerShard) t.longer->tiles[shard][at] = tile;
    }
}

// From which length on a tile's list is shared out (see blend_kernel_shared): by what a SIMD walks of the
// whole frame, as the lists of 256 tiles spread over it say.  Lists are cut alike whether
// the tiles are ranked or not, so the image is the same.  Called by a whole wave.
template <class Length>
__device__ __forceinline__ int least_shared(Length length, int num_tiles, int squares, int simds)
{
    constexpr int kSamples = 256;
    uint32_t sum = 0;
#pragma unroll
    for (int k = 0; k < kSamples / kWave; k++) {
        sum += (uint32_t)max(0, length((int)((long long)(k * kWave + lane_id()) * num_tiles / kSamples)));
    }
    sum = (uint32_t)bcast_i((int)wave_inclusive_sum(sum), kWave - 1);
    const uint64_t each = (uint64_t)sum * (uint32_t)num_tiles / kSamples * (uint32_t)squares / (uint32_t)simds;
    return least_shared_of(each);
}

// Tiles of a small frame ranked by the length of their lists, longest first (in steps of kOrderStep;
// the order inside a step is whatever the atomics make it), and behind the ranking how many of them are shared out and from
// which length on.  Called by a workgroup of 1024 threads; s_count: kOrderBins words.
template <class Length>
__device__ __forceinline__ void rank_tiles(Length length, int num_tiles, uint32_t* __restrict__ tile_order, int squares, int simds, uint32_t* s_count)
{
    constexpr int kPerThread = kOrderCap / 1024;
    const int tid = threadIdx.x;
    if (tid < kOrderBins) s_count[tid] = 0;
    __syncthreads();
    uint32_t bin[kPerThread], slot[kPerThread];
#pragma unroll
    for (int k = 0; k < kPerThread; k++) {
        const int t = tid + k * 1024;
        bin[k] = 0; slot[k] = 0;
        if (t < num_tiles) {
            bin[k] = (uint32_t)order_bin(length(t));
            slot[k] = atomicAdd(&s_count[bin[k]], 1u);
        }
    }
    __syncthreads();
    if (tid < kWave) {
        // exclusive prefix over the bins, four per lane
        static_assert(kOrderBins == 4 * kWave, "four bins per lane");
        const uint32_t a = s_count[4 * tid], b = s_count[4 * tid + 1], c = s_count[4 * tid + 2], d = s_count[4 * tid + 3];
        const uint32_t all = a + b + c + d;
        uint32_t incl = all;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const uint32_t up = (uint32_t)__shfl_up((int)incl, o);
            if (tid >= o) incl += up;
        }
        const uint32_t excl = incl - all;
        s_count[4 * tid] = excl;
        s_count[4 * tid + 1] = excl + a;
        s_count[4 * tid + 2] = excl + a + b;
        s_count[4 * tid + 3] = excl + a + b + c;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPerThread; k++) {
        const int t = tid + k * 1024;
        if (t < num_tiles) tile_order[s_count[bin[k]] + slot[k]] = (uint32_t)t;
    }
    if (tid < kWave) {
        const int least = least_shared(length, num_tiles, squares, simds);
        if (tid == 0) {
            tile_order[kOrderCap] = s_count[first_bin_below(least)];
            tile_order[kOrderCap + 1] = (uint32_t)least;
        }
    }
}

} // namespace fgs
