// Device-wide stable sort of (u64 key, u32 value) pairs for gfx950 (wave64).
//
// Stands in for the cub::DeviceRadixSort::SortPairs call of FlashGS
// (csrc/cuda_rasterizer/sort.cu:28-44): ascending, stable, on key bits [0, 32 + tile_bits).
//
// The key is (tile id << 32 | depth bits), and what the renderer needs is every tile's pairs,
// contiguous and ordered by depth.  So the sort runs most-significant part first:
//
//  1. Partition by tile id: one stable counting pass per 8 bits of tile id (two passes for up to
//     65536 tiles; above that digits of 9 bits, so an 8K frame of 129 600 tiles still takes two).
//     A pass is count -> offsets -> scatter: `count_chunk_kernel` builds one digit histogram per
//     block of 4096 pairs (fewer on shorter lists) and the sums of every chunk of blocks,
//     `offsets_kernel` turns them into the exclusive start of every (block, digit) run, and
//     `scatter_kernel` ranks its block in LDS (wave64 ballot matching, so equal digits keep
//     their input order) and writes each run to its start.  A short list takes
//     count -> scatter.  Up to 8191 tiles and some millions of pairs the tile id is one digit instead (see tile_scatter_kernel).
//     No workgroup ever waits for another one.  With one or two passes the pairs leave the
//     partition as 64-bit words depth << 32 | value, the tile known from the place.
//  2. Sort every tile's segment by the 32 depth bits without touching memory in between: the
//     last scatter pass also tabulates where each tile id's segment begins (with more than two
//     passes `segment_starts_kernel` does, from the sorted keys), then segments are handled by
//     size class.  Up to 1024 pairs one wave holds a 32-bit word per pair, the upper bits of its depth in front of its place,
//     in registers and runs a merging network on them, then fetches the pairs in that order and puts the few that the
//     bits left out tell apart in order, or sorts again by those (the result is that of a stable sort by depth); lane exchanges inside a row of 16 lanes are
//     data-parallel-primitive moves.  Up to 4096 (4 waves), 8192 (8) and 16384 pairs (16) every wave
//     of a workgroup sorts its part like that and the parts are merged, the steps between two waves
//     through LDS.  Longer segments go
//     through stable 8-bit counting passes with a ping-pong copy in HBM, skipping a pass in which all
//     pairs share the digit.
//
// Bytes moved per pair with two partition passes of 8-bit digits: 8 (count) + 12 + 9 (scatter) + 1 + 9 + 8, and 8 + 12 for the
// segment sort of up to 1024 pairs: 67 (70 with 9-bit digits), against 8 + 6 * 24 = 152 for a six-pass LSD sort of 47 bits.  Segments of 1025 to
// 16384 pairs are read a second time, behind the merges; what sorts again is written and read twice more, and the longest segments are read twice and written once per counting pass.
#include "fgs_internal.h"
#include "sort.h"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace fgs {
namespace {

constexpr int kBins = 256;                      // counters of a counting pass inside a segment (8-bit digits)
constexpr int kSortBlock = 256;
constexpr int kXcds = 8;                        // accelerator dies of the device, workgroup i of a launch runs on die i % 8

// Shape of a partition pass: digits of kBitsT bits, kItemsT pairs per thread of a scatter workgroup of kThreadsT.
// Up to 65 536 tiles two passes of 8 bits do; above that (an 8K frame has 129 600) digits of 9 bits keep
// it at two passes up to 262 144 tiles.
// A scatter workgroup has sixteen waves with a few pairs per lane each, not four waves with sixteen: ranking 64 pairs is a
// chain of some hundred instructions that a wave goes through once per pair of its lanes, and with the one or two
// waves per SIMD that the LDS of a block of 4096 pairs left, a SIMD issued an instruction every four to seven cycles.
// Sort of the frame of 110M pairs 3160 -> 2690 us, 8K / 14.5M pairs 446 -> 416, 4K / 8M 216 -> 199, 1080p / 1.7M 98 -> 90,
// 720p / 0.2M 38 -> 31.  (Blocks of 2048 pairs lose 2 % on 4K and 8K, of 3072 and 5120 no difference to 4096, of
// 6144 to 8192 5 to 20 %: one workgroup per CU.)
template <int kBitsT, int kItemsT, int kThreadsT>
struct PassShape {
    static constexpr int kBits = kBitsT;
    static constexpr int kBinsP = 1 << kBitsT;
    static constexpr int kItems = kItemsT;                  // pairs per thread in scatter
    static constexpr int kThreads = kThreadsT;              // of a scatter workgroup
    static constexpr int kWaves = kThreadsT / kWave;
    static constexpr int kTile = kThreadsT * kItemsT;       // pairs per count/scatter workgroup
    static constexpr int kCountItems = kTile / kSortBlock;  // pairs per thread in count
    static constexpr int kPerThread = kBinsP / kSortBlock;  // digits per thread of a count row
    static constexpr int kDigits = kThreadsT < kBinsP ? kBinsP / kThreadsT : 1;     // digits per scatter thread that stands for digits
    static constexpr int kGroups = kThreadsT < kBinsP ? 1 : kThreadsT / kBinsP;     // scatter threads per digit
    static constexpr bool kAlone = false;
    static_assert(kBinsP % kSortBlock == 0 && kTile % kSortBlock == 0 && kTile <= 65535, "16-bit counts per wave and digit");
    static_assert(kThreadsT < kBinsP ? kBinsP % kThreadsT == 0 : kThreadsT % kBinsP == 0, "whole digits per thread, or whole groups of threads");
};
using Narrow = PassShape<8, 4, 1024>;
using Wide = PassShape<9, 4, 1024>;
constexpr int kNarrowMaxTileBits = 16;
constexpr int kWordsMaxTileBits = 18;           // two passes of Wide: up to here pairs are carried as words (Form::kWords)
// The 0.2M pairs of a 720p frame are 49 blocks of 4096, which would leave four CUs in five without one: shorter lists
// are cut into smaller blocks (0.2M pairs 36.7 us with 2048 a block, 30.6 with 1024; 0.4M 54.5 with 1024,
// 50 with 1536, 44 with 2048; 1.2M 83 with 4096, 79 with 2048; 1.7M 92.5 and 90; 0.1M on an 8K frame 78 and, with 1024, 64).
using Middle = PassShape<8, 2, 1024>;
using Short = PassShape<8, 1, 1024>;
using WideShort = PassShape<9, 1, 1024>;
constexpr int kShortPairs = 1 << 18;
// A list of one block counts its own digits (scatter_kernel's kAlone), and in few tiles one launch sorts segments of any length
// (segment_sort_alone_kernel): frame of 256x192 with 2.8k pairs, two launches less, 39.7 -> 35.1 us.
template <class Shape> struct Alone : Shape { static constexpr bool kAlone = true; };
constexpr int kAlonePairs = Narrow::kTile, kAloneIds = 1024;
constexpr int kMiddlePairs = 1 << 21;

// A list with at most this many histogram entries (256 blocks, or 128 with 9-bit digits) needs no launch that turns
// the histogram rows into starts: the scatter workgroups add the rows up themselves (0.4M pairs, 193 rows: 44 us against 50
// with that launch; 0.6M, 295 rows: 78 and 72).
constexpr int kMostRowWords = 65536;
constexpr int kMaxChunks = 256;

inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// Tile ids up to this count get a table of segment starts in the workspace; beyond it every
// segment workgroup searches for its own bounds.
constexpr uint32_t kMaxTableIds = 1u << 20;

// The ids of the longer segments are listed per size class in kListShards separate lists (each
// with its own counter, a workgroup appends to the list of its index modulo kListShards): one
// shared counter would serialise thousands of atomic additions on one address.
constexpr int kListShards = 32;
constexpr int kListClasses = 4;
static_assert(kListClasses * kListShards * 4 <= 512, "the list counters fit in the 512 bytes in front of the lists");

struct Workspace {
    size_t alt_keys, alt_values, hist, chunk_sums, seg_start, marks, seg_lists, total;
};

// Words of the workspace that the launches of one sort hand to each other.
constexpr int kMarkBeyond = 0;                  // one word per count workgroup of the first pass: some key differs from the first one above the sorted range
constexpr int kMarkByIndex = kMaxChunks;        // the same for the whole list: the launches behind the first scatter read this one
constexpr int kMarkAbove = kMarkByIndex + 1;    // the bits above the sorted range, the same in every key where that word is 0
constexpr int kMarkLowStart = kMaxChunks + 8;   // first index of every digit of the first of two passes
constexpr int kMarks = kMarkLowStart + 512;

struct PassGrid {
    int tiles, chunk, chunks;       // workgroups of a count/scatter launch; chunks of `chunk` histogram rows each
};

PassGrid pass_grid(int n, int tile)
{
    PassGrid g;
    g.tiles = (n + tile - 1) / tile;
    g.chunk = g.tiles > kMaxChunks ? (g.tiles + kMaxChunks - 1) / kMaxChunks : 1;       // one count workgroup each: about one per CU
    g.chunks = (g.tiles + g.chunk - 1) / g.chunk;
    return g;
}

// Sized for whichever pass shape the frame turns out to need (the tile count is not known here).
Workspace workspace_for(int n)
{
    Workspace w;
    // (monotone in n: a workspace sized for more pairs serves fewer)
    auto rows_of = [](auto shape, int pairs) {
        using Shape = decltype(shape);
        return (size_t)pass_grid(pairs, Shape::kTile).tiles * Shape::kBinsP;
    };
    const size_t hist = std::max({rows_of(Short(), std::min(n, kShortPairs)), rows_of(Middle(), std::min(n, kMiddlePairs)),
                                  rows_of(WideShort(), std::min(n, kShortPairs)), rows_of(Narrow(), n), rows_of(Wide(), n)});
    const size_t sums = (size_t)std::min(n, kMaxChunks) * Wide::kBinsP;
    w.alt_keys = 0;
    w.alt_values = align_up((size_t)n * 8, 256);
    w.hist = w.alt_values + align_up((size_t)n * 4, 256);
    w.chunk_sums = w.hist + hist * 4;
    w.seg_start = align_up(w.chunk_sums + sums * 4, 256);
    w.marks = w.seg_start + align_up(((size_t)kMaxTableIds + 1) * 4, 256);
    w.seg_lists = align_up(w.marks + kMarks * 4, 256);
    // counters (kListClasses * kListShards words), then per class kListShards lists, each able to
    // hold every segment of its class
    w.total = w.seg_lists + 512 + (size_t)kListShards * (((size_t)n / 512 + 2) + ((size_t)n / 1024 + 2) + ((size_t)n / 4096 + 2) +
                                                         ((size_t)n / 8192 + 2)) * 4;
    return w;
}

long long tiles_of(int width, int height, int block_x, int block_y)
{
    return (long long)((width + block_x - 1) / block_x) * ((height + block_y - 1) / block_y);
}

// What a partition pass reads and writes.
enum class Form {
    kPairs,         // keys and values as the caller has them
    kWords,         // depth << 32 | value, and of the tile field only the digit that the next pass needs (one or two bytes)
    kSegments,      // depth << 32 | value: the last pass, the segment a pair stands in is its tile
};

// The part of the tile field that the second of two passes sorts by.
template <class Shape>
using NextDigit = std::conditional_t<(Shape::kBits > 8), uint16_t, uint8_t>;

// ---- partition pass, step 1: hist[block][digit] ---------------------------------------------------

// The kCountItems digits of a thread, from keys (kSortBlock apart) or from the bytes or half words that the pass before left (consecutive
// ones, loaded together: the bytes behind the last digit are inside the buffer, their counts are not taken).
template <class Shape, class In>
struct Digits {
    static constexpr bool kKeys = sizeof(In) == 8;
    static constexpr int kItems = Shape::kCountItems;
    static constexpr int kWords = kKeys ? kItems : kItems * (int)sizeof(In) / 4;     // (of keys the upper halves alone)
    uint32_t w[kWords];

    __device__ __forceinline__ int index(int i, int tid) const { return kKeys ? i * kSortBlock + tid : tid * kItems + i; }

    __device__ __forceinline__ void load(const In* __restrict__ in, int base, int tid, int n)
    {
        if constexpr (kKeys) {
#pragma unroll
            for (int i = 0; i < kItems; i++) {
                const int idx = base + i * kSortBlock + tid;
                w[i] = idx < n ? ((const uint32_t*)in)[2 * (size_t)idx + 1] : 0u;
            }
        } else {
            const int first = base + tid * kItems;
            constexpr int kVector = kWords < 4 ? kWords : 4;
            typedef uint32_t Vector __attribute__((ext_vector_type(kVector)));
            const Vector* const at = (const Vector*)(in + first);
#pragma unroll
            for (int v = 0; v < kWords / kVector; v++) {
                Vector x = 0;
                if (first + v * (kItems / (kWords / kVector)) < n) x = at[v];
#pragma unroll
                for (int j = 0; j < kVector; j++) w[v * kVector + j] = kVector == 1 ? ((const uint32_t*)&x)[0] : x[j];
            }
        }
    }
    __device__ __forceinline__ uint32_t digit(int i, int shift, uint32_t mask) const
    {
        if constexpr (kKeys) return (w[i] >> shift) & mask;
        constexpr int kPer = 4 / (sizeof(In) < 4 ? (int)sizeof(In) : 4);
        return (w[i / kPer] >> (i % kPer * (32 / kPer))) & mask;
    }
    __device__ __forceinline__ uint32_t field(int i) const { return kKeys ? w[i] : 0u; }
};

// The tile field of the list's first key, whose bits above the sorted range are those of every key unless marked (kMarkBeyond).
template <class In>
__device__ __forceinline__ uint32_t first_field(const In* in)
{
    if constexpr (sizeof(In) == 8) return (uint32_t)(in[0] >> 32);
    return 0;
}

template <class Shape, class In>
__global__ __launch_bounds__(kSortBlock) void count_kernel(const In* __restrict__ in, int n,
                                                           int shift, int nbits, uint32_t* __restrict__ hist,
                                                           uint32_t above, uint32_t* __restrict__ beyond,
                                                           uint32_t* __restrict__ seg_counts)
{
    constexpr int kB = Shape::kBinsP;
    __shared__ uint32_t h[kB];
    __shared__ uint32_t s_beyond;
    const int tid = threadIdx.x;
    if (seg_counts) {       // the last pass also clears what the segment launches append to
        const uint32_t gid = blockIdx.x * kSortBlock + tid;
        if (gid < (uint32_t)(kListClasses * kListShards)) seg_counts[gid] = 0;
    }
#pragma unroll
    for (int q = 0; q < Shape::kPerThread; q++) h[q * kSortBlock + tid] = 0;
    if (tid == 0) s_beyond = 0;
    __syncthreads();
    const uint32_t mask = (1u << nbits) - 1u;
    const int base = blockIdx.x * Shape::kTile;
    Digits<Shape, In> digits;
    digits.load(in, base, tid, n);
    uint32_t seen = 0;
    const uint32_t field_of_first = beyond ? first_field(in) : 0u;
#pragma unroll
    for (int i = 0; i < Shape::kCountItems; i++) {
        if (base + digits.index(i, tid) < n) atomicAdd(&h[digits.digit(i, shift, mask)], 1u);
        if (base + digits.index(i, tid) < n) seen |= digits.field(i) ^ field_of_first;
    }
    if (beyond && (seen & above) != 0) s_beyond = 1;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Shape::kPerThread; q++)
        hist[(size_t)blockIdx.x * kB + q * kSortBlock + tid] = h[q * kSortBlock + tid];
    if (beyond && tid == 0) beyond[blockIdx.x] = s_beyond;
}

// The same for a list of more than kMostRowWords histogram entries: one workgroup counts a whole chunk of
// `chunk` consecutive blocks, blockDim.x / kSortBlock of them at a time, and so also has the
// chunk's digit sums, which the offsets launch needs (a launch of their own would read the rows
// back just to add them up).  The digits of the next blocks are requested before those at hand are counted: second count of 110M pairs 76 -> 66 us, of 14.3M
// 17.4 -> 15.3, first count of 4.9M 12.8 -> 11.3.  The first count of 110M pairs stays at 205: behind preprocess, whose pairs are still on their way to memory, no
// order of its reads changes it (on a list that rests the same change is 251 -> 189, and a plain read of the 0.87 GB 138).
constexpr int kCountGroups = 4;

template <class Shape, class In>
__global__ __launch_bounds__(kCountGroups * kSortBlock) void count_chunk_kernel(
    const In* __restrict__ in, int n, int shift, int nbits, uint32_t* __restrict__ hist,
    int tiles, int chunk, uint32_t* __restrict__ chunk_sums,
    uint32_t above, uint32_t* __restrict__ beyond, uint32_t* __restrict__ seg_counts)
{
    constexpr int kB = Shape::kBinsP, kPer = Shape::kPerThread;
    __shared__ uint32_t h[2][kCountGroups][kB];         // in turn: while the one is written out the other counts
    __shared__ uint32_t s_beyond;
    const int tid = threadIdx.x % kSortBlock, group = threadIdx.x / kSortBlock;
    const int groups = (int)blockDim.x / kSortBlock;
    if (seg_counts) {       // the last pass also clears what the segment launches append to
        const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
        if (gid < (uint32_t)(kListClasses * kListShards)) seg_counts[gid] = 0;
    }
    const uint32_t mask = (1u << nbits) - 1u;
    const int t0 = blockIdx.x * chunk, t1 = min(tiles, t0 + chunk);
    Digits<Shape, In> next = {};
    if (t0 + group < t1) next.load(in, (t0 + group) * Shape::kTile, tid, n);
    uint32_t sum[kPer];
#pragma unroll
    for (int q = 0; q < kPer; q++) { sum[q] = 0; h[0][group][q * kSortBlock + tid] = 0; h[1][group][q * kSortBlock + tid] = 0; }
    if (threadIdx.x == 0) s_beyond = 0;
    __syncthreads();
    uint32_t seen = 0;
    const uint32_t field_of_first = beyond ? first_field(in) : 0u;
    int turn = 0;
    for (int first = t0; first < t1; first += groups, turn ^= 1) {      // the same trips for every group
        const int row = first + group;
        const Digits<Shape, In> digits = next;
        if (row + groups < t1) next.load(in, (row + groups) * Shape::kTile, tid, n);
        if (row < t1) {
            const int base = row * Shape::kTile;
#pragma unroll
            for (int i = 0; i < Shape::kCountItems; i++) {
                if (base + digits.index(i, tid) < n) atomicAdd(&h[turn][group][digits.digit(i, shift, mask)], 1u);
                if (base + digits.index(i, tid) < n) seen |= digits.field(i) ^ field_of_first;
            }
        }
        __syncthreads();
        if (row < t1) {
#pragma unroll
            for (int q = 0; q < kPer; q++) {
                const uint32_t c = h[turn][group][q * kSortBlock + tid];
                h[turn][group][q * kSortBlock + tid] = 0;       // read and cleared by the same thread, a barrier in front of the next counts
                hist[(size_t)row * kB + q * kSortBlock + tid] = c;
                sum[q] += c;
            }
        }
    }
    __syncthreads();
    if (beyond && (seen & above) != 0) s_beyond = 1;
#pragma unroll
    for (int q = 0; q < kPer; q++) h[0][group][q * kSortBlock + tid] = sum[q];
    __syncthreads();
    if (group == 0) {
#pragma unroll
        for (int q = 0; q < kPer; q++) {
            uint32_t total = 0;
            for (int g = 0; g < groups; g++) total += h[0][g][q * kSortBlock + tid];
            chunk_sums[(size_t)blockIdx.x * kB + q * kSortBlock + tid] = total;
        }
    }
    if (beyond && threadIdx.x == 0) beyond[blockIdx.x] = s_beyond;
}

// ---- step 2: exclusive start of every (block, digit) run ----------------------------------------
// start[b][d] = sum of hist[*][d' < d] + sum of hist[b' < b][d]   (digit-major, then block)

// One workgroup per chunk.  Every one of them adds up the sums of all chunks, four digits a thread and eight rows a trip to memory: two trips for 256 chunks of
// 256 digits and four with 512, where a digit a thread took four and eight (8K / 14.3M pairs 14.1 -> 11.3 us a launch, 110M 29.6 -> 25.4, 4K / 8M 8.1 -> 8.0).  (Sixteen rows a trip, or the chunk's own rows requested in front of the
// sums, are no faster.)
constexpr int kOffsetThreads = 1024;

template <class Shape>
__global__ __launch_bounds__(kOffsetThreads) void offsets_kernel(uint32_t* __restrict__ hist, int tiles, int chunk,
                                                                 const uint32_t* __restrict__ chunk_sums, int chunks,
                                                                 uint32_t* marks)       // of the first pass, else null
{
    typedef uint32_t Four __attribute__((ext_vector_type(4)));
    constexpr int kB = Shape::kBinsP, kQuads = kB / 4, kGroups = kOffsetThreads / kQuads, kSumsAtOnce = 8, kRowsAtOnce = 16;
    __shared__ Four s_total[kGroups][kQuads], s_before[kGroups][kQuads];
    __shared__ uint32_t s_wave[kB / kWave];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int mine = (int)blockIdx.x;
    if (marks && mine == 0) {       // one word out of the count workgroups' words
        uint32_t seen = 0;
        for (int c = tid; c < chunks; c += kOffsetThreads) seen |= marks[kMarkBeyond + c];
        const int any = __syncthreads_or(seen != 0);
        if (tid == 0) marks[kMarkByIndex] = any ? 1u : 0u;
    }
    {
        const int quad = tid & (kQuads - 1), group = tid / kQuads;
        Four total = 0, before = 0;
        for (int c0 = group * kSumsAtOnce; c0 < chunks; c0 += kSumsAtOnce * kGroups) {
            Four v[kSumsAtOnce];
#pragma unroll
            for (int j = 0; j < kSumsAtOnce; j++) {
                v[j] = 0;
                if (c0 + j < chunks) v[j] = ((const Four*)chunk_sums)[(size_t)(c0 + j) * kQuads + quad];
            }
#pragma unroll
            for (int j = 0; j < kSumsAtOnce; j++) {
                if (c0 + j < mine) before += v[j];
                total += v[j];
            }
        }
        s_total[group][quad] = total;
        s_before[group][quad] = before;
    }
    __syncthreads();
    uint32_t total = 0, before = 0, incl = 0;
    if (tid < kB) {
#pragma unroll
        for (int g = 0; g < kGroups; g++) { total += ((const uint32_t*)s_total[g])[tid]; before += ((const uint32_t*)s_before[g])[tid]; }
        // exclusive scan of the digit totals over the digits
        incl = wave_inclusive_sum(total);
        if (lane == kWave - 1) s_wave[wave] = incl;
    }
    __syncthreads();
    if (tid >= kB) return;
    uint32_t run = incl - total + before;
    for (int w = 0; w < wave; w++) run += s_wave[w];
    const int t0 = mine * chunk, t1 = min(tiles, t0 + chunk);
    for (int row = t0; row < t1; row += kRowsAtOnce) {
        uint32_t c[kRowsAtOnce];
#pragma unroll
        for (int j = 0; j < kRowsAtOnce; j++) c[j] = row + j < t1 ? hist[(size_t)(row + j) * kB + tid] : 0u;
#pragma unroll
        for (int j = 0; j < kRowsAtOnce; j++) {
            if (row + j < t1) hist[(size_t)(row + j) * kB + tid] = run;
            run += c[j];
        }
    }
}


// ---- step 3: stable scatter ---------------------------------------------------------------------------

// With at most two passes the pairs leave the first one as 64-bit words depth << 32 | value beside the one digit that the
// second pass needs, and the last one as words alone: the segment sort works on such words anyhow and knows the
// tile from the segment, and it writes the pairs in full.  10 bytes (9 with 8-bit digits) in place of 12 are written, 8 in
// place of 12 by the last pass, and the second count reads a byte or two per pair in place of its key.  With pairs carried
// in full, and nine instructions per bit of the ranking in place of four: 8K frame of 110M pairs scatter 541 + 533 -> 519 + 425 us,
// second count 213 -> 79; 4K / 8M 48 + 46 -> 43 + 40, 14.4 -> 8; 8K / 14.5M 82 + 83 -> 80 + 71, 27 -> 18.
// A list whose keys differ in bits above the sorted range carries every pair's index in place of its value (the partition is stable, so
// equal depths keep their order by it as well), and the segment sort fetches the pairs from the input.  (8M pairs of a 4K frame 145 -> 417 us;
// bits that every key has in common there are set again by the segment sort, 145.)
//
// The last pass of at most two (Form::kSegments) also writes the table of segment starts,
// seg_start[v] = first index of the output whose tile field is >= v, v in [0, ids], ids = 2^(bits of
// the tile field).  The input of that pass is ordered by the low part of the tile field (the bits
// below this pass's digit), so the first pair with low part >= L lies in exactly one workgroup's
// block, and that workgroup writes the entries (d, L) of every digit d: the destination of its
// first pair with digit d and low part >= L, or, if it has none, the end of its run of digit d,
// which is where the next workgroup's run of d begins.  Every entry has one writer, empty ids
// included, and no launch has to read the keys again.  Where the low parts begin is what the first pass
// began with, left by its workgroup of block 0.
// kAlone: the whole list is one block, whose own counts say where its digits start: no launch counts them.
template <class Shape, Form kIn, Form kOut, bool kAlone = false>
__global__ __launch_bounds__(Shape::kThreads) void scatter_kernel(
    const uint64_t* __restrict__ keys_in, const void* __restrict__ values_in,       // the digits of Form::kWords stand where the values do
    uint64_t* __restrict__ keys_out, void* __restrict__ values_out,
    int n, int shift, int nbits, int low_bits,   // kSegments: low_bits tile bits below this pass's digit
    const uint32_t* __restrict__ start,          // [blocks][bins] from offsets_kernel, or ...
    int raw_rows,                                // ... if > 0, the raw_rows histogram rows themselves (a short list)
    uint32_t above,                              // the bits of the tile field above the sorted range
    uint32_t* marks, const uint32_t* beyond, int beyond_rows,       // beyond_rows > 0: the first pass
    int* __restrict__ seg_start)                 // kSegments: [2^(low_bits + nbits) + 1]
{
    constexpr bool kTable = kOut == Form::kSegments;
    constexpr int kB = Shape::kBinsP, kItems = Shape::kItems, kTile = Shape::kTile, kPer = Shape::kDigits;
    constexpr int kThreads = Shape::kThreads, kWaves = Shape::kWaves;
    typedef NextDigit<Shape> Next;
    // what is staged beside a word: the tile field (pairs: all of it, else up to 16 or 18 bits)
    typedef std::conditional_t<kOut == Form::kPairs || (Shape::kBits > 8), uint32_t, uint16_t> Field;
    // per-wave digit counts, then per-wave digit offsets: at most kTile, so 16 bits do, and with
    // them the workgroup's LDS stays under half of the CU's
    __shared__ __align__(4) uint16_t s_count[kWaves][kB];
    __shared__ uint16_t s_bin_start[kB];              // where each digit starts in the ranked block
    __shared__ uint32_t s_global[kB];                 // destination of ranked slot p with digit d: s_global[d] + p
    constexpr int kScanWaves = kB / kWave;           // waves' worth of digits
    __shared__ uint32_t s_wave_sum[kScanWaves];
    __shared__ uint64_t s_words[kTile];
    __shared__ Field s_field[kTile];
    __shared__ int s_low_start[kIn == Form::kWords ? kB : 1];

    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = tid / kWave;
    const uint32_t mask = (1u << nbits) - 1u;
    // Workgroups go round-robin to the 8 XCDs, each with an L2 of its own.  Every XCD takes a
    // contiguous range of blocks: the runs that neighbouring blocks write for one digit are
    // neighbours in memory, and the cache line where two of them meet is then completed in one
    // L2 instead of being written out in parts by two (first pass at 4K: 62 -> 51 us).
    const int xcd = (int)blockIdx.x % kXcds, per = (int)gridDim.x / kXcds, rest = (int)gridDim.x % kXcds;
    const int tile = xcd * per + min(xcd, rest) + (int)blockIdx.x / kXcds;
    const int tile_base = tile * kTile;
    const int in_tile = min(kTile, n - tile_base);

    // wave w owns slots [w*64*kItems, (w+1)*64*kItems) of the block, item-major; everything is
    // requested before the first use so the latencies overlap
    uint64_t word[kItems];          // depth << 32 | value
    uint32_t field[kItems];         // (kWords: this pass's digit)
    uint32_t slot[kItems];
    if constexpr (kIn == Form::kWords) {
#pragma unroll
        for (int i = 0; i < kItems; i++) {
            const int off = wave * (kWave * kItems) + i * kWave + lane;
            word[i] = off < in_tile ? keys_in[tile_base + off] : ~0ull;
        }
#pragma unroll
        for (int i = 0; i < kItems; i++) {
            const int off = wave * (kWave * kItems) + i * kWave + lane;
            field[i] = off < in_tile ? (uint32_t)((const Next*)values_in)[tile_base + off] : ~0u;
        }
    } else {
        uint32_t val[kItems];
#pragma unroll
        for (int i = 0; i < kItems; i++) {
            const int off = wave * (kWave * kItems) + i * kWave + lane;
            word[i] = off < in_tile ? keys_in[tile_base + off] : ~0ull;
        }
#pragma unroll
        for (int i = 0; i < kItems; i++) {
            const int off = wave * (kWave * kItems) + i * kWave + lane;
            val[i] = off < in_tile ? ((const uint32_t*)values_in)[tile_base + off] : 0u;
        }
        bool by_index = false;
        if constexpr (kAlone) {
            uint32_t seen = 0;
            const uint32_t field_of_first = first_field(keys_in);
#pragma unroll
            for (int i = 0; i < kItems; i++)
                if (wave * (kWave * kItems) + i * kWave + lane < in_tile) seen |= ((uint32_t)(word[i] >> 32) ^ field_of_first) & above;
            by_index = __syncthreads_or(seen != 0) != 0;
            if (tid == 0) { marks[kMarkByIndex] = by_index ? 1u : 0u; marks[kMarkAbove] = field_of_first & above; }
        } else if (beyond_rows > 0) {
            uint32_t seen = 0;
            for (int r = lane; r < beyond_rows; r += kWave) seen |= beyond[r];
            by_index = ballot(seen != 0) != 0;
            if (blockIdx.x == 0 && tid == 0) { marks[kMarkByIndex] = by_index ? 1u : 0u; marks[kMarkAbove] = first_field(keys_in) & above; }
        }
#pragma unroll
        for (int i = 0; i < kItems; i++) {
            const int off = wave * (kWave * kItems) + i * kWave + lane;
            field[i] = (uint32_t)(word[i] >> 32);
            word[i] = (word[i] << 32) | (by_index ? (uint32_t)(tile_base + off) : val[i]);
        }
    }
    // A thread stands for the digits tid, tid + kThreads, ...; with more threads than digits the first kB do.
    const bool has_digits = tid < kB;
    uint32_t my_start[kPer] = {};
    if constexpr (kAlone) {
        // (known behind the ranking)
    } else if (raw_rows == 0) {
        if (has_digits) {
#pragma unroll
            for (int q = 0; q < kPer; q++) my_start[q] = start[(size_t)tile * kB + q * kThreads + tid];
        }
    } else {
        // A list of at most kMostRowWords histogram entries: every workgroup adds up the histogram rows itself
        // (the digit totals, and what the blocks in front of it hold of each digit), which
        // saves the launch that would do it.
        uint32_t total[kPer], before[kPer], incl[kPer];
        const int group = tid / kB;
#pragma unroll
        for (int q = 0; q < kPer; q++) {
            const int d = (q * kThreads + tid) % kB;
            total[q] = 0; before[q] = 0;
#pragma unroll 16
            for (int b = group; b < raw_rows; b += Shape::kGroups) {
                const uint32_t c = start[(size_t)b * kB + d];
                total[q] += c;
                before[q] += b < tile ? c : 0u;
            }
        }
        if constexpr (Shape::kGroups > 1) {
            uint32_t* const s_part = (uint32_t*)s_words;
            static_assert(sizeof(uint32_t) * 2 * Shape::kGroups * kB <= sizeof(uint64_t) * kTile, "the partial sums fit in the space of the words");
            s_part[2 * tid] = total[0];
            s_part[2 * tid + 1] = before[0];
            __syncthreads();
            if (has_digits) {
#pragma unroll
                for (int g = 1; g < Shape::kGroups; g++) {
                    total[0] += s_part[2 * (g * kB + tid)];
                    before[0] += s_part[2 * (g * kB + tid) + 1];
                }
            }
        }
        if (has_digits) {
#pragma unroll
            for (int q = 0; q < kPer; q++) {
                incl[q] = wave_inclusive_sum(total[q]);
                if (lane == kWave - 1) s_wave_sum[q * kWaves + wave] = incl[q];
            }
        }
        __syncthreads();
        if (has_digits) {
#pragma unroll
            for (int q = 0; q < kPer; q++) {
                uint32_t digit_base = incl[q] - total[q];
#pragma unroll
                for (int w = 0; w < kScanWaves; w++)
                    if (w < q * kWaves + wave) digit_base += s_wave_sum[w];
                my_start[q] = digit_base + before[q];
            }
        }
    }
    {
        uint32_t* const words = (uint32_t*)&s_count[0][0];
#pragma unroll
        for (int w = 0; w < kWaves * kB / 2; w += kThreads)
            if (w + tid < kWaves * kB / 2) words[w + tid] = 0;
    }
    if (kOut == Form::kWords && !kAlone && tile == 0 && has_digits) {
#pragma unroll
        for (int q = 0; q < kPer; q++) marks[kMarkLowStart + q * kThreads + tid] = my_start[q];
    }
    if (kIn == Form::kWords) {
        for (int l = tid; l < kB; l += kThreads) s_low_start[l] = (int)marks[kMarkLowStart + l];
    }
    __syncthreads();
    // The low parts L whose first pair (the first of the input with low part >= L) lies in this
    // block: those above the low part of the pair in front of the block, up to that of the
    // block's last pair; the last block also takes the ones no pair reaches.
    // (a pair's low part: the last one that begins at its index or in front of it)
    auto low_part = [&](int index) {
        int low = 0;
#pragma unroll
        for (int step = kB / 2; step > 0; step >>= 1)
            if (s_low_start[low + step] <= index) low += step;
        return low;
    };
    int own_lo = 0, own_hi = -1;
    if constexpr (kIn == Form::kWords) {
        own_lo = tile > 0 ? low_part(tile_base - 1) + 1 : 0;
        own_hi = tile == (int)gridDim.x - 1 ? kB - 1 : low_part(tile_base + in_tile - 1);
    } else if (kTable) {
        own_hi = tile == 0 ? 0 : -1;
    }

    // rank inside the wave: lanes with equal digits find each other with one ballot per digit bit.  The pass issues instructions
    // 77 % of its time on long lists, most of them here: a bit is taken as 0 or all ones, so that four instructions a bit do (the
    // field, the comparison, and the peers of either half as one three-operand function), and every lane reads its
    // digit's counter itself in place of a move from the lane that will update it.
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        const int off = wave * (kWave * kItems) + i * kWave + lane;
        const bool valid = off < in_tile;
        const uint32_t d = (field[i] >> shift) & mask;
        const uint64_t all = ballot(valid);
        uint32_t peers_lo = (uint32_t)all, peers_hi = (uint32_t)(all >> 32);
#pragma unroll
        for (int b = 0; b < Shape::kBits; b++) {
            uint32_t bit = (uint32_t)__builtin_amdgcn_sbfe((int)d, b, 1);
            asm("" : "+v"(bit));                                                            // one instruction, or every use makes a field of its own
            const uint64_t with_bit = ballot(bit != 0);
            peers_lo = __builtin_amdgcn_bitop3_b32(peers_lo, (uint32_t)with_bit, bit, 0x90);          // peers & ~(with_bit ^ bit)
            peers_hi = __builtin_amdgcn_bitop3_b32(peers_hi, (uint32_t)(with_bit >> 32), bit, 0x90);
        }
        const uint32_t below = __builtin_amdgcn_mbcnt_hi(peers_hi, __builtin_amdgcn_mbcnt_lo(peers_lo, 0u));
        const uint32_t before = s_count[wave][d];
        if (valid && below == 0)        // the lowest lane of each group updates the wave's counter
            s_count[wave][d] = (uint16_t)(before + (uint32_t)__popc(peers_lo) + (uint32_t)__popc(peers_hi));
        slot[i] = before + below;
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();

    // digit totals of the block; per-wave offsets inside each digit.  A thread stands for the
    // digits tid, tid + 256, ...; the scan runs over the digits in their order.
    uint32_t total[kPer] = {}, incl[kPer] = {};
    if (has_digits) {
#pragma unroll
        for (int q = 0; q < kPer; q++) {
            const int d = q * kThreads + tid;
#pragma unroll
            for (int w = 0; w < kWaves; w++) {
                const uint32_t c = s_count[w][d];
                s_count[w][d] = (uint16_t)total[q];
                total[q] += c;
            }
            incl[q] = wave_inclusive_sum(total[q]);
            if (lane == kWave - 1) s_wave_sum[q * kWaves + wave] = incl[q];
        }
    }
    __syncthreads();
    if (has_digits) {
#pragma unroll
        for (int q = 0; q < kPer; q++) {
            const int d = q * kThreads + tid;
            uint32_t before_wave = 0;
#pragma unroll
            for (int w = 0; w < kScanWaves; w++)
                if (w < q * kWaves + wave) before_wave += s_wave_sum[w];
            const uint32_t bin_start = before_wave + incl[q] - total[q];
            s_bin_start[d] = (uint16_t)bin_start;
            if constexpr (kAlone) {
                my_start[q] = bin_start;
                if (kOut == Form::kWords) marks[kMarkLowStart + d] = bin_start;
            }
            s_global[d] = my_start[q] - bin_start;
        }
    }
    __syncthreads();

    // move the pairs to their ranked slots in LDS
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        const int off = wave * (kWave * kItems) + i * kWave + lane;
        if (off < in_tile) {
            const uint32_t dg = (field[i] >> shift) & mask;
            const uint32_t p = (uint32_t)s_bin_start[dg] + s_count[wave][dg] + slot[i];
            s_words[p] = word[i];
            // the whole tile field again where the table needs it
            if (kIn == Form::kWords && own_lo <= own_hi) field[i] = (dg << low_bits) | (uint32_t)low_part(tile_base + off);
            s_field[p] = (Field)field[i];
        }
    }
    __syncthreads();
    const bool whole_fields = kIn != Form::kWords || own_lo <= own_hi;
    const int field_shift = kIn == Form::kWords && whole_fields ? low_bits : shift;

    // write out: neighbouring threads hold neighbouring ranked slots.  All LDS reads first (a slot
    // past the end reads the last pair and stores nothing), so their latencies overlap.
    {
        uint64_t out_word[kItems];
        uint32_t out_field[kItems], out_at[kItems];
#pragma unroll
        for (int i = 0; i < kItems; i++) {
            const int p = min(i * kThreads + tid, in_tile - 1);
            out_word[i] = s_words[p];
            out_field[i] = s_field[p];
        }
#pragma unroll
        for (int i = 0; i < kItems; i++)
            out_at[i] = s_global[(out_field[i] >> field_shift) & mask] + (uint32_t)(i * kThreads + tid);
#pragma unroll
        for (int i = 0; i < kItems; i++) {
            if (i * kThreads + tid < in_tile) {
                if constexpr (kOut == Form::kPairs) {
                    keys_out[out_at[i]] = ((uint64_t)out_field[i] << 32) | (out_word[i] >> 32);
                    ((uint32_t*)values_out)[out_at[i]] = (uint32_t)out_word[i];
                } else {
                    keys_out[out_at[i]] = out_word[i];
                    if (kOut == Form::kWords) ((Next*)values_out)[out_at[i]] = (Next)(out_field[i] >> Shape::kBits);
                }
            }
        }
    }
    if (kTable) {
        if (own_lo <= own_hi) {
            const uint32_t low_mask = (1u << low_bits) - 1u;
            // the first pair of digit d with a low part >= L, for every owned L up to its own
            // (a loop of its own: in the one above the LDS reads of all slots are in flight together)
#pragma unroll 4
            for (int i = 0; i < kItems; i++) {
                const int p = i * kThreads + tid;
                if (p >= in_tile) break;
                const uint32_t f = s_field[p];
                const uint32_t d = (f >> low_bits) & mask;
                const int low = (int)(f & low_mask);
                int prev = own_lo - 1;
                if (p > (int)s_bin_start[d]) prev = (int)(s_field[p - 1] & low_mask);
                for (int l = max(prev + 1, own_lo); l <= low; l++)
                    seg_start[(d << low_bits) | (uint32_t)l] = (int)(s_global[d] + (uint32_t)p);
            }
            // owned low parts above the last pair of a digit's run: the end of the run
#pragma unroll
            for (int q = 0; q < kPer; q++) {
                const uint32_t d = (uint32_t)(q * kThreads + tid);
                if (d > mask) continue;         // (d is below kB then, a digit of this thread)
                int last = own_lo - 1;
                if (total[q]) last = (int)(s_field[(uint32_t)s_bin_start[d] + total[q] - 1u] & low_mask);
                const int end = (int)(my_start[q] + total[q]);
                for (int l = max(last + 1, own_lo); l <= own_hi; l++) seg_start[(d << low_bits) | (uint32_t)l] = end;
            }
        }
        if (tile == 0 && tid == 0) seg_start[(size_t)1 << (low_bits + nbits)] = n;
    }
}

// ---- the partition in one pass ---------------------------------------------------------------------
//
// In frames of up to 2^kOnePassBits tile ids, and lists that are not too long for them, the whole tile id is one digit: `tile_count_kernel` writes
// a row of counts per block, 16 bits for every tile id, `tile_offsets_kernel` turns every column of the rows into what the blocks in front
// hold of that tile, and `tile_scatter_kernel` sorts its block by tile id in LDS (two stable passes, seven bits first) and writes every pair's
// word to its place.  The pairs travel once and there are three launches, where two passes of 8 bits take four to six, each of which lasts 3 to 14 us on
// such a list whatever it moves: 3 + 4 + 8 us for 22 in all on 0.2M pairs of a 720p frame, 5 + 8 + 21 for 52 on 1.7M of a 1080p frame (that one reads 36 MB, of which
// 14 are offsets, and writes 16 for 14 in runs of one or two pairs).  The whole sort, two passes -> one: 3600 tiles 0.1M pairs 27 -> 22 us, 0.4M 41 -> 35,
// 1.6M 97 -> 77, 6.4M 275 -> 255; 8160 tiles 0.1M 28 -> 25, 0.8M 59 -> 48, 1.6M 78 -> 62, 3.2M 121 -> 113; 300 tiles 25k 27 -> 22, 0.8M 117 -> 96.
// A block's rows cost 6 bytes per tile id, so it stops paying where blocks x ids do: 8160 tiles 6.4M pairs 170 -> 180 us, 14 400 tiles 0.2M 32 -> 34, 0.8M
// 53 -> 48, 3.2M 100 -> 133.
// (Instead of the two passes in LDS, pairs that put their places down by tile and count the smaller ones there, words written from
// registers in any order: the scatter 21 -> 28 us, 12 -> 18 where some tiles are crowded.  Counters in memory in place of the rows, by atomic additions
// of a block's counts and of bases taken from them: 0.4M and 1.7M pairs 17 and 45 us in all for 20 and 34, and an order to be mended behind it.)
// With few ids the rows are many, and it still pays at the longest list that has any: 300 tiles 20M pairs 1574 -> 1520 us, 60M 4982 -> 4677 (14 649 rows of 512), 1000 tiles
// 16.5M 806 -> 748, 2048 tiles 16M 376 -> 373, 3600 tiles 8.3M 200 -> 181.
// Rows and offsets stand in the space of the copy that longer segments go through later, or, where that is too small, behind what the sort needs, in whatever more
// space the caller has passed (with neither, larger blocks or two passes: see kOnePassShort).
constexpr int kOnePassBits = 13, kOnePassIds = 1 << kOnePassBits, kOnePassLeastBits = 9;
constexpr int kOnePassThreads = 1024, kOnePassWaves = kOnePassThreads / kWave;
constexpr int kOnePassLow = 7;                  // bits of the tile id that the first sort of a block takes
// Blocks of 2048 pairs up to this many pairs, of 4096 above: 3600 tiles 0.2M pairs 25 and 28 us, 0.8M 50 and 48; 8160 tiles 0.2M 26 and 28, 0.4M 32 and 31, 1.6M 73 and 62.
// (Of 8192: 0.2M 33, 1.7M 1 % more.)
// The rows of blocks of 2048 pairs and 8192 ids are 24 bytes a pair, twice the copy: a caller with no space to spare has blocks of 4096 there.  5700 tiles, 0.1M pairs: 23.3
// us, 26.0 without, 27.1 by two passes; 8160 tiles 24.7, 27.5, 28.3; 0.4M 30.8, 30.7, 33.5.  With 4096 ids there is room as it is.
constexpr int kOnePassShort = 1 << 19;
constexpr size_t kOnePassCells = (size_t)1 << 23;       // the most cells of rows: 4.2M pairs with 8192 ids, 8.4M with 4096

// rows[block][tile]: 16-bit counts, two in a word.
template <int kItems>
__global__ __launch_bounds__(kOnePassThreads) void tile_count_kernel(const uint64_t* __restrict__ keys, int n, uint32_t ids,
                                                                     uint32_t* __restrict__ rows, uint32_t* __restrict__ beyond,
                                                                     uint32_t* __restrict__ seg_counts)
{
    static_assert(kOnePassThreads * kItems <= 65535, "16-bit counts");
    __shared__ uint32_t s_counts[kOnePassIds / 2];
    __shared__ uint32_t s_beyond;
    const int tid = threadIdx.x;
    if (blockIdx.x == 0 && tid < kListClasses * kListShards) seg_counts[tid] = 0;       // what the segment launches append to
    uint32_t field[kItems];
    const int base = (int)blockIdx.x * (kOnePassThreads * kItems) + tid;
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        field[i] = 0;
        if (base + i * kOnePassThreads < n) field[i] = ((const uint32_t*)keys)[2 * (size_t)(base + i * kOnePassThreads) + 1];
    }
    const uint32_t field_of_first = first_field(keys);
    for (uint32_t t = tid; t < ids / 2; t += kOnePassThreads) s_counts[t] = 0;
    if (tid == 0) s_beyond = 0;
    __syncthreads();
    uint32_t seen = 0;
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        if (base + i * kOnePassThreads < n) {
            const uint32_t tile = field[i] & (ids - 1u);
            atomicAdd(&s_counts[tile >> 1], tile & 1u ? 0x10000u : 1u);
            seen |= field[i] ^ field_of_first;
        }
    }
    if ((seen & ~(ids - 1u)) != 0) s_beyond = 1;
    __syncthreads();
    for (uint32_t t = tid; t < ids / 2; t += kOnePassThreads) rows[(size_t)blockIdx.x * (ids / 2) + t] = s_counts[t];
    if (tid == 0) beyond[blockIdx.x] = s_beyond;
}

// offsets[block][tile] = pairs of the tile in the blocks in front; totals[tile].  A workgroup takes kColumnTiles tiles, in as many parts of the rows
// as it has threads for.
constexpr int kColumnTiles = 32, kColumnParts = kOnePassThreads / kColumnTiles;
__global__ __launch_bounds__(kOnePassThreads) void tile_offsets_kernel(const uint16_t* __restrict__ rows, int blocks, uint32_t ids,
                                                                       uint32_t* __restrict__ offsets, uint32_t* __restrict__ totals,
                                                                       const uint64_t* __restrict__ keys, const uint32_t* __restrict__ beyond,
                                                                       uint32_t* __restrict__ marks)
{
    constexpr int kAtOnce = 16;
    __shared__ uint32_t s_sum[kColumnParts][kColumnTiles];
    const int column = threadIdx.x % kColumnTiles, part = threadIdx.x / kColumnTiles;
    const uint32_t tile = blockIdx.x * kColumnTiles + column;
    const int per = (blocks + kColumnParts - 1) / kColumnParts;
    const int r0 = min(blocks, part * per), r1 = min(blocks, r0 + per);
    if (blockIdx.x == 0) {          // one word out of the count workgroups' words
        uint32_t seen = 0;
        for (int b = (int)threadIdx.x; b < blocks; b += kOnePassThreads) seen |= beyond[b];
        const int any = __syncthreads_or(seen != 0);
        if (threadIdx.x == 0) { marks[kMarkByIndex] = any ? 1u : 0u; marks[kMarkAbove] = first_field(keys) & ~(ids - 1u); }
    }
    uint32_t c[kAtOnce], sum = 0;
    auto load = [&](int r) {
#pragma unroll
        for (int j = 0; j < kAtOnce; j++) c[j] = r + j < r1 ? rows[(size_t)(r + j) * ids + tile] : 0u;
    };
    for (int r = r0; r < r1; r += kAtOnce) {
        load(r);
#pragma unroll
        for (int j = 0; j < kAtOnce; j++) sum += c[j];
    }
    s_sum[part][column] = sum;
    __syncthreads();
    uint32_t run = 0, total = 0;
#pragma unroll
    for (int p = 0; p < kColumnParts; p++) {
        const uint32_t s = s_sum[p][column];
        run += p < part ? s : 0u;
        total += s;
    }
    if (part == 0) totals[tile] = total;
    for (int r = r0; r < r1; r += kAtOnce) {
        if (per > kAtOnce) load(r);
#pragma unroll
        for (int j = 0; j < kAtOnce; j++) {
            if (r + j < r1) offsets[(size_t)(r + j) * ids + tile] = run;
            run += c[j];
        }
    }
}

// Where the pairs of a block stand when it is stably sorted by kBits bits of their fields from `shift` up.  Slot i of lane l of wave w is place
// w * 64 * kItems + i * 64 + l; places from in_tile on are none.
template <int kItems, int kBits>
__device__ __forceinline__ void rank_block(const uint32_t (&field)[kItems], int shift, int in_tile, uint32_t (&place)[kItems],
                                           uint16_t (*s_count)[1 << kBits], uint16_t* s_start, uint32_t* s_wave_sum)
{
    constexpr int kB = 1 << kBits;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    for (int w = tid; w < kOnePassWaves * kB / 2; w += kOnePassThreads) ((uint32_t*)&s_count[0][0])[w] = 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kItems; i++) {          // (the ranking of scatter_kernel)
        const bool valid = wave * (kWave * kItems) + i * kWave + lane < in_tile;
        const uint32_t d = __builtin_amdgcn_ubfe(field[i], shift, kBits);
        const uint64_t all = ballot(valid);
        uint32_t peers_lo = (uint32_t)all, peers_hi = (uint32_t)(all >> 32);
#pragma unroll
        for (int b = 0; b < kBits; b++) {
            uint32_t bit = (uint32_t)__builtin_amdgcn_sbfe((int)d, b, 1);
            asm("" : "+v"(bit));
            const uint64_t with_bit = ballot(bit != 0);
            peers_lo = __builtin_amdgcn_bitop3_b32(peers_lo, (uint32_t)with_bit, bit, 0x90);
            peers_hi = __builtin_amdgcn_bitop3_b32(peers_hi, (uint32_t)(with_bit >> 32), bit, 0x90);
        }
        const uint32_t below = __builtin_amdgcn_mbcnt_hi(peers_hi, __builtin_amdgcn_mbcnt_lo(peers_lo, 0u));
        const uint32_t before = s_count[wave][d];
        if (valid && below == 0)
            s_count[wave][d] = (uint16_t)(before + (uint32_t)__popc(peers_lo) + (uint32_t)__popc(peers_hi));
        place[i] = before + below;
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    uint32_t total = 0, incl = 0;
    if (tid < kB) {
#pragma unroll
        for (int w = 0; w < kOnePassWaves; w++) {
            const uint32_t c = s_count[w][tid];
            s_count[w][tid] = (uint16_t)total;
            total += c;
        }
        incl = wave_inclusive_sum(total);
        if (lane == kWave - 1) s_wave_sum[wave] = incl;
    }
    __syncthreads();
    if (tid < kB) {
        uint32_t start = incl - total;
        for (int w = 0; w < wave; w++) start += s_wave_sum[w];
        s_start[tid] = (uint16_t)start;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        const uint32_t d = __builtin_amdgcn_ubfe(field[i], shift, kBits);
        place[i] += (uint32_t)s_start[d] + s_count[wave][d];
    }
}

// words: depth << 32 | value, every tile's pairs together and in input order; seg_start as in scatter_kernel.
template <int kItems>
__global__ __launch_bounds__(kOnePassThreads) void tile_scatter_kernel(const uint64_t* __restrict__ keys, const uint32_t* __restrict__ values,
                                                                       uint64_t* __restrict__ words, int n, uint32_t ids,
                                                                       const uint32_t* __restrict__ offsets, const uint32_t* __restrict__ totals,
                                                                       const uint32_t* __restrict__ marks, int* __restrict__ seg_start, TileRanking ranks)
{
    constexpr int kTile = kOnePassThreads * kItems, kPer = kOnePassIds / kOnePassThreads, kHigh = kOnePassBits - kOnePassLow;
    typedef uint32_t Four __attribute__((ext_vector_type(4)));
    static_assert(kPer % 4 == 0, "whole vectors");
    __shared__ uint64_t s_words[kTile];
    __shared__ uint16_t s_field[kTile];
    __shared__ __align__(16) uint32_t s_to[kOnePassIds];        // place of the pair at place p of the sorted block, of tile t: s_to[t] + p
    __shared__ __align__(4) uint16_t s_count[kOnePassWaves][1 << kOnePassLow];
    __shared__ uint16_t s_start[1 << kOnePassLow];
    __shared__ uint32_t s_wave_sum[kOnePassWaves];
    static_assert(kHigh <= kOnePassLow, "the counts of either pass");
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    // The first workgroup of a launch with one more than there are blocks ranks the frame's tiles meanwhile.
    const int ranking = ranks.order ? 1 : 0, blocks = (int)gridDim.x - ranking, index = (int)blockIdx.x - ranking;
    if (index < 0) {
        rank_tiles([&](int t) { return (int)totals[t]; }, ranks.num_tiles, ranks.order, ranks.squares, ranks.simds, s_to);
        return;
    }
    // (neighbouring blocks on one XCD, as in scatter_kernel)
    const int xcd = index % kXcds, each = blocks / kXcds, rest = blocks % kXcds;
    const int block = xcd * each + min(xcd, rest) + index / kXcds;
    const int base = block * kTile, in_tile = min(kTile, n - base);
    const int first = wave * (kWave * kItems) + lane;
    uint64_t word[kItems];
    uint32_t field[kItems], place[kItems];
    {
        uint32_t value[kItems];
#pragma unroll
        for (int i = 0; i < kItems; i++) word[i] = first + i * kWave < in_tile ? keys[base + first + i * kWave] : ~0ull;
#pragma unroll
        for (int i = 0; i < kItems; i++) value[i] = first + i * kWave < in_tile ? values[base + first + i * kWave] : 0u;
        // where every tile's pairs begin, and this block's among them
        Four total[kPer / 4], before[kPer / 4];
        const uint32_t t0 = (uint32_t)(tid * kPer);
        uint32_t sum = 0;
#pragma unroll
        for (int q = 0; q < kPer / 4; q++) {
            total[q] = 0; before[q] = 0;
            if (t0 < ids) {
                total[q] = ((const Four*)(totals + t0))[q];
                before[q] = ((const Four*)(offsets + (size_t)block * ids + t0))[q];
            }
        }
        const bool by_index = marks[kMarkByIndex] != 0;
#pragma unroll
        for (int q = 0; q < kPer / 4; q++) sum += total[q].x + total[q].y + total[q].z + total[q].w;
        const uint32_t incl = wave_inclusive_sum(sum);
        if (lane == kWave - 1) s_wave_sum[wave] = incl;
        __syncthreads();
        uint32_t start = incl - sum;
#pragma unroll
        for (int w = 0; w < kOnePassWaves; w++) start += w < wave ? s_wave_sum[w] : 0u;
        if (t0 < ids) {
#pragma unroll
            for (int q = 0; q < kPer / 4; q++) {
                Four at;
                at.x = start; at.y = at.x + total[q].x; at.z = at.y + total[q].y; at.w = at.z + total[q].z;
                start = at.w + total[q].w;
                if (block == 0) ((Four*)(seg_start + t0))[q] = at;
                *(Four*)(s_to + t0 + 4 * q) = at + before[q];
            }
        }
        if (block == 0 && tid == 0) seg_start[ids] = n;
#pragma unroll
        for (int i = 0; i < kItems; i++) {
            field[i] = (uint32_t)(word[i] >> 32) & (ids - 1u);
            word[i] = (word[i] << 32) | (by_index ? (uint32_t)(base + first + i * kWave) : value[i]);
        }
    }
    rank_block<kItems, kOnePassLow>(field, 0, in_tile, place, s_count, s_start, s_wave_sum);
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        if (first + i * kWave < in_tile) {
            s_words[place[i]] = word[i];
            s_field[place[i]] = (uint16_t)field[i];
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        const int p = min(first + i * kWave, in_tile - 1);
        word[i] = s_words[p];
        field[i] = s_field[p];
    }
    rank_block<kItems, kHigh>(field, kOnePassLow, in_tile, place, (uint16_t(*)[1 << kHigh])s_count, s_start, s_wave_sum);
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        if (first + i * kWave < in_tile) {
            s_words[place[i]] = word[i];
            s_field[place[i]] = (uint16_t)field[i];
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        const int p = min(i * kOnePassThreads + tid, in_tile - 1);
        word[i] = s_words[p];
        field[i] = s_field[p];
        if (i * kOnePassThreads + tid < in_tile && (p == 0 || s_field[p - 1] != field[i])) s_to[field[i]] -= (uint32_t)p;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        const int p = i * kOnePassThreads + tid;
        if (p < in_tile) words[s_to[field[i]] + (uint32_t)p] = word[i];
    }
}

// ---- per-tile segment sort on the 32 depth bits ----------------------------------------------------

// size classes of the segments: pairs per segment
constexpr int kCapTiny = 512, kCapSmall = 1024, kCapMedium = 4096, kCapLarge = 8192;
constexpr int kMergedLargeMax = 1 << 24;     // up to this many pairs the last launch also takes the class of 4097 .. 8192 pairs
constexpr int kManyPairs = 1 << 26;
// Up to kMergedTailMax pairs the last launch also takes the classes of 1025 .. 8192 pairs, and up to kMergedTailSpread where a tile has at most kMergedTailEach on
// average.  Sort, merged and not: 1M pairs of 3600 tiles, crowded, 68.5 and 82.3 us, of 8160 tiles, spread evenly, 39.7 and 41.4, 0.6M of 8160, crowded,
// 169.5 and 178, the frame of 1599x901 in 32x16 tiles 174.6 and 180.5; 1M pairs of 704 tiles, nearly all of them in these classes, 51 and 42.  Up to 2^21: 1.5M pairs of 3600
// tiles of 32x32 pixels 446 and 438.
constexpr int kMergedTailMax = 1 << 19, kMergedTailSpread = 1 << 20, kMergedTailEach = 512;

// First index in [0, n) whose tile field is >= v (n if none), found by the whole wave probing 64
// evenly spaced positions per step.  `keys` is ordered by tile field.  All lanes return the same.
__device__ __forceinline__ int wave_lower_bound(const uint64_t* __restrict__ keys, int n, uint32_t v, uint32_t tile_mask)
{
    const int lane = lane_id();
    int lo = 0, hi = n;                 // the answer lies in [lo, hi]; every index < lo is < v, index hi (if < n) is >= v
    while (hi > lo) {
        const int span = hi - lo;
        const int step = (span + kWave - 1) / kWave;        // >= 1
        const int pos = lo + lane * step;                    // probes at lo, lo+step, ...
        bool ge = true;                                      // a probe at or past hi counts as ">= v"
        if (pos < hi) ge = ((uint32_t)(keys[pos] >> 32) & tile_mask) >= v;
        const uint64_t m = ballot(ge);
        const int first = m ? __ffsll((long long)m) - 1 : kWave;     // first probe that is >= v
        if (first == 0) return lo;
        const int new_hi = first < kWave ? min(hi, lo + first * step) : hi;
        lo = lo + (first - 1) * step + 1;                    // the probe before `first` is < v
        hi = new_hi;
    }
    return lo;
}

// seg_start[v] = first index whose tile field is >= v, for v in [0, ids]; seg_start[ids] = n.
// A thread looks at kStartsPerThread pairs, 256 apart so that the loads of a workgroup stay
// contiguous: where the tile field changes, it fills the entries of the ids in between (empty ids
// get the same start as the next non-empty one).  Also clears the list counters.
constexpr int kStartsPerThread = 8;

__global__ __launch_bounds__(256) void segment_starts_kernel(const uint64_t* __restrict__ keys, int n, uint32_t tile_mask,
                                                             uint32_t ids, int* __restrict__ seg_start,
                                                             uint32_t* __restrict__ seg_counts)
{
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
    if (gid < (uint32_t)(kListClasses * kListShards)) seg_counts[gid] = 0;
    const long long base = (long long)blockIdx.x * (256 * kStartsPerThread) + threadIdx.x;
    uint32_t cur[kStartsPerThread], before[kStartsPerThread];
#pragma unroll
    for (int k = 0; k < kStartsPerThread; k++) {
        const long long i = base + k * 256;
        cur[k] = 0; before[k] = 0;
        if (i < n) {
            cur[k] = (uint32_t)(keys[i] >> 32) & tile_mask;
            before[k] = i == 0 ? 0u : ((uint32_t)(keys[i - 1] >> 32) & tile_mask) + 1u;
        }
    }
    // A run of up to kOwnFill entries is written by the thread that found it; a longer one (a band
    // of empty tiles, and the ids behind the last pair) by the whole wave, 64 entries per step.
    constexpr uint32_t kOwnFill = 4;
    const int lane = threadIdx.x & (kWave - 1);
    auto fill_by_wave = [&](bool mine, uint32_t lo, uint32_t hi, int value) {
        for (uint64_t todo = ballot(mine); todo; todo &= todo - 1) {
            const int src = __ffsll((long long)todo) - 1;
            const uint32_t from = (uint32_t)__shfl((int)lo, src), to = (uint32_t)__shfl((int)hi, src);
            const int what = __shfl(value, src);
            for (uint32_t v = from + (uint32_t)lane; v <= to; v += kWave) seg_start[v] = what;
        }
    };
#pragma unroll
    for (int k = 0; k < kStartsPerThread; k++) {
        const long long i = base + k * 256;
        const bool valid = i < n;
        // ids before[k]..cur[k] start at pair i: nothing to do when the field repeats
        const bool some = valid && before[k] <= cur[k];
        const bool longer = some && cur[k] - before[k] >= kOwnFill;
        if (some && !longer)
            for (uint32_t v = before[k]; v <= cur[k]; v++) seg_start[v] = (int)i;
        fill_by_wave(longer, before[k], cur[k], (int)i);
        fill_by_wave(valid && i == n - 1 && cur[k] < ids, cur[k] + 1, ids, n);
    }
}

// One stable counting pass of a segment over bits shift..shift+7 of its keys or words, by the kWaves
// waves of one workgroup.  Wave w owns the contiguous part [w*per, (w+1)*per) of the segment.
// Returns false (and moves nothing) when every pair has the same digit.  All threads of the
// workgroup must call it.  src_v null: words, without values beside them.
template <int kWaves>
__device__ __forceinline__ bool counting_pass(const uint64_t* src_k, const uint32_t* src_v, uint64_t* dst_k, uint32_t* dst_v,
                                              int n, int shift, uint32_t (*cnt)[kBins], uint32_t* wave_sum, int* flag)
{
    static_assert(kWaves > 1 && kWaves * kWave >= kBins, "one thread per digit");
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & (kWave - 1);
    const int wave = tid / kWave;
    const int per = ((n + kWaves - 1) / kWaves + kWave - 1) / kWave * kWave;   // a multiple of 64
    const int w_lo = min(n, wave * per), w_hi = min(n, w_lo + per);

    for (int d = lane; d < kBins; d += kWave) cnt[wave][d] = 0;
    if (tid == 0) *flag = 0;
    __syncthreads();
    for (int i = w_lo + lane; i < w_hi; i += kWave)
        atomicAdd(&cnt[wave][(uint32_t)(src_k[i] >> shift) & 255u], 1u);
    __syncthreads();
    // thread t < 256 handles digit t
    uint32_t total = 0;
    if (tid < kBins) {
        for (int w = 0; w < kWaves; w++) {
            const uint32_t c = cnt[w][tid];
            cnt[w][tid] = total;          // offset of wave w inside digit tid
            total += c;
        }
        if (total == (uint32_t)n) *flag = 1;
        uint32_t incl = wave_inclusive_sum(total);
        if (lane == kWave - 1) wave_sum[wave] = incl;
        total = incl - total;             // exclusive inside this wave's 64 digits
    }
    __syncthreads();
    if (tid < kBins) {
        uint32_t base = total;
        for (int w = 0; w < wave; w++) base += wave_sum[w];
        for (int w = 0; w < kWaves; w++) cnt[w][tid] += base;     // absolute start of (wave, digit)
    }
    __syncthreads();
    const bool uniform = *flag != 0;
    if (uniform) return false;

    // stable ranking, 64 pairs at a time in segment order
    for (int base = w_lo; base < w_hi; base += kWave) {
        const int i = base + lane;
        const bool valid = i < w_hi;
        uint64_t k = 0;
        uint32_t v = 0;
        if (valid) { k = src_k[i]; if (src_v) v = src_v[i]; }
        const uint32_t d = (uint32_t)(k >> shift) & 255u;
        uint64_t peers = ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const bool bit = (d >> b) & 1u;
            const uint64_t with_bit = ballot(bit);
            peers &= bit ? with_bit : ~with_bit;
        }
        const int below = popc_below(peers);
        uint32_t before = 0;
        if (valid && below == 0) {
            before = cnt[wave][d];
            cnt[wave][d] = before + (uint32_t)__popcll(peers);
        }
        const int leader = valid ? __ffsll((long long)peers) - 1 : lane;
        before = (uint32_t)__shfl((int)before, leader);
        if (valid) {
            dst_k[before + (uint32_t)below] = k;
            if (src_v) dst_v[before + (uint32_t)below] = v;
        }
        __builtin_amdgcn_wave_barrier();
    }
    return true;
}

// x of lane (l ^ kMask).  Within a row of 16 lanes most exchanges are one data-parallel-primitive move; the others go
// through the lane crossbar, which is idle otherwise: two moves in its place cost the vector unit more than the crossbar delays.
template <int kMask>
__device__ __forceinline__ uint32_t from_lane_xor(uint32_t x, int lane)
{
    constexpr int kQuadXor1 = 0xB1, kQuadXor2 = 0x4E, kQuadReverse = 0x1B, kRowHalfMirror = 0x141, kRowMirror = 0x140, kRowRor8 = 0x128;
    constexpr int kMove = kMask == 1 ? kQuadXor1 : kMask == 2 ? kQuadXor2 : kMask == 3 ? kQuadReverse : kMask == 7 ? kRowHalfMirror
                        : kMask == 8 ? kRowRor8 : kMask == 15 ? kRowMirror : 0;
    if constexpr (kMove != 0) return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, kMove, 0xf, 0xf, true);
    else if constexpr (kMask < 32) return (uint32_t)__builtin_amdgcn_ds_swizzle((int)x, kMask << 10 | 0x1f);
    else return (uint32_t)__builtin_amdgcn_ds_bpermute((lane ^ kMask) * 4, (int)x);
}

// The smaller word with limit 0, the larger one with limit ~0: one instruction (v_med3_u32), whichever a lane keeps.
__device__ __forceinline__ uint32_t keep_word(uint32_t a, uint32_t b, uint32_t limit)
{
    return max(min(a, b), min(max(a, b), limit));
}

__device__ __forceinline__ void order_words(uint32_t& a, uint32_t& b)
{
    const uint32_t lo = min(a, b), hi = max(a, b);
    a = lo;
    b = hi;
}

// Comparators of Batcher's odd-even merge sort (63 for 16 slots, where a bitonic network has 80).
template <int kT>
struct SlotNetwork {
    int first[kT * kT], second[kT * kT], count;
    constexpr SlotNetwork() : first(), second(), count(0)
    {
        for (int p = 1; p < kT; p *= 2)
            for (int k = p; k >= 1; k /= 2)
                for (int j = k % p; j + k < kT; j += 2 * k)
                    for (int i = 0; i < k && i + j + k < kT; i++)
                        if ((i + j) / (2 * p) == (i + j + k) / (2 * p)) {
                            first[count] = i + j;
                            second[count] = i + j + k;
                            count++;
                        }
    }
};

template <int kT, int... kI>
__device__ __forceinline__ void sort_slots_by(uint32_t (&c)[kT], std::integer_sequence<int, kI...>)
{
    constexpr SlotNetwork<kT> net;
    (order_words(c[net.first[kI]], c[net.second[kI]]), ...);
}

template <int kT>
__device__ __forceinline__ void sort_slots(uint32_t (&c)[kT])
{
    constexpr SlotNetwork<kT> net;
    sort_slots_by<kT>(c, std::make_integer_sequence<int, net.count>());
}

// One step of a merge across lanes: against the same slot of lane (l ^ kMask) or, kMirrored, the slots in reverse order.
template <int kMask, bool kMirrored, int kT>
__device__ __forceinline__ void compare_lanes(uint32_t (&c)[kT], int lane)
{
    constexpr int kTop = kMask >= 32 ? 5 : kMask >= 16 ? 4 : kMask >= 8 ? 3 : kMask >= 4 ? 2 : kMask >= 2 ? 1 : 0;
    const uint32_t limit = (uint32_t)__builtin_amdgcn_sbfe(lane, kTop, 1);          // the upper lane keeps the larger word
    // (eight slots at a time, with their mirror images: what is in flight stays in few registers)
    constexpr int kHalf = kT / 2, kGroup = kHalf < 4 ? kHalf : 4;
    if constexpr (kT == 1) {
        c[0] = keep_word(c[0], from_lane_xor<kMask>(c[0], lane), limit);
    } else {
#pragma unroll
        for (int g = 0; g < kHalf; g += kGroup) {
            uint32_t other[2 * kGroup];
#pragma unroll
            for (int i = 0; i < kGroup; i++) {
                const int t = g + i, u = kT - 1 - t;
                other[2 * i] = from_lane_xor<kMask>(c[kMirrored ? u : t], lane);
                other[2 * i + 1] = from_lane_xor<kMask>(c[kMirrored ? t : u], lane);
            }
#pragma unroll
            for (int i = 0; i < kGroup; i++) {
                const int t = g + i, u = kT - 1 - t;
                c[t] = keep_word(c[t], other[2 * i], limit);
                c[u] = keep_word(c[u], other[2 * i + 1], limit);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// The steps of a merge whose lanes differ in one bit, from 2^(kFrom) down, as far as the run has them (below `bits`), then those inside a lane.
template <int kT>
__device__ __forceinline__ void merge_lanes(uint32_t (&c)[kT], int lane, int bits)
{
    if (bits > 5) compare_lanes<32, false>(c, lane);
    if (bits > 4) compare_lanes<16, false>(c, lane);
    if (bits > 3) compare_lanes<8, false>(c, lane);
    if (bits > 2) compare_lanes<4, false>(c, lane);
    if (bits > 1) compare_lanes<2, false>(c, lane);
    if (bits > 0) compare_lanes<1, false>(c, lane);
#pragma unroll
    for (int j = kT / 2; j > 0; j >>= 1)
#pragma unroll
        for (int t = 0; t < kT; t++)
            if ((t & j) == 0) order_words(c[t], c[t | j]);
}

// Sorts 64 * kT words, element i in slot i % kT of lane i / kT: every lane its slots, then runs are merged two by two.  A merge
// begins with element i of the lower run against element i from the end of the upper one, so that all runs ascend, and
// goes on with halved distances.  A distance below kT pairs two slots of one lane (registers only); a larger one the same slot of
// two lanes: 21 steps cross lanes whatever kT is, where the slot-major layout (element i in lane i % 64) makes it 33 of 36 for 256
// elements and 45 of 55 for 1024.  The merges run in a loop and the distances are written out, so the code holds every exchange
// pattern once.
template <int kT>
__device__ __forceinline__ void sort_words(uint32_t (&c)[kT], int lane)
{
    if constexpr (kT > 1) sort_slots(c);
#pragma unroll 1
    for (int m = 0; m < 6; m++) {               // runs of 2^m lanes
        if (m == 0) compare_lanes<1, true>(c, lane);
        else if (m == 1) compare_lanes<3, true>(c, lane);
        else if (m == 2) compare_lanes<7, true>(c, lane);
        else if (m == 3) compare_lanes<15, true>(c, lane);
        else if (m == 4) compare_lanes<31, true>(c, lane);
        else compare_lanes<63, true>(c, lane);
        merge_lanes(c, lane, m);
    }
}

// A list as the segment sort finds and leaves it.  kWords: keys holds depth << 32 | value words and values nothing yet.
struct Lists {
    uint64_t* keys;
    uint32_t* values;
    const uint64_t* keys_in;            // the caller's unsorted list
    const uint32_t* values_in;
    const uint32_t* by_index;           // not zero where the values are indices into that list; behind it, what is above every key's sorted range where not
};

// The tile field of tile id v's pairs, where they are not indices.
__device__ __forceinline__ uint32_t field_of(const Lists& l, uint32_t v) { return v | l.by_index[1]; }

// Stores a pair of tile field v.
__device__ __forceinline__ void store_pair(const Lists& l, bool by_index, int i, uint32_t v, uint64_t word)
{
    uint64_t key = ((uint64_t)v << 32) | (word >> 32);
    uint32_t value = (uint32_t)word;
    if (by_index) {
        key = l.keys_in[value];
        value = l.values_in[value];
    }
    l.keys[i] = key;
    l.values[i] = value;
}

// A segment [lo, hi) as buffers with their lengths: a load past the end gives 0, a store there is dropped, without a comparison.
typedef uint32_t Pair2 __attribute__((ext_vector_type(2)));
struct Segment {
    __amdgpu_buffer_rsrc_t keys, values;
    __device__ __forceinline__ Segment(const Lists& l, int lo, int len)
    {
        constexpr int kRawDwords = 0x00020000;      // word 3 of the descriptor: 32-bit data, no swizzle
        keys = __builtin_amdgcn_make_buffer_rsrc(l.keys + lo, 0, len * 8, kRawDwords);
        values = __builtin_amdgcn_make_buffer_rsrc(l.values + lo, 0, len * 4, kRawDwords);
    }
    template <bool kWords>
    __device__ __forceinline__ void load(int i, uint32_t& depth, uint32_t& value) const
    {
        if constexpr (kWords) {
            const Pair2 w = __builtin_amdgcn_raw_buffer_load_b64(keys, i * 8, 0, 0);
            value = w.x;
            depth = w.y;
        } else {
            depth = __builtin_amdgcn_raw_buffer_load_b32(keys, i * 8, 0, 0);
            value = __builtin_amdgcn_raw_buffer_load_b32(values, i * 4, 0, 0);
        }
    }
    template <bool kWords>
    __device__ __forceinline__ uint32_t load_depth(int i) const
    {
        return __builtin_amdgcn_raw_buffer_load_b32(keys, i * 8 + (kWords ? 4 : 0), 0, 0);
    }
    // a pair as load() finds it
    template <bool kWords>
    __device__ __forceinline__ void put_back(int i, uint64_t word) const
    {
        if constexpr (kWords) {
            __builtin_amdgcn_raw_buffer_store_b64(Pair2{ (uint32_t)word, (uint32_t)(word >> 32) }, keys, i * 8, 0, 0);
        } else {
            __builtin_amdgcn_raw_buffer_store_b32((uint32_t)(word >> 32), keys, i * 8, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b32((uint32_t)word, values, i * 4, 0, 0);
        }
    }
    __device__ __forceinline__ void store(int i, uint32_t field, uint64_t word) const
    {
        const Pair2 key = { (uint32_t)(word >> 32), field };
        __builtin_amdgcn_raw_buffer_store_b64(key, keys, i * 8, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32((uint32_t)word, values, i * 4, 0, 0);
    }
};

// Words of LDS a wave needs to sort up to n pairs: a 32-bit word for every pair or one 64-bit word for every
// second pair (the sorted pairs go through it in two halves), one word of padding after every 16 (lane l puts its kUse consecutive ranks down at once; without
// the padding the lanes of a wave would all start in the same bank).
__host__ __device__ constexpr int staging_words(int n) { return n <= 64 ? n + n / 16 : n / 2 + n / 32; }
__device__ __forceinline__ int staged(int i) { return i + (i >> 4); }

// (two 32-bit words: as one of 64 bits the pairs of all slots would have to sit in neighbouring registers)
__device__ __forceinline__ void stage(uint64_t* at, uint32_t depth, uint32_t value)
{
    ((uint32_t*)at)[0] = value;
    ((uint32_t*)at)[1] = depth;
}

__host__ __device__ constexpr int log2_of(int n) { return n <= 1 ? 0 : 1 + log2_of(n / 2); }

__device__ __forceinline__ uint32_t wave_least(uint32_t x)
{
    constexpr int kRowShr1 = 0x111, kRowShr2 = 0x112, kRowShr4 = 0x114, kRowShr8 = 0x118, kRowBcast15 = 0x142, kRowBcast31 = 0x143;
    x = min(x, (uint32_t)__builtin_amdgcn_update_dpp(~0, (int)x, kRowShr1, 0xf, 0xf, false));
    x = min(x, (uint32_t)__builtin_amdgcn_update_dpp(~0, (int)x, kRowShr2, 0xf, 0xf, false));
    x = min(x, (uint32_t)__builtin_amdgcn_update_dpp(~0, (int)x, kRowShr4, 0xf, 0xf, false));
    x = min(x, (uint32_t)__builtin_amdgcn_update_dpp(~0, (int)x, kRowShr8, 0xf, 0xf, false));
    x = min(x, (uint32_t)__builtin_amdgcn_update_dpp(~0, (int)x, kRowBcast15, 0xa, 0xf, false));
    x = min(x, (uint32_t)__builtin_amdgcn_update_dpp(~0, (int)x, kRowBcast31, 0xc, 0xf, false));
    return (uint32_t)__builtin_amdgcn_readlane((int)x, kWave - 1);
}
__device__ __forceinline__ uint32_t wave_most(uint32_t x) { return ~wave_least(~x); }

// The largest of the words of this lane and of those below it.
__device__ __forceinline__ uint32_t wave_inclusive_most(uint32_t x)
{
    constexpr int kRowShr1 = 0x111, kRowShr2 = 0x112, kRowShr4 = 0x114, kRowShr8 = 0x118, kRowBcast15 = 0x142, kRowBcast31 = 0x143;
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kRowShr1, 0xf, 0xf, false));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kRowShr2, 0xf, 0xf, false));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kRowShr4, 0xf, 0xf, false));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kRowShr8, 0xf, 0xf, false));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kRowBcast15, 0xa, 0xf, false));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kRowBcast31, 0xc, 0xf, false));
    return x;
}

// How the words of a segment are made.  The network orders 32-bit words: the depth above the segment's least one, without the low
// `shift` bits that do not fit, in front of the pair's place in the segment, which keeps equal depths in input order and tells where the
// pair's depth and value are fetched from afterwards.  64-bit words of depth and value (min and max of doubles) took four
// instructions per word for a step across lanes, where these take two, twice the registers and twice the LDS between waves.
// Where bits were left out (depths that span more than 2^22 of their units for 1024 pairs, i.e. more than a few octaves of
// distances apart: most segments) pairs that agree in the others, a few in a thousand, can stand in the wrong order:
// neighbours are exchanged until none does.  A segment that kRepairs rounds of that leave unsorted, or of which half the lanes still have such
// neighbours behind kHopeless rounds (a surface seen face on in front of a far background: tens of pairs agree in the bits that fit), is sorted
// once more from the order it has: its pairs stand in groups that agree in those bits, and a word holds where the pair's group begins, the bits left out, and
// the pair's place in its group.  Where these three do not fit (more than 8192 pairs and groups of hundreds), it is sorted by
// the bits left out and then, from that order, by the others.
// (The bits that fit: 32 - log2 of the capacity; the shift is at most log2 of the capacity, so two such sorts cover every depth.)
// 60M pairs of a 1080p frame with nineteen in twenty inside a thousandth of their distance, in front of a background: 1531 us with the 64-bit words,
// which no depths slow down, 1887 with low bits and others always, 1535 with the groups (without such depths 1473, 1115, 1109); 20M 539, 680,
// 563 (425), 8M of a 4K frame inside a millionth 178, 198, 178 (139).  What sorts again is written out beside what does not, not in a loop with
// it: in one the kernels take eight registers more or spill them, 1 to 2 % of the sort of every frame.
struct WordBits {
    uint32_t least, range;
    int shift, stage;
    int in_group;               // of stage 1: bits of the places in a group, -1 where the words have no groups
    template <int kPlace>
    __device__ __forceinline__ void span(uint32_t lo, uint32_t hi)
    {
        least = (uint32_t)__builtin_amdgcn_readfirstlane((int)lo);
        range = (uint32_t)__builtin_amdgcn_readfirstlane((int)hi) - least;
        shift = max(0, kPlace - __builtin_clz(range | 1u));
        in_group = -1;
    }
    __device__ __forceinline__ bool complete() const { return shift == 0 || stage == 2 || in_group >= 0; }
    // stage 0 and 2: the bits from `shift` up; 1: those below
    template <int kPlace>
    __device__ __forceinline__ uint32_t word(uint32_t depth, bool valid, uint32_t place) const
    {
        const uint32_t above = valid ? depth - least : stage == 1 ? ~0u : range;         // (a place past the end sorts behind every pair)
        return __builtin_amdgcn_ubfe(above, stage == 1 ? 0 : shift, stage == 1 ? shift : 32 - kPlace) << kPlace | place;
    }
    // most: the last place of the longest group of a segment of len pairs
    __device__ __forceinline__ void group(uint32_t most, int len)
    {
        const int places = 32 - __builtin_clz((uint32_t)__builtin_amdgcn_readfirstlane((int)most) | 1u);
        in_group = 32 - __builtin_clz((uint32_t)len) + shift + places <= 32 ? places : -1;
    }
    __device__ __forceinline__ uint32_t group_word(uint32_t start, uint32_t low, bool valid, uint32_t place) const
    {
        return valid ? start << (shift + in_group) | low << in_group | (place - start) : ~0u;
    }
    template <int kPlace>
    __device__ __forceinline__ uint32_t place_in_group(uint32_t word) const
    {
        return min((word >> (shift + in_group)) + __builtin_amdgcn_ubfe(word, 0, in_group), (1u << kPlace) - 1u);      // (a word past the end: anywhere)
    }
};
constexpr int kRepairs = 8, kHopeless = 4;

// The words of stage 1 through LDS, places first .. first + 64 * kT - 1 of the segment, s[i] of place first + i.
// 1. Where the group of every pair begins, the largest place up to its own that differs from the one in front of it in the bits
// from `shift` up, or 0 (of a group that begins in front of `first`), in the upper half of s[i] and the bits below `shift` in the lower one.
// s: the depths; before: the one in front of `first`.  Returns the start that holds at the end.
template <int kT>
__device__ __forceinline__ uint32_t group_starts(const WordBits& bits, int lane, int first, uint32_t before, uint32_t* s)
{
    uint32_t left = (before - bits.least) >> bits.shift, at = 0;
#pragma unroll 4
    for (int t = 0; t < kT; t++) {
        const int i = t * kWave + lane;
        const uint32_t above = s[i] - bits.least, mine = above >> bits.shift;
        uint32_t neighbour = (uint32_t)__shfl_up((int)mine, 1);
        if (lane == 0) neighbour = left;
        left = (uint32_t)bcast_i((int)mine, kWave - 1);
        const uint32_t start = max(wave_inclusive_most(mine != neighbour ? (uint32_t)(first + i) : 0u), at);
        at = (uint32_t)bcast_i((int)start, kWave - 1);
        s[i] = start << 16 | __builtin_amdgcn_ubfe(above, 0, bits.shift);
    }
    return at;
}

// 2. The last place of the longest group, every start being `before` at least.
template <int kT>
__device__ __forceinline__ uint32_t longest_group(int lane, int first, int len, uint32_t before, const uint32_t* s)
{
    uint32_t most = 0;
#pragma unroll
    for (int t = 0; t < kT; t++) {
        const int i = t * kWave + lane;
        if (first + i < len) most = max(most, (uint32_t)(first + i) - max(s[i] >> 16, before));
    }
    return wave_most(most);
}

// 3. The words.
template <int kT>
__device__ __forceinline__ void group_words(uint32_t (&c)[kT], const WordBits& bits, int lane, int first, int len, uint32_t before, const uint32_t* s)
{
#pragma unroll
    for (int t = 0; t < kT; t++) {
        const int i = t * kWave + lane;
        c[t] = bits.group_word(max(s[i] >> 16, before), s[i] & 0xffffu, first + i < len, (uint32_t)(first + i));
    }
}

// Exchanges neighbours whose depths descend, ranks lane * kT + t: slots 0 and 1, 2 and 3, ... (first 0) or 1 and 2, 3 and 4, ...
template <int kT>
__device__ __forceinline__ void exchange_slots(uint32_t (&depth)[kT], uint32_t (&value)[kT], int first)
{
#pragma unroll
    for (int t = 0; t + 1 < kT; t++) {
        if (t % 2 != first) continue;
        const bool swap = depth[t] > depth[t + 1];
        const uint32_t v = value[t];
        order_words(depth[t], depth[t + 1]);
        value[t] = swap ? value[t + 1] : v;
        value[t + 1] = swap ? v : value[t + 1];
        __builtin_amdgcn_sched_barrier(0);      // one pair after the other: a copy of all of them would set the registers of the kernel
    }
}

// The last slot of every lane against the first of the next one; what stands in front of lane 0 and behind lane 63 is given.
template <int kT>
__device__ __forceinline__ void exchange_ends(uint32_t (&depth)[kT], uint32_t (&value)[kT], int lane,
                                              uint32_t depth_before, uint32_t value_before, uint32_t depth_behind, uint32_t value_behind)
{
    static_assert(kT >= 2, "a slot for either end of a lane");
    uint32_t db = (uint32_t)__shfl_up((int)depth[kT - 1], 1), vb = (uint32_t)__shfl_up((int)value[kT - 1], 1);
    uint32_t dn = (uint32_t)__shfl_down((int)depth[0], 1), vn = (uint32_t)__shfl_down((int)value[0], 1);
    if (lane == 0) { db = depth_before; vb = value_before; }
    if (lane == kWave - 1) { dn = depth_behind; vn = value_behind; }
    value[0] = db > depth[0] ? vb : value[0];
    depth[0] = max(db, depth[0]);
    value[kT - 1] = depth[kT - 1] > dn ? vn : value[kT - 1];
    depth[kT - 1] = min(dn, depth[kT - 1]);
}

// How many lanes of the wave have a depth that is larger than the next one; behind: the depth behind lane 63.
template <int kT>
__device__ __forceinline__ int descends(const uint32_t (&depth)[kT], int lane, uint32_t behind)
{
    uint32_t next = (uint32_t)__shfl_down((int)depth[0], 1);
    if (lane == kWave - 1) next = behind;
    bool any = depth[kT - 1] > next;
#pragma unroll
    for (int t = 0; t + 1 < kT; t++) any |= depth[t] > depth[t + 1];
    return __popcll(ballot(any));
}

// Sorts the segment [lo, hi) of tile id v with the network over kUse slots per lane, 64 * kUse >= hi - lo.
// The network does not care which slot a word starts in: the loads are the contiguous ones (element t*64 + lane in slot t),
// the network leaves rank lane*kUse + t in slot t, depths and values are fetched from LDS by the place in the word, one
// after the other through the same space, and the sorted pairs go through LDS to be stored contiguously again.
// False where exchanges of neighbours do not finish it (see WordBits): the pairs are then put back in the order they have, for kAgain, a second
// call.
template <int kUse, bool kWords, bool kAgain>
__device__ __forceinline__ bool sort_segment_wave_of(const Lists& lists, uint32_t v, int lo, int hi, uint64_t* s_w)
{
    constexpr int kCap = kUse * kWave, kPlace = log2_of(kCap);
    uint32_t* const s_one = (uint32_t*)s_w;
    // The lane number is made opaque here and again behind the network: otherwise every index and
    // address derived from it, for every width of the network, is computed once in front of the loop
    // over the segments and kept in registers through all of it.
    int lane = threadIdx.x & (kWave - 1);
    asm volatile("" : "+v"(lane));
    const int len = hi - lo;
    const Segment segment(lists, lo, len);
    constexpr int kRounds = kUse >= 2 ? 2 : 1, kHalf = kCap / kRounds;
    WordBits bits;
    bits.stage = kAgain ? 1 : 0;
    uint32_t depth[kUse], value[kUse], c[kUse];
#pragma unroll
    for (int t = 0; t < kUse; t++) segment.load<kWords>(t * kWave + lane, depth[t], value[t]);
    uint32_t least = ~0u, most = 0;
#pragma unroll
    for (int t = 0; t < kUse; t++) {
        most = max(most, depth[t]);                                         // 0 past the end
        depth[t] = t * kWave + lane < len ? depth[t] : ~0u;
        least = min(least, depth[t]);
    }
    bits.span<kPlace>(wave_least(least), wave_most(most));
    if constexpr (!kAgain) {
#pragma unroll
        for (int t = 0; t < kUse; t++) {
            s_one[t * kWave + lane] = value[t];
            c[t] = bits.word<kPlace>(depth[t], t * kWave + lane < len, (uint32_t)(t * kWave + lane));
        }
    } else {        // (the groups of a wave always fit: places, shift and places are at most 31 bits)
#pragma unroll
        for (int t = 0; t < kUse; t++) s_one[t * kWave + lane] = depth[t];
        group_starts<kUse>(bits, lane, 0, 0u, s_one);
        bits.group(longest_group<kUse>(lane, 0, len, 0u, s_one), len);
        group_words<kUse>(c, bits, lane, 0, len, 0u, s_one);
    }
    sort_words(c, lane);
    __builtin_amdgcn_wave_barrier();
    asm volatile("" : "+v"(lane));
    if constexpr (kAgain) {         // (a second time from memory: held through the network they would set the registers of the kernel)
#pragma unroll
        for (int t = 0; t < kUse; t++) {
            c[t] = bits.place_in_group<kPlace>(c[t]);
            segment.load<kWords>(t * kWave + lane, depth[t], value[t]);
            s_one[t * kWave + lane] = value[t];
        }
        __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int t = 0; t < kUse; t++) {
        c[t] &= (uint32_t)(kCap - 1);
        value[t] = s_one[c[t]];
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int t = 0; t < kUse; t++) s_one[t * kWave + lane] = depth[t];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int t = 0; t < kUse; t++) depth[t] = s_one[c[t]];
    __builtin_amdgcn_wave_barrier();
    bool sorted = kAgain || bits.shift == 0 || descends(depth, lane, ~0u) == 0;
    if constexpr (kUse >= 2 && !kAgain) {
#pragma unroll 1
        for (int r = 0; !sorted && r < kRepairs; r++) {
            exchange_slots(depth, value, 0);
            exchange_slots(depth, value, 1);
            exchange_ends(depth, value, lane, 0u, 0u, ~0u, 0u);
            const int wrong = descends(depth, lane, ~0u);
            sorted = wrong == 0;
            if (r + 1 == kHopeless && wrong * 2 * kUse > len) break;
        }
    }
    asm volatile("" : "+v"(lane));
    // (looked at here: through the network they would take scalar registers that it needs)
    const uint32_t* mark = lists.by_index;
    asm volatile("" : "+s"(mark));
    const bool by_index = mark[0] != 0;
    const uint32_t field = v | mark[1];
    // back to contiguous stores through LDS, the lower half of the ranks (lanes 0..31) first, then
    // the upper half through the same words: half the LDS, twice the waves per CU
#pragma unroll
    for (int h = 0; h < kRounds; h++) {
        __builtin_amdgcn_wave_barrier();
        if (lane / (kWave / kRounds) == h) {
#pragma unroll
            for (int t = 0; t < kUse; t++) stage(s_w + staged(lane * kUse + t - h * kHalf), depth[t], value[t]);
        }
        __builtin_amdgcn_wave_barrier();
        if (!sorted) {
#pragma unroll
            for (int t = h * (kUse / kRounds); t < (h + 1) * (kUse / kRounds); t++)
                segment.put_back<kWords>(t * kWave + lane, s_w[staged(t * kWave + lane - h * kHalf)]);
        } else if (!by_index) {
#pragma unroll
            for (int t = h * (kUse / kRounds); t < (h + 1) * (kUse / kRounds); t++)
                segment.store(t * kWave + lane, field, s_w[staged(t * kWave + lane - h * kHalf)]);
        } else {
#pragma unroll
            for (int t = h * (kUse / kRounds); t < (h + 1) * (kUse / kRounds); t++)
                if (t * kWave + lane < len) store_pair(lists, true, lo + t * kWave + lane, field, s_w[staged(t * kWave + lane - h * kHalf)]);
        }
    }
    __builtin_amdgcn_wave_barrier();
    if (!sorted) __threadfence_block();         // (other lanes read it back)
    return sorted;
}

// The network over the smallest power of two of register slots (at most kT) that holds the segment.
// s_w: staging_words(64 * kT) 64-bit words.
template <int kT, bool kWords, bool kAgain>
__device__ __forceinline__ bool sort_segment_wave_once(const Lists& lists, uint32_t v, int lo, int hi, uint64_t* s_w)
{
    const int len = hi - lo;
    if (len <= kWave) return sort_segment_wave_of<1, kWords, kAgain>(lists, v, lo, hi, s_w);
    if (kT >= 2 && len <= 2 * kWave) return sort_segment_wave_of<(kT >= 2 ? 2 : 1), kWords, kAgain>(lists, v, lo, hi, s_w);
    if (kT >= 4 && len <= 4 * kWave) return sort_segment_wave_of<(kT >= 4 ? 4 : 1), kWords, kAgain>(lists, v, lo, hi, s_w);
    if (kT >= 8 && len <= 8 * kWave) return sort_segment_wave_of<(kT >= 8 ? 8 : 1), kWords, kAgain>(lists, v, lo, hi, s_w);
    return sort_segment_wave_of<kT, kWords, kAgain>(lists, v, lo, hi, s_w);
}

template <int kT, bool kWords>
__device__ __forceinline__ void sort_segment_wave(const Lists& lists, uint32_t v, int lo, int hi, uint64_t* s_w)
{
    if (!sort_segment_wave_once<kT, kWords, false>(lists, v, lo, hi, s_w)) sort_segment_wave_once<kT, kWords, true>(lists, v, lo, hi, s_w);
}

// One step of the network between two waves: the wave's words against those of `partner`, in the same
// slots and lanes or (kMirrored) in reverse order, through LDS; a wave that takes no part only meets the barriers.
template <int kT, bool kMirrored>
__device__ __forceinline__ void compare_waves(uint32_t (&c)[kT], int lane, int wave, int partner, bool present, bool takes_part, uint32_t* s_one)
{
    if (present) {
        uint32_t* const to = s_one + wave * (kT * kWave) + lane;
#pragma unroll
        for (int t = 0; t < kT; t++) to[t * kWave] = c[t];
    }
    __syncthreads();
    if (takes_part) {
        const uint32_t* const from = s_one + partner * (kT * kWave) + (kMirrored ? kWave - 1 - lane : lane);
        const uint32_t limit = wave < partner ? 0u : ~0u;
#pragma unroll
        for (int t = 0; t < kT; t++) c[t] = keep_word(c[t], from[(kMirrored ? kT - 1 - t : t) * kWave], limit);
    }
    __syncthreads();
}

// What the waves that sort one segment tell each other.
template <int kWaves>
struct Between {
    uint32_t least[kWaves], most[kWaves], wrong[kWaves];
    uint32_t first_depth[kWaves], first_value[kWaves], last_depth[kWaves], last_value[kWaves];
};

// Sorts the segment [lo, hi) of tile id v, 64 * kWaves * kUse >= hi - lo, with the network over kUse
// slots per lane of kWaves waves.  Called by all waves of a workgroup with the same arguments.  s_w: kWaves times the
// staging words of 64 * kUse.
// Every wave sorts 64 * kUse words as above.  Runs are then merged in pairs: the first step compares
// element i of the lower run with element i from the end of the upper one, the next ones halve the
// distance, between waves through LDS and inside a wave as above.  All runs ascend, so the words
// past the end of the segment stay behind it, and waves that hold nothing else have nothing to do.
// stage: of WordBits; kAgain: 1 or 2, on what an earlier stage put back.  False where the segment has to be sorted again, with the next stage.
template <int kWaves, int kUse, bool kWords, bool kAgain>
__device__ __forceinline__ bool sort_segment_waves_of(const Lists& lists, uint32_t v, int lo, int hi, int at_stage, uint64_t* s_w, Between<kWaves>& s_between)
{
    static_assert(kUse >= 2, "the ranks leave in two halves of a wave's slots");
    constexpr int kPart = kUse * kWave;                 // words of a wave
    constexpr int kCap = kPart * kWaves, kPlace = log2_of(kCap);
    static_assert(kCap * 4 <= kWaves * staging_words(kPart) * 8, "a word for every pair");
    uint32_t* const s_one = (uint32_t*)s_w;
    int lane = threadIdx.x & (kWave - 1);
    asm volatile("" : "+v"(lane));
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const int len = hi - lo;
    const int first = wave * kPart;                     // this wave's part of the segment
    const bool present = first < len;
    const Segment segment(lists, lo, len);
    uint64_t* const s_mine = s_w + wave * staging_words(kPart);
    WordBits bits;
    bits.stage = kAgain ? at_stage : 0;
    uint32_t c[kUse];
    {
        uint32_t depth[kUse], least = ~0u, most = 0;
#pragma unroll
        for (int t = 0; t < kUse; t++) depth[t] = segment.load_depth<kWords>(first + t * kWave + lane);
#pragma unroll
        for (int t = 0; t < kUse; t++) {
            most = max(most, depth[t]);                                     // 0 past the end
            depth[t] = first + t * kWave + lane < len ? depth[t] : ~0u;
            least = min(least, depth[t]);
        }
        least = wave_least(least);
        most = wave_most(most);
        if (lane == 0) { s_between.least[wave] = least; s_between.most[wave] = most; }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kWaves; w++) {
            least = min(least, s_between.least[w]);
            most = max(most, s_between.most[w]);
        }
        bits.span<kPlace>(least, most);
        if (kAgain && bits.stage == 1) {
            uint32_t* const s_part = s_one + first;
#pragma unroll
            for (int t = 0; t < kUse; t++) s_part[t * kWave + lane] = depth[t];
            const uint32_t at = group_starts<kUse>(bits, lane, first, segment.load_depth<kWords>(max(first - 1, 0)), s_part);
            if (lane == 0) s_between.first_value[wave] = at;
            __syncthreads();
            uint32_t before = 0;                    // where the group begins that reaches into this wave's part
#pragma unroll 1
            for (int w = 0; w < wave; w++) before = max(before, s_between.first_value[w]);
            uint32_t longest = longest_group<kUse>(lane, first, len, before, s_part);
            if (lane == 0) s_between.wrong[wave] = longest;
            __syncthreads();
#pragma unroll 1
            for (int w = 0; w < kWaves; w++) longest = max(longest, s_between.wrong[w]);
            bits.group(longest, len);
            if (bits.in_group >= 0) group_words<kUse>(c, bits, lane, first, len, before, s_part);
        }
        if (!kAgain || bits.in_group < 0) {
#pragma unroll
            for (int t = 0; t < kUse; t++)
                c[t] = bits.word<kPlace>(depth[t], first + t * kWave + lane < len, (uint32_t)(first + t * kWave + lane));
        }
    }
    if (present) sort_words(c, lane);
#pragma unroll 1
    for (int group = 2; group <= kWaves && (group / 2) * kPart < len; group <<= 1) {      // waves of a merged run
        int partner = wave ^ (group - 1);
        compare_waves<kUse, true>(c, lane, wave, partner, present, present && partner * kPart < len, s_one);
#pragma unroll 1
        for (int d = group / 4; d > 0; d >>= 1) {
            partner = wave ^ d;
            compare_waves<kUse, false>(c, lane, wave, partner, present, present && partner * kPart < len, s_one);
        }
        if (present) merge_lanes(c, lane, 6);
    }
    asm volatile("" : "+v"(lane));
    if (kAgain && bits.in_group >= 0) {
#pragma unroll
        for (int t = 0; t < kUse; t++) c[t] = bits.place_in_group<kPlace>(c[t]);
    }
    // The pairs come from memory a second time: held through the merges they would take half of the registers, and with them the
    // waves that another segment's merges need.
    uint32_t depth[kUse], value[kUse];
#pragma unroll
    for (int t = 0; t < kUse; t++) segment.load<kWords>(first + t * kWave + lane, depth[t], value[t]);
#pragma unroll
    for (int t = 0; t < kUse; t++) {
        s_one[first + t * kWave + lane] = value[t];
        depth[t] = first + t * kWave + lane < len ? depth[t] : ~0u;
        c[t] &= (uint32_t)(kCap - 1);
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < kUse; t++) value[t] = s_one[c[t]];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < kUse; t++) s_one[first + t * kWave + lane] = depth[t];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < kUse; t++) depth[t] = s_one[c[t]];
    bool sorted = bits.complete();
    if (!kAgain && !sorted) {
        const int next = min(wave + 1, kWaves - 1), previous = max(wave - 1, 0);
#pragma unroll 1
        for (int r = 0; ; r++) {
            if (lane == 0) { s_between.first_depth[wave] = depth[0]; s_between.first_value[wave] = value[0]; }
            __syncthreads();
            const int wrong = descends(depth, lane, wave == kWaves - 1 ? ~0u : s_between.first_depth[next]);
            if (lane == 0) s_between.wrong[wave] = (uint32_t)wrong;
            __syncthreads();
            uint32_t all = 0;
#pragma unroll
            for (int w = 0; w < kWaves; w++) all += s_between.wrong[w];
            all = (uint32_t)__builtin_amdgcn_readfirstlane((int)all);
            sorted = all == 0;
            if (sorted || r == kRepairs || (r == kHopeless && all * 2 * kUse > (uint32_t)len)) break;
            exchange_slots(depth, value, 0);
            if (lane == 0) { s_between.first_depth[wave] = depth[0]; s_between.first_value[wave] = value[0]; }
            if (lane == kWave - 1) { s_between.last_depth[wave] = depth[kUse - 1]; s_between.last_value[wave] = value[kUse - 1]; }
            __syncthreads();
            exchange_slots(depth, value, 1);
            exchange_ends(depth, value, lane, wave == 0 ? 0u : s_between.last_depth[previous], s_between.last_value[previous],
                          wave == kWaves - 1 ? ~0u : s_between.first_depth[next], s_between.first_value[next]);
            __syncthreads();
        }
    }
    __syncthreads();
    asm volatile("" : "+v"(lane));
    // (looked at here: through the network they would take scalar registers that it needs)
    const uint32_t* mark = lists.by_index;
    asm volatile("" : "+s"(mark));
    const bool by_index = mark[0] != 0;
    const uint32_t field = v | mark[1];
    // back to contiguous stores through this wave's part of the LDS, half of the ranks at a time
#pragma unroll
    for (int h = 0; h < 2; h++) {
        __builtin_amdgcn_wave_barrier();
        if (lane / (kWave / 2) == h) {
#pragma unroll
            for (int t = 0; t < kUse; t++) stage(s_mine + staged(lane * kUse + t - h * (kPart / 2)), depth[t], value[t]);
        }
        __builtin_amdgcn_wave_barrier();
        if (!sorted) {
#pragma unroll
            for (int t = h * (kUse / 2); t < (h + 1) * (kUse / 2); t++)
                segment.put_back<kWords>(first + t * kWave + lane, s_mine[staged(t * kWave + lane - h * (kPart / 2))]);
        } else if (!by_index) {
#pragma unroll
            for (int t = h * (kUse / 2); t < (h + 1) * (kUse / 2); t++)
                segment.store(first + t * kWave + lane, field, s_mine[staged(t * kWave + lane - h * (kPart / 2))]);
        } else {
#pragma unroll
            for (int t = h * (kUse / 2); t < (h + 1) * (kUse / 2); t++) {
                const int i = first + t * kWave + lane;
                if (i < len) store_pair(lists, true, lo + i, field, s_mine[staged(t * kWave + lane - h * (kPart / 2))]);
            }
        }
    }
    if (!sorted) __threadfence_block();         // (other waves read it back)
    __syncthreads();
    return sorted;
}

// With the smallest number of slots per lane, from kLeast on, that holds the segment: hi - lo <= kCap.
template <int kWaves, int kCap, int kLeast, bool kWords, bool kAgain>
__device__ __forceinline__ bool sort_segment_waves_once(const Lists& lists, uint32_t v, int lo, int hi, int at_stage, uint64_t* s_w, Between<kWaves>& s_between)
{
    constexpr int kMost = kCap / (kWaves * kWave);
    if constexpr (kLeast < kMost)
        if (hi - lo > kLeast * kWaves * kWave)
            return sort_segment_waves_once<kWaves, kCap, 2 * kLeast, kWords, kAgain>(lists, v, lo, hi, at_stage, s_w, s_between);
    return sort_segment_waves_of<kWaves, kLeast, kWords, kAgain>(lists, v, lo, hi, at_stage, s_w, s_between);
}

template <int kWaves, int kCap, int kLeast, bool kWords>
__device__ __forceinline__ void sort_segment_waves(const Lists& lists, uint32_t v, int lo, int hi, uint64_t* s_w, Between<kWaves>& s_between)
{
    if (sort_segment_waves_once<kWaves, kCap, kLeast, kWords, false>(lists, v, lo, hi, 0, s_w, s_between)) return;
#pragma unroll 1
    for (int at_stage = 1; at_stage <= 2; at_stage++)
        if (sort_segment_waves_once<kWaves, kCap, kLeast, kWords, true>(lists, v, lo, hi, at_stage, s_w, s_between)) break;
}

// Segment sort by the waves of a workgroup for one size class: segments with min_len < length <= kCap.  Seven waves per SIMD: 110M pairs
// 328 -> 308 us against five of 82 registers, eight, with spilled registers, 357.  Of pairs eight: on frames of more than 2^20 tile ids most of the workgroups
// search for bounds that enclose nothing and end (16400x16400 pixels, 50 000 pairs: the sort 13.0 ms with seven, 12.3 with eight, 14.0 with five).
// With a table of segment starts, the first launch has listed the segments of the class.  Without a table
// (more tile ids than it holds) the grid has one workgroup per tile id and each searches for its bounds.
template <int kWaves, int kCap, int kLeast, bool kWords>
__global__ __launch_bounds__(kWaves * kWave) __attribute__((amdgpu_waves_per_eu(kWords ? 7 : 8))) void segment_sort_kernel(
    Lists lists, int n, uint32_t tile_mask, int min_len, const int* __restrict__ seg_start,
    const uint32_t* __restrict__ list, const uint32_t* __restrict__ list_count, uint32_t list_cap)
{
    __shared__ uint64_t s_w[kWaves * staging_words(kCap / kWaves)];
    __shared__ Between<kWaves> s_between;
    __shared__ int s_bounds[2];

    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);

    if (!kWords && !seg_start) {        // (words have a table)
        const uint32_t v = blockIdx.x;
        if (tid < kWave) {
            const int a = wave_lower_bound(lists.keys, n, v, tile_mask);
            const int b = v == tile_mask ? n : wave_lower_bound(lists.keys, n, v + 1, tile_mask);
            if (lane == 0) { s_bounds[0] = a; s_bounds[1] = b; }
        }
        __syncthreads();
        const int lo = s_bounds[0], hi = s_bounds[1];
        if (hi - lo <= min_len || hi - lo > kCap) return;
        sort_segment_waves<kWaves, kCap, kLeast, kWords>(lists, v, lo, hi, s_w, s_between);
        return;
    }

    // the listed segments are dealt out round-robin, shard by shard
    const uint32_t shard = blockIdx.x % kListShards;
    const uint32_t count = list_count[shard];
    for (uint32_t i = blockIdx.x / kListShards; i < count; i += gridDim.x / kListShards) {
        const uint32_t v = list[(size_t)shard * list_cap + i];
        sort_segment_waves<kWaves, kCap, kLeast, kWords>(lists, v, seg_start[v], seg_start[v + 1], s_w, s_between);
    }
}

// One wave per workgroup: it sorts the segments of up to 64*kT pairs of one tile id or of several, a grid apart.  Their bounds come from
// the table of segment starts or, without one, from a search.
// kNotes: writes what it finds of the tiles too.  (Compiled apart: a sort by itself does not pay for the question, 8K frame 0.1M pairs 57.5 -> 56.2 us, 0.4M 80.4 -> 79.4.)
template <int kT, bool kWords, bool kNotes>
__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(7))) void segment_sort_wave_kernel(
    Lists lists, int n, uint32_t tile_mask, const int* __restrict__ seg_start,
    int list_max0, int list_max1, int list_max2,
    uint32_t* __restrict__ seg_counts, uint32_t* __restrict__ list0, uint32_t* __restrict__ list1,
    uint32_t* __restrict__ list2, uint32_t* __restrict__ list3,
    uint32_t list_cap0, uint32_t list_cap1, uint32_t list_cap2, uint32_t list_cap3, TileNotes notes)
{
    __shared__ uint64_t s_w[staging_words(kT * kWave)];
    for (uint32_t v = blockIdx.x; v <= tile_mask; v += gridDim.x) {
        int lo, hi;
        if (!kWords && !seg_start) {
            lo = wave_lower_bound(lists.keys, n, v, tile_mask);
            hi = v == tile_mask ? n : wave_lower_bound(lists.keys, n, v + 1, tile_mask);
        } else {
            lo = seg_start[v];
            hi = seg_start[v + 1];
            // This launch sees every tile id once: it also lists the ids of the longer segments by class
            // (lengths up to list_max0, list_max1, list_max2, and everything longer), so that those
            // fewer, longer-running segments can be dealt out evenly by the launches that follow.
            const int len = hi - lo;
            if (kNotes && threadIdx.x == 0) note_tile(notes, v, lo, hi);
            if (len > kT * kWave && threadIdx.x == 0) {
                // neighbouring tiles tend to be equally busy: mix the index so that every list gets its share
                const uint32_t shard = (v ^ (v >> 5) ^ (v >> 10) ^ (v >> 15)) % kListShards;
                if (kT * kWave < kCapSmall && len <= list_max0)
                    list0[(size_t)shard * list_cap0 + atomicAdd(&seg_counts[0 * kListShards + shard], 1u)] = v;
                else if (len <= list_max1)
                    list1[(size_t)shard * list_cap1 + atomicAdd(&seg_counts[1 * kListShards + shard], 1u)] = v;
                else if (len <= list_max2)
                    list2[(size_t)shard * list_cap2 + atomicAdd(&seg_counts[2 * kListShards + shard], 1u)] = v;
                else
                    list3[(size_t)shard * list_cap3 + atomicAdd(&seg_counts[3 * kListShards + shard], 1u)] = v;
            }
        }
        // (words become pairs here, and indices values, also where there is nothing to sort)
        if (hi > lo && hi - lo <= kT * kWave) sort_segment_wave<kT, kWords>(lists, v, lo, hi, s_w);
    }
}

// A list of at most kAlonePairs pairs in few tiles: one workgroup per tile id, of which one wave does unless the segment has more than
// 1024 pairs, so that no other launch is needed for those.
static_assert(Short::kTile <= kCapSmall, "a list of one such block has no segment of the listed classes");
__global__ __launch_bounds__(4 * kWave) void segment_sort_alone_kernel(Lists lists, const int* __restrict__ seg_start, TileNotes notes)
{
    static_assert(kAlonePairs <= kCapMedium, "four waves hold any segment");
    __shared__ uint64_t s_w[4 * staging_words(kCapMedium / 4)];
    __shared__ Between<4> s_between;
    const uint32_t v = blockIdx.x;
    const int lo = seg_start[v], hi = seg_start[v + 1];
    if (threadIdx.x == 0) note_tile(notes, v, lo, hi);
    if (hi - lo > kCapSmall) sort_segment_waves<4, kCapMedium, 8, true>(lists, v, lo, hi, s_w, s_between);
    else if (hi > lo && threadIdx.x < kWave) sort_segment_wave<kCapSmall / kWave, true>(lists, v, lo, hi, s_w);
}

// The listed segments of one class (at most 64*kT pairs each), dealt out round-robin to
// single-wave workgroups.
template <int kT, bool kWords>
__global__ __launch_bounds__(kWave) void segment_sort_wave_list_kernel(
    Lists lists, const int* __restrict__ seg_start, const uint32_t* __restrict__ list, const uint32_t* __restrict__ list_count,
    uint32_t list_cap)
{
    __shared__ uint64_t s_w[staging_words(kT * kWave)];
    const uint32_t shard = blockIdx.x % kListShards;
    const uint32_t count = list_count[shard];
    for (uint32_t i = blockIdx.x / kListShards; i < count; i += gridDim.x / kListShards) {
        const uint32_t v = list[(size_t)shard * list_cap + i];
        sort_segment_wave<kT, kWords>(lists, v, seg_start[v], seg_start[v + 1], s_w);
        __builtin_amdgcn_wave_barrier();
    }
}

// Stable counting passes with a ping-pong copy in HBM: for segments of more than min_len pairs.
// Sixteen waves per workgroup: such a segment has thousands of pairs, every pass reads them from
// memory 64 per wave and step, and the workgroup has the CU almost to itself (a frame of 109M
// pairs with 534 such segments: 0.55 ms for the launch with four waves).
constexpr int kGeneralWaves = 16;

template <bool kWords>
__device__ __forceinline__ void sort_segment_general(const Lists& lists, uint64_t* __restrict__ alt_keys, uint32_t* __restrict__ alt_values,
                                                     uint32_t v, int lo, int hi, uint32_t (*s_cnt)[kBins], uint32_t* s_wave_sum, int* s_flag)
{
    // opaque, like the lane number of the networks: or the addresses of the copy below stay in
    // registers beside a network's words in a workgroup that does both
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int len = hi - lo;
    uint64_t* kbuf[2] = { lists.keys + lo, alt_keys + lo };
    uint32_t* vbuf[2] = { kWords ? nullptr : lists.values + lo, kWords ? nullptr : alt_values + lo };
    int cur = 0;
    constexpr int kDepth = kWords ? 32 : 0;             // where the depth bits begin
#pragma unroll 1
    for (int shift = kDepth; shift < kDepth + 32; shift += 8) {
        const bool moved = counting_pass<kGeneralWaves>(kbuf[cur], vbuf[cur], kbuf[cur ^ 1], vbuf[cur ^ 1], len, shift, s_cnt, s_wave_sum, s_flag);
        __threadfence_block();
        __syncthreads();
        if (moved) cur ^= 1;
    }
    const bool by_index = *lists.by_index != 0;
    if (kWords || cur == 1 || by_index)
        for (int i = tid; i < len; i += kGeneralWaves * kWave)
            store_pair(lists, by_index, lo + i, v, kWords ? kbuf[cur][i] : (kbuf[cur][i] << 32) | vbuf[cur][i]);
    __threadfence_block();
    __syncthreads();
}

// With a table of segment starts the workgroups take the listed segments (the
// ones longer than min_len: neighbouring tiles tend to be equally crowded, so they are dealt out
// one segment at a time, round-robin).
// With a table (kTable) a listed segment of up to kCapHuge pairs is sorted by the network over the
// sixteen waves: the passes through memory take 7 us each for 12 000 pairs.  (A workgroup has a CU to itself; two of
// 64 registers a lane, the counters in the space of the words: 113 -> 145 us on the frame of 110M pairs.)
// The workgroups first sort the listed segments of the classes below (first_class 1:
// 1025 .. kCapLarge pairs, 2: only those above kCapMedium, 3: none; shard by shard like the
// launches of those classes): a frame with a short list of pairs has few such segments or none,
// and one launch instead of three is what counts there; up to kMergedLargeMax pairs the class
// above kCapMedium still has few.
constexpr int kCapHuge = 16384;

template <bool kTable, bool kWords>
__global__ __launch_bounds__(kGeneralWaves * kWave) void segment_sort_general_kernel(
    Lists lists, uint64_t* __restrict__ alt_keys, uint32_t* __restrict__ alt_values,
    int n, uint32_t tile_mask, int min_len, const int* __restrict__ seg_start,
    const uint32_t* __restrict__ list, const uint32_t* __restrict__ list_count, uint32_t list_cap,
    const uint32_t* __restrict__ list_medium, uint32_t cap_medium, const uint32_t* __restrict__ list_large, uint32_t cap_large,
    int first_class, TileRanking ranks)
{
    __shared__ uint64_t s_w[kTable ? kGeneralWaves * staging_words(kCapHuge / kGeneralWaves) : 1];
    __shared__ Between<kGeneralWaves> s_between;
    __shared__ uint32_t s_cnt[kGeneralWaves][kBins];
    __shared__ uint32_t s_wave_sum[kGeneralWaves];
    __shared__ int s_bounds[2];
    __shared__ int s_flag;

    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);

    if constexpr (!kTable) {
        const uint32_t v = blockIdx.x;
        if (tid < kWave) {
            const int a = wave_lower_bound(lists.keys, n, v, tile_mask);
            const int b = v == tile_mask ? n : wave_lower_bound(lists.keys, n, v + 1, tile_mask);
            if (lane == 0) { s_bounds[0] = a; s_bounds[1] = b; }
        }
        __syncthreads();
        const int lo = s_bounds[0], hi = s_bounds[1];
        if (hi - lo > min_len) sort_segment_general<kWords>(lists, alt_keys, alt_values, field_of(lists, v), lo, hi, s_cnt, s_wave_sum, &s_flag);
    } else {
        // The first workgroup of a launch with one more than the lists are dealt out to ranks the frame's tiles meanwhile.
        const uint32_t ranking = kWords && ranks.order ? 1u : 0u;
        if (blockIdx.x < ranking) {
            static_assert(kGeneralWaves * kWave == 1024 && kBins >= kOrderBins, "a workgroup and the counters as rank_tiles wants them");
            rank_tiles([&](int t) { return seg_start[t + 1] - seg_start[t]; }, ranks.num_tiles, ranks.order, ranks.squares, ranks.simds, s_cnt[0]);
            return;
        }
        const uint32_t block = blockIdx.x - ranking, blocks = gridDim.x - ranking, shard = block % kListShards;
        // list_count: the counters of all classes, class c at c * kListShards (1: medium, 2: large, 3: long)
        for (int c = first_class; c <= 3; c++) {
            const uint32_t* const ids_of = c == 1 ? list_medium : c == 2 ? list_large : list;
            const uint32_t cap = c == 1 ? cap_medium : c == 2 ? cap_large : list_cap;
            const uint32_t count = list_count[c * kListShards + shard];
            for (uint32_t i = block / kListShards; i < count; i += blocks / kListShards) {
                const uint32_t v = ids_of[(size_t)shard * cap + i];
                const int lo = seg_start[v], hi = seg_start[v + 1];
                if (hi - lo <= kCapHuge)
                    sort_segment_waves<kGeneralWaves, kCapHuge, 2, kWords>(lists, v, lo, hi, s_w, s_between);
                else
                    sort_segment_general<kWords>(lists, alt_keys, alt_values, field_of(lists, v), lo, hi, s_cnt, s_wave_sum, &s_flag);
            }
        }
    }
}

// A list of one pair is sorted: neither the partition nor the launch over every tile id has anything to do (one pair on an 8K frame 110 -> 5 us,
// in 16400x16400 pixels 463 -> 5).
__global__ void copy_pair_kernel(const uint64_t* __restrict__ key_in, const uint32_t* __restrict__ value_in,
                                 uint64_t* __restrict__ key_out, uint32_t* __restrict__ value_out)
{
    *key_out = *key_in;
    *value_out = *value_in;
}

} // namespace
} // namespace fgs

extern "C" size_t fgs_get_sort_buffer_size(int num_rendered)
{
    if (num_rendered < 0 || num_rendered > FGS_MAX_RENDERED) return 0;
    return fgs::workspace_for(num_rendered).total;
}

namespace fgs {

int check_sort(int num_rendered, int width, int height, int block_x, int block_y, const char* list_sorting_space, size_t sorting_size,
               const uint64_t* gaussian_keys_unsorted, const uint32_t* gaussian_values_unsorted,
               const uint64_t* gaussian_keys_sorted, const uint32_t* gaussian_values_sorted, const char* who)
{
    if (num_rendered < 0)
        return fail(FGS_E_INVALID, "%s: num_rendered = %d is negative "
                                   "(a negative count is what a failed preprocess leaves behind)", who, num_rendered);
    if (num_rendered > FGS_MAX_RENDERED)
        return fail(FGS_E_INVALID, "%s: num_rendered = %d exceeds %d", who, num_rendered, FGS_MAX_RENDERED);
    if (width <= 0 || height <= 0 || block_x <= 0 || block_y <= 0)
        return fail(FGS_E_INVALID, "%s: width/height/block must be positive", who);
    if (num_rendered == 0) return FGS_OK;
    if (!list_sorting_space || !gaussian_keys_unsorted || !gaussian_values_unsorted ||
        !gaussian_keys_sorted || !gaussian_values_sorted)
        return fail(FGS_E_INVALID, "%s: null buffer", who);
    if ((uintptr_t)list_sorting_space % 256 != 0)
        return fail(FGS_E_INVALID, "%s: list_sorting_space must be 256-byte aligned", who);
    if (((uintptr_t)gaussian_keys_unsorted | (uintptr_t)gaussian_keys_sorted) % 8 != 0)
        return fail(FGS_E_INVALID, "%s: key buffers must be 8-byte aligned", who);
    const size_t needed = workspace_for(num_rendered).total;
    if (sorting_size < needed)
        return fail(FGS_E_WORKSPACE, "%s: list_sorting_space holds %zu bytes, %zu needed for %d pairs",
                    who, sorting_size, needed, num_rendered);
    if (tiles_of(width, height, block_x, block_y) >= (1LL << 30)) return fail(FGS_E_INVALID, "%s: too many tiles", who);
    return FGS_OK;
}

int sort_impl(int num_rendered, int width, int height, int block_x, int block_y, char* list_sorting_space, size_t sorting_size,
              const uint64_t* gaussian_keys_unsorted, const uint32_t* gaussian_values_unsorted,
              uint64_t* gaussian_keys_sorted, uint32_t* gaussian_values_sorted, FrameTables* frame, void* stream, const char* who)
{
    FrameTables tables = {};
    if (frame) std::swap(tables, *frame);           // what is written comes back
    int rc = check_sort(num_rendered, width, height, block_x, block_y, list_sorting_space, sorting_size, gaussian_keys_unsorted,
                        gaussian_values_unsorted, gaussian_keys_sorted, gaussian_values_sorted, who);
    if (rc != FGS_OK || num_rendered == 0) return rc;

    const int n = num_rendered;
    const Workspace ws = workspace_for(n);
    const long long tiles_xy = tiles_of(width, height, block_x, block_y);
    const int tile_bits = bit_length((uint32_t)tiles_xy);         // sort.cu:34-39: bits [0, 32 + tile_bits)
    const uint32_t tile_mask = (1u << tile_bits) - 1u;

    hipStream_t st = (hipStream_t)stream;
    if (n == 1) {
        hipLaunchKernelGGL(copy_pair_kernel, dim3(1), dim3(1), 0, st, gaussian_keys_unsorted, gaussian_values_unsorted,
                           gaussian_keys_sorted, gaussian_values_sorted);
        return check_hip(hipGetLastError(), "sort launch");
    }
    uint64_t* alt_keys = (uint64_t*)(list_sorting_space + ws.alt_keys);
    uint32_t* alt_values = (uint32_t*)(list_sorting_space + ws.alt_values);
    uint32_t* hist = (uint32_t*)(list_sorting_space + ws.hist);
    uint32_t* chunk_sums = (uint32_t*)(list_sorting_space + ws.chunk_sums);

    uint32_t* marks = (uint32_t*)(list_sorting_space + ws.marks);

    // The table of segment starts (with it the lists of the longer segments)
    // exists up to kMaxTableIds tile ids.  The last partition pass writes it when there are at
    // most two passes: with more, one workgroup could own 2^18 and more entries of a sparse frame.
    const uint32_t ids = 1u << tile_bits;
    int* seg_start = nullptr;
    uint32_t* seg_counts = nullptr;
    if (ids <= kMaxTableIds) {
        seg_start = (int*)(list_sorting_space + ws.seg_start);
        seg_counts = (uint32_t*)(list_sorting_space + ws.seg_lists);
    }
    const bool words = tile_bits <= kWordsMaxTileBits;              // at most two passes
    if (frame && words) frame->notes = tables.notes;

    // 1. stable partition by tile id, least significant tile digit first
    auto partition = [&](auto shape) {
        using Shape = decltype(shape);
        using Next = NextDigit<Shape>;
        // (what the forms below are compiled for: digits of 8 bits take one or two passes, which carry words, digits of 9 bits two or more)
        constexpr bool kOnePass = Shape::kBits == 8;
        static_assert(kNarrowMaxTileBits <= 16 && kNarrowMaxTileBits <= kWordsMaxTileBits && kNarrowMaxTileBits >= 9, "digits of 8 and 9 bits");
        constexpr bool kAlwaysSmall = std::is_same_v<Shape, Short>;
        static_assert(kShortPairs / Short::kTile * Short::kBinsP <= kMostRowWords, "a list of such blocks has few rows");
        const PassGrid g = pass_grid(n, Shape::kTile);
        const bool small = g.tiles * Shape::kBinsP <= kMostRowWords;     // the scatter workgroups add up the histogram rows themselves
        const int passes = (tile_bits + Shape::kBits - 1) / Shape::kBits;
        const uint64_t* src_k = gaussian_keys_unsorted;
        const void* src_v = gaussian_values_unsorted;
        for (int p = 0; p < passes; p++) {
            const bool to_sorted = ((passes - p) & 1) != 0;      // the last pass lands in the caller's sorted buffers
            uint64_t* dst_k = to_sorted ? gaussian_keys_sorted : alt_keys;
            uint32_t* dst_v = to_sorted ? gaussian_values_sorted : alt_values;
            const int nbits = tile_bits - Shape::kBits * p < Shape::kBits ? tile_bits - Shape::kBits * p : Shape::kBits;
            const bool first = p == 0, last = p == passes - 1;
            const bool from_words = words && !first;
            const int shift = from_words ? 0 : Shape::kBits * p;            // of the digit in what is read
#define FGS_SCATTER(IN, OUT, ...)                                                                                               \
            hipLaunchKernelGGL((scatter_kernel<Shape, Form::IN, Form::OUT __VA_ARGS__>), dim3(g.tiles), dim3(Shape::kThreads), 0, st, \
                               src_k, src_v, dst_k, (void*)dst_v, n, shift, nbits, last && passes == 2 ? Shape::kBits : 0,      \
                               (const uint32_t*)hist, small ? g.tiles : 0, ~tile_mask, marks, beyond_at, beyond_rows, seg_start)
            if constexpr (Shape::kAlone) {
                const uint32_t* const beyond_at = nullptr;
                const int beyond_rows = 0;
                if (first && last) FGS_SCATTER(kPairs, kSegments, , true);
                else if (first) FGS_SCATTER(kPairs, kWords, , true);
                else FGS_SCATTER(kWords, kSegments, , true);
            } else {
                uint32_t* const beyond = first ? marks + kMarkBeyond : nullptr;
                uint32_t* const clear = last ? seg_counts : nullptr;
                auto count = [&](auto* in) {
                    using In = std::remove_cv_t<std::remove_pointer_t<decltype(in)>>;
                    if (small) {
                        hipLaunchKernelGGL((count_kernel<Shape, In>), dim3(g.tiles), dim3(kSortBlock), 0, st,
                                           in, n, shift, nbits, hist, ~tile_mask, beyond, clear);
                    } else if constexpr (!kAlwaysSmall) {
                        const int groups = g.chunk < kCountGroups ? g.chunk : kCountGroups;
                        hipLaunchKernelGGL((count_chunk_kernel<Shape, In>), dim3(g.chunks), dim3(groups * kSortBlock), 0, st,
                                           in, n, shift, nbits, hist, g.tiles, g.chunk, chunk_sums, ~tile_mask, beyond, clear);
                        hipLaunchKernelGGL((offsets_kernel<Shape>), dim3(g.chunks), dim3(kOffsetThreads), 0, st,
                                           hist, g.tiles, g.chunk, chunk_sums, g.chunks, first ? marks : nullptr);
                    }
                };
                if (from_words) count((const Next*)src_v);
                else count(src_k);
                const uint32_t* const beyond_at = marks + (small ? kMarkBeyond : kMarkByIndex);
                const int beyond_rows = !first ? 0 : small ? g.tiles : 1;
                if constexpr (kOnePass) {
                    if (first && last) FGS_SCATTER(kPairs, kSegments);
                } else {
                    if (!words) FGS_SCATTER(kPairs, kPairs);
                }
                if (words && first && !last) FGS_SCATTER(kPairs, kWords);
                if (words && !first) FGS_SCATTER(kWords, kSegments);
            }
#undef FGS_SCATTER
            src_k = dst_k;
            src_v = dst_v;
        }
    };
    // (the launches that sort longer segments from lists need counters that the counting launches clear)
    const bool few_ids = n <= kAlonePairs && ids <= (uint32_t)kAloneIds;
    // (false where there is no room for the rows, or they are too many)
    auto one_pass = [&](auto items) {
        constexpr int kItems = decltype(items)::value;
        const int blocks = (n + kOnePassThreads * kItems - 1) / (kOnePassThreads * kItems);
        const size_t cells = (size_t)blocks * ids, bytes = cells * 6 + ((size_t)ids + blocks) * 4;
        if (cells > kOnePassCells) return false;
        const size_t behind = align_up(ws.total, 256);
        char* const at = bytes <= ws.seg_start - ws.alt_keys ? (char*)alt_keys
                       : behind < sorting_size && bytes <= sorting_size - behind ? list_sorting_space + behind : nullptr;
        if (!at) return false;
        uint32_t* const offsets = (uint32_t*)at;
        uint32_t* const rows = offsets + cells;
        uint32_t* const totals = rows + cells / 2;
        uint32_t* const beyond = totals + ids;
        hipLaunchKernelGGL((tile_count_kernel<kItems>), dim3(blocks), dim3(kOnePassThreads), 0, st, gaussian_keys_unsorted, n, ids, rows, beyond, seg_counts);
        hipLaunchKernelGGL(tile_offsets_kernel, dim3(ids / kColumnTiles), dim3(kOnePassThreads), 0, st, (const uint16_t*)rows, blocks, ids, offsets, totals,
                           gaussian_keys_unsorted, (const uint32_t*)beyond, marks);
        if (frame) frame->ranking = tables.ranking;
        hipLaunchKernelGGL((tile_scatter_kernel<kItems>), dim3(blocks + (tables.ranking.order ? 1 : 0)), dim3(kOnePassThreads), 0, st, gaussian_keys_unsorted,
                           gaussian_values_unsorted, gaussian_keys_sorted, n, ids, (const uint32_t*)offsets, (const uint32_t*)totals,
                           (const uint32_t*)marks, seg_start, tables.ranking);
        return true;
    };
    const bool one_digit = tile_bits >= kOnePassLeastBits && tile_bits <= kOnePassBits;         // (up to 8 bits are one pass of that digit)
    if (n <= Short::kTile && tile_bits <= kNarrowMaxTileBits) {
        partition(Alone<Short>());
    } else if (few_ids) {
        partition(Alone<Narrow>());
    } else if (one_digit && ((n <= kOnePassShort && one_pass(std::integral_constant<int, 2>())) || one_pass(std::integral_constant<int, 4>()))) {
        // (done)
    } else if (tile_bits <= kNarrowMaxTileBits) {
        if (n <= kShortPairs) partition(Short());
        else if (n <= kMiddlePairs) partition(Middle());
        else partition(Narrow());
    } else if (n <= kShortPairs) {
        partition(WideShort());
    } else {
        partition(Wide());
    }

    // 2. every tile id's segment by depth, in place in the sorted buffers
    const Lists lists = { gaussian_keys_sorted, gaussian_values_sorted, gaussian_keys_unsorted, gaussian_values_unsorted, marks + kMarkByIndex };
    if (seg_start && !words) {
        const unsigned blocks = (unsigned)(((size_t)n + 256 * kStartsPerThread - 1) / (256 * kStartsPerThread));
        hipLaunchKernelGGL(segment_starts_kernel, dim3(blocks), dim3(256), 0, st,
                           (const uint64_t*)gaussian_keys_sorted, n, tile_mask, ids, seg_start, seg_counts);
    }
    seg_counts = (uint32_t*)(list_sorting_space + ws.seg_lists);
    const uint32_t cap_small = (uint32_t)(n / 512 + 2), cap_medium = (uint32_t)(n / 1024 + 2), cap_large = (uint32_t)(n / 4096 + 2),
                   cap_long = (uint32_t)(n / 8192 + 2);
    uint32_t* list_small = seg_counts + 128;
    uint32_t* list_medium = list_small + (size_t)kListShards * cap_small;
    uint32_t* list_large = list_medium + (size_t)kListShards * cap_medium;
    uint32_t* list_long = list_large + (size_t)kListShards * cap_large;
    const uint32_t* no_list = nullptr;
    // grids of the list-driven launches: a multiple of kListShards, enough for every listed segment
    // (the limits are several times what is resident at once: a workgroup takes every
    // (grid / kListShards)-th segment of its shard, and the shards are not equally long)
    auto list_grid = [](unsigned most, unsigned limit) {
        const unsigned g = most < limit ? most : limit;
        return (g + kListShards - 1) / kListShards * kListShards;
    };
#define FGS_SEGMENT_WAVE(CAP, WORDS, NOTES)                                                                   \
    hipLaunchKernelGGL((segment_sort_wave_kernel<(CAP) / kWave, WORDS, NOTES>), dim3((ids + ids_per_wave - 1) / ids_per_wave), dim3(kWave),              \
                       0, st, lists, n, tile_mask, (const int*)seg_start,                                     \
                       kCapSmall, kCapMedium, kCapLarge, seg_counts, list_small, list_medium,                 \
                       list_large, list_long, cap_small, cap_medium, cap_large, cap_long, tables.notes)
#define FGS_SEGMENT_CLASS(WAVES, CAP, LEAST, WORDS, MINLEN, GRID, LIST, COUNT, LISTCAP)                         \
    hipLaunchKernelGGL((segment_sort_kernel<WAVES, CAP, LEAST, WORDS>), dim3(GRID), dim3((WAVES) * kWave), 0, st,  \
                       lists, n, tile_mask, MINLEN, (const int*)seg_start,                                    \
                       (const uint32_t*)(LIST), (const uint32_t*)(COUNT), LISTCAP)
#define FGS_SEGMENT_GENERAL(TABLE, WORDS, GRID, FIRST)                                                                  \
    hipLaunchKernelGGL((segment_sort_general_kernel<TABLE, WORDS>), dim3((GRID) + (ranks.order ? 1 : 0)), dim3(kGeneralWaves * kWave), 0, st,     \
                       lists, alt_keys, alt_values, n, tile_mask, kCapLarge, (const int*)seg_start,                    \
                       (const uint32_t*)list_long, (const uint32_t*)seg_counts, cap_long,                              \
                       (const uint32_t*)list_medium, cap_medium, (const uint32_t*)list_large, cap_large, FIRST, ranks)
    // A short list of pairs has few segments of more than 1024 pairs, or none: there the one
    // launch below takes those classes too (720p, 0.2M pairs: two launches less).
    const bool merged_tail = seg_start && (n <= kMergedTailMax || (n <= kMergedTailSpread && n <= kMergedTailEach * tiles_xy));
    // On a long list a wave takes several tile ids (a grid apart): its successor would start some 3 us after its end.  The segments of up
    // to 1024 pairs with 1, 2, 4 and 8 ids a wave: 110M pairs of an 8K frame 279, 256, 232, 224 us, 29M 113, 107, 109, 118, 36M of a 4K frame
    // 93, 76, 85, 103; below, the last waves' second segments count for more: 14.5M 82, 77, 80, 8M 34.7, 39.7, 41.1.
    const uint32_t ids_per_wave = n > kManyPairs ? 4 : n > kMergedLargeMax ? 2 : 1;
    const bool merged_large = seg_start && !merged_tail && n <= kMergedLargeMax;
    const int smallest = merged_tail ? kCapSmall : merged_large ? kCapMedium : kCapLarge;
    const unsigned tail_blocks = n > smallest ? list_grid((unsigned)(n / (smallest + 1) + 1), n > kMergedLargeMax ? 2048u : 256u) : 0u;
    const int first_class = merged_tail ? 1 : merged_large ? 2 : 3;
    const unsigned medium_blocks = list_grid((unsigned)(n / (kCapSmall + 1) + 1), 4096u), large_blocks = list_grid((unsigned)(n / (kCapMedium + 1) + 1), 1024u);
    // What the one-pass scatter did not rank is ranked beside the longest segments: a launch of its own behind the sort takes 8 us of 8160 tiles
    // (orbit of 2M at 1080p, 4.9M pairs a frame, six poses: 1668 -> 1643 us).
    TileRanking ranks = {};
    if (frame && words && !few_ids && tail_blocks && !frame->ranking.order) frame->ranking = ranks = tables.ranking;
    if (few_ids) {
        hipLaunchKernelGGL(segment_sort_alone_kernel, dim3(ids), dim3(4 * kWave), 0, st, lists, (const int*)seg_start, tables.notes);
    } else if (words) {
        // Up to 1024 pairs: one wave, network in registers; one tile id per wave on all but long lists (neighbouring
        // tiles tend to be equally busy, so a wave that took several of them would become the tail
        // of the launch).  The launch also lists the longer segments.  Segments of 513..1024 pairs in a launch of
        // their own last as long as one such sort on a frame of few tiles, which has about one per SIMD (1080p: -15 us, 4K:
        // -8 us, 8K -12 us without it, and -0.28 ms on the 8K frame of 109M pairs).
        if (tables.notes.ranges) FGS_SEGMENT_WAVE(kCapSmall, true, true);
        else FGS_SEGMENT_WAVE(kCapSmall, true, false);
        if (n > kCapSmall && !merged_tail) {
            FGS_SEGMENT_CLASS(4, kCapMedium, 8, true, kCapSmall, medium_blocks, list_medium, seg_counts + kListShards, cap_medium);
            if (n > kCapMedium && !merged_large)
                FGS_SEGMENT_CLASS(8, kCapLarge, 16, true, kCapMedium, large_blocks, list_large, seg_counts + 2 * kListShards, cap_large);
        }
        // longer segments from their list, one workgroup per segment
        if (tail_blocks) FGS_SEGMENT_GENERAL(true, true, tail_blocks, first_class);
    } else {
        FGS_SEGMENT_WAVE(kCapTiny, false, false);
        if (seg_start) {
            if (n > kCapTiny)       // 513..1024: the same network over 16 register slots, from the lists
                hipLaunchKernelGGL((segment_sort_wave_list_kernel<kCapSmall / kWave, false>),
                                   dim3(list_grid((unsigned)(n / (kCapTiny + 1) + 1), 8192u)),
                                   dim3(kWave), 0, st, lists, (const int*)seg_start,
                                   (const uint32_t*)list_small, (const uint32_t*)seg_counts, cap_small);
            if (n > kCapSmall && !merged_tail) {
                FGS_SEGMENT_CLASS(4, kCapMedium, 8, false, kCapSmall, medium_blocks, list_medium, seg_counts + kListShards, cap_medium);
                if (n > kCapMedium && !merged_large)
                    FGS_SEGMENT_CLASS(8, kCapLarge, 16, false, kCapMedium, large_blocks, list_large, seg_counts + 2 * kListShards, cap_large);
            }
            if (tail_blocks) FGS_SEGMENT_GENERAL(true, false, tail_blocks, first_class);
        } else {
            if (n > kCapTiny) FGS_SEGMENT_CLASS(4, kCapSmall, 4, false, kCapTiny, ids, no_list, no_list, 0u);
            if (n > kCapSmall) FGS_SEGMENT_CLASS(4, kCapMedium, 8, false, kCapSmall, ids, no_list, no_list, 0u);
            if (n > kCapMedium) FGS_SEGMENT_CLASS(8, kCapLarge, 16, false, kCapMedium, ids, no_list, no_list, 0u);
            if (n > kCapLarge) FGS_SEGMENT_GENERAL(false, false, ids, 0);
        }
    }
#undef FGS_SEGMENT_WAVE
#undef FGS_SEGMENT_CLASS
#undef FGS_SEGMENT_GENERAL
    return check_hip(hipGetLastError(), "sort launch");
}

} // namespace fgs

extern "C" int fgs_sort_gaussian(int num_rendered,
                                 int width, int height, int block_x, int block_y,
                                 char* list_sorting_space, size_t sorting_size,
                                 const uint64_t* gaussian_keys_unsorted, const uint32_t* gaussian_values_unsorted,
                                 uint64_t* gaussian_keys_sorted, uint32_t* gaussian_values_sorted, void* stream)
{
    return fgs::sort_impl(num_rendered, width, height, block_x, block_y, list_sorting_space, sorting_size, gaussian_keys_unsorted,
                          gaussian_values_unsorted, gaussian_keys_sorted, gaussian_values_sorted, nullptr, stream, "fgs_sort_gaussian");
}
