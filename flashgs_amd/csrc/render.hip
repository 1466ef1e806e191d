// Tile ranges and front-to-back alpha blending for gfx950 (wave64).
//
// Replaces FlashGS render<BX,BY> (csrc/cuda_rasterizer/render.cu:549-576): zero the ranges,
// identifyTileRanges (:9-31) and renderCUDA (:199-547).
//
// Blend layout: one wave64 works on 16x16 pixels, four per lane; a wide tile (32x16, 32x32) is a workgroup
// of two or four such waves.  Gaussians are taken 16 at a time: their exponents at all pixels come from the
// matrix unit, while the loads of the following batch are already in flight; then the wave shades its pixels
// Gaussian by Gaussian.  After every second Gaussian one ballot tests whether all pixels of the tile
// have T < 1e-4, which is the reference's stop rule (render.cu:394-408).  Every kernel exists in
// two forms: all sums and products in fp32 (the default; from the weight on the operations of the reference's pixel
// shader, the weight itself by other means than its formula: see below), and with the colour sums on the matrix unit too, four Gaussians at a time (f16 operands, fp32
// accumulation), which a caller asks for per call (FGS_BLEND_MATRIX_F16) or per process
// (fgs_set_colour_sums).
#include "fgs_internal.h"
#include "sort.h"
#include "tile_order.h"
#include "tile_rank.h"

#include <algorithm>
#include <atomic>
#include <map>
#include <mutex>
#include <utility>

namespace fgs {

// v_mul_legacy_f32: a product in which zero times anything, infinity included, is zero
__device__ float mul_zero_wins(float a, float b) __asm("llvm.amdgcn.fmul.legacy");

namespace {

__global__ __launch_bounds__(256) void fill_i32_kernel(int* p, size_t n, int v)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}


// The ranking (rank_tiles) is a launch of one workgroup behind the ranges, or a workgroup of the sort's in front of them (fgs_sort_render).
// (Ranking in the last workgroup of tile_ranges_kernel instead costs more than this launch: every
// workgroup then has to push its ranges out of its XCD's L2 before it counts itself done.)
// The ranking is written by one launch and read by the next, so it needs memory of its own: one
// table per (device, stream), allocated on the first such blend on that stream (blends on
// different streams may overlap and get a table each).  Blends on one stream follow each other, and
// its lock is held until both launches are enqueued: else another thread's ranking of another
// frame, enqueued between them, would be the one the blend reads.
// No tile needs its rank to be blended, so there is none under capture, where the table's address
// would stay in the graph and be shared by whatever replays it beside this stream's own blends, and
// none where no memory is left.
struct OrderTable {
    std::mutex enqueue;
    uint32_t* ranks = nullptr;          // kOrderCap + 2 words, then two LongLists
    int turn = 0;                       // which of those the next large frame uses: cleared by the last blend that was enqueued
};
std::map<StreamKey, OrderTable> g_order_tables;      // (entries stay where they are)
std::mutex g_order_mutex;

// *out is null where the tiles go unranked; enqueue is locked for as long as nobody else may enqueue a
// launch that writes *out.
int tile_order_table(hipStream_t stream, uint32_t** out, std::unique_lock<std::mutex>* enqueue, OrderTable** table = nullptr)
{
    int device = 0;
    *out = nullptr;
    FGS_HIP_TRY(hipGetDevice(&device));
    if (stream) {
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        FGS_HIP_TRY(hipStreamIsCapturing(stream, &capture));
        if (capture != hipStreamCaptureStatusNone) return FGS_OK;
    }
    OrderTable* entry;
    {
        std::lock_guard<std::mutex> lock(g_order_mutex);
        entry = &g_order_tables[stream_key(device, stream)];
    }
    *enqueue = std::unique_lock<std::mutex>(entry->enqueue);
    if (!entry->ranks && malloc_kept((void**)&entry->ranks, (kOrderCap + 2) * sizeof(uint32_t) + 2 * sizeof(LongLists)) != hipSuccess) {
        (void)hipGetLastError();
        entry->ranks = nullptr;
    }
    *out = entry->ranks;
    if (table) *table = entry;
    return FGS_OK;
}

struct RangeLength {
    const int2* ranges;
    __device__ __forceinline__ int operator()(int tile) const { const int2 r = ranges[tile]; return r.y - r.x; }
};

__global__ __launch_bounds__(1024) void tile_order_kernel(const int2* __restrict__ ranges, int num_tiles,
                                                          uint32_t* __restrict__ tile_order, int squares, int simds)
{
    __shared__ uint32_t s_count[kOrderBins];
    rank_tiles(RangeLength{ranges}, num_tiles, tile_order, squares, simds, s_count);
}

// render.cu:9-31, with the tile index checked against the number of tiles: what the pair at idx, of tile cur (num_tiles:
// outside the image) behind a pair of tile prev, says about the ranges.
// Also writes (0, 0) for the tiles without pairs (the reference clears the whole table first,
// render.cu:557): the pair that opens tile c clears the tiles between its predecessor's tile and
// c, the first pair those before it and the last pair those behind it.  A run of up to 4 tiles is
// cleared by the thread that found it, a longer one by its whole wave.  All lanes of a wave call it.
__device__ __forceinline__ void mark_ranges(long long idx, bool valid, uint32_t cur, uint32_t prev, int L,
                                            int2* __restrict__ ranges, uint32_t num_tiles)
{
    const int lane = threadIdx.x & (kWave - 1);
    auto clear_by_wave = [&](bool mine, uint32_t lo, uint32_t hi) {         // tiles [lo, hi)
        for (uint64_t todo = ballot(mine); todo; todo &= todo - 1) {
            const int src = __ffsll((long long)todo) - 1;
            const uint32_t from = (uint32_t)__shfl((int)lo, src), to = (uint32_t)__shfl((int)hi, src);
            for (uint32_t t = from + (uint32_t)lane; t < to; t += kWave) ranges[t] = make_int2(0, 0);
        }
    };
    const bool opens = valid && (idx == 0 || cur != prev);
    if (opens) {
        if (idx > 0 && prev < num_tiles) ranges[prev].y = (int)idx;
        if (cur < num_tiles) ranges[cur].x = (int)idx;
    }
    if (valid && idx == L - 1 && cur < num_tiles) ranges[cur].y = L;
    // empty tiles in front of this pair's tile
    const uint32_t lo = idx == 0 ? 0u : min(prev + 1u, num_tiles);
    const bool gap = opens && lo < cur;
    const bool wide = gap && cur - lo > 4u;
    if (gap && !wide)
        for (uint32_t t = lo; t < cur; t++) ranges[t] = make_int2(0, 0);
    clear_by_wave(wide, lo, cur);
    clear_by_wave(valid && idx == L - 1 && cur + 1u < num_tiles, cur + 1u, num_tiles);
}

// A thread looks at kRangesPerThread pairs, 256 apart so that the loads of a workgroup stay contiguous.
constexpr int kRangesPerThread = 4;

__global__ __launch_bounds__(256) void tile_ranges_kernel(int L, const uint64_t* __restrict__ keys,
                                                          int2* __restrict__ ranges, uint32_t num_tiles)
{
    const long long base = (long long)blockIdx.x * (256 * kRangesPerThread) + threadIdx.x;
    uint32_t cur[kRangesPerThread], prev[kRangesPerThread];
#pragma unroll
    for (int k = 0; k < kRangesPerThread; k++) {
        const long long idx = base + k * 256;
        cur[k] = 0; prev[k] = 0;
        if (idx < L) {
            cur[k] = min((uint32_t)(keys[idx] >> 32), num_tiles);
            if (idx > 0) prev[k] = min((uint32_t)(keys[idx - 1] >> 32), num_tiles);
        }
    }
#pragma unroll
    for (int k = 0; k < kRangesPerThread; k++) {
        const long long idx = base + k * 256;
        mark_ranges(idx, idx < L, cur[k], prev[k], L, ranges, num_tiles);
    }
}

// The same for a long list of pairs, most of which say nothing: a wave takes kRangeRuns runs of 64 keys, looks at the last
// key of each, and reads only the runs that end in another tile than they begin in (and the first and the last one of the
// list), kRangesPerThread of them at a time.  Reading every key is bound by the memory, 881 MB for 110M pairs; this reads a
// line of each run's four and the runs that hold a tile's border: 110M pairs in 129 600 tiles 185 us by the kernel above,
// 66 by this one, 14.5M pairs there 22.1 and 18.2, 11.6M in 32 400 18.5 and 12.7, 8.0M 13.9 and 10.7, 5.2M in 8160 10.3 and 5.5.
// (16 runs per wave: 51, 20.4, 12.0, 12.4 and 5.8.  A bisection by each lane where its 64 keys end in another tile: 41, 26.5, 5.6,
// 7.4 and 4.3, but 19.6 in place of 4.4 where 1.7M pairs lie unevenly: one dependent chain per border.)
//
// kList: it also lists the tiles whose lists are long (LongLists): the one tile of the wave that begins in its runs and goes on behind them is looked
// for again long_list pairs (more than the wave's) further on.  That is a line of its own, and it is waited for behind the borders.
constexpr int kRangeRuns = 8;

template <bool kList>
__global__ __launch_bounds__(256) void tile_ranges_sampled_kernel(int L, const uint64_t* __restrict__ keys,
                                                                  int2* __restrict__ ranges, uint32_t num_tiles,
                                                                  LongLists* __restrict__ longer, int long_list)
{
    const int lane = threadIdx.x & (kWave - 1);
    const long long base = ((long long)blockIdx.x * (256 / kWave) + threadIdx.x / kWave) * (kRangeRuns * kWave);
    auto tile_at = [&](long long idx) { return min((uint32_t)(keys[idx] >> 32), num_tiles); };
    const long long begin = base + lane * kWave, end = min((long long)L, begin + kWave);
    const bool mine = lane < kRangeRuns && begin < L;
    uint32_t last = 0, before = 0;
    if (mine) last = tile_at(end - 1);
    if (lane == 0 && mine && begin > 0) before = tile_at(begin - 1);
    const uint32_t left = (uint32_t)__shfl_up((int)last, 1);
    if (lane > 0) before = left;
    const bool goes_on = last == (uint32_t)__shfl((int)last, kRangeRuns - 1) && end - 1 + long_list < L;
    const bool begins = kList && mine && goes_on && (last != before || begin == 0) && last < num_tiles;
    uint32_t ahead = ~0u;
    if (begins) ahead = ((const uint32_t*)keys)[2 * (end - 1 + long_list) + 1];     // (nothing but the load: a use in here would be waited for)
    uint64_t todo = ballot(mine && (last != before || begin == 0 || end == L));
    while (todo) {
        long long idx[kRangesPerThread];
        uint32_t cur[kRangesPerThread], prev[kRangesPerThread];
        bool valid[kRangesPerThread];
#pragma unroll
        for (int k = 0; k < kRangesPerThread; k++) {
            const int run = todo ? __ffsll((long long)todo) - 1 : 0;
            idx[k] = base + run * kWave + lane;
            valid[k] = todo != 0 && idx[k] < L;
            cur[k] = valid[k] ? tile_at(idx[k]) : 0u;
            prev[k] = (uint32_t)__shfl((int)before, run);
            todo &= todo - 1;           // (0 stays 0)
        }
#pragma unroll
        for (int k = 0; k < kRangesPerThread; k++) {
            const uint32_t left_key = (uint32_t)__shfl_up((int)cur[k], 1);
            mark_ranges(idx[k], valid[k], cur[k], lane > 0 ? left_key : prev[k], L, ranges, num_tiles);
        }
    }
    if (begins && ahead == last) {
        const uint32_t shard = long_shard(last), at = atomicAdd(&longer->count[shard], 1u);
        if (at < (uint32_t)kLongPerShard) longer->tiles[shard][at] = last;
    }
}

// render.cu:54-57
__device__ __forceinline__ uint8_t encode_u8(float x)
{
    float v = x * 255.0f;
    v = v > 0.0f ? v : 0.0f;       // also maps NaN to 0
    v = v < 255.0f ? v : 255.0f;
    return (uint8_t)v;
}

// How a wave shades 16x16 pixels.  Lane l holds a strip of four pixels, (l % 16, 4 (l / 16) + j) for
// j = 0 .. 3.  The exponent of a Gaussian, q = w + cx dx^2 + cz dy^2 + cy dx dy with (dx, dy) the offset of
// the pixel from the Gaussian's centre (render.cu:42-45), is a quadratic along the strip, so its
// weights alpha_j = 2^q_j follow from the value and the slope at the strip's first pixel:
//     alpha_{j+1} = alpha_j rho_j,   rho_{j+1} = rho_j E,   rho_0 = 2^(q_1 - q_0),   E = 2^(2 cz),
// two exponentials and five multiplications for four pixels.  (v_exp_f32 takes the vector unit 8.4
// cycles a wave, a multiplication 2.6.)
//
// Values and slopes are a matrix product.  With (X, Y) the strip's first pixel relative to the centre
// of the square and (ex, ey) the Gaussian's centre relative to it,
//     q_0       = [w + cx ex^2 + cz ey^2 + cy ex ey] + bx X + by Y + cx X^2 + cz Y^2 + cy XY,
//     q_1 - q_0 = [by + cz] + cy X + 2 cz Y,     bx = -(2 cx ex + cy ey),  by = -(2 cz ey + cy ex),
// Gaussians x coefficients times {1, X, X^2, Y, Y^2, XY} x strips, and go through the matrix unit, whose
// bf16 instructions run beside the vector instructions of other waves (its fp32 ones do not: the same
// product with v_mfma_f32_32x32x2_f32 made a 4K frame 9 % slower).  Nothing is lost by bf16: the
// coordinates are small whole numbers, a coefficient is the sum of three bf16 numbers of eight bits of its
// significand each, products are exact and sums are fp32.  A slope is as exact as a value; its error
// counts up to three times in alpha_3, some 1e-6 of it.  Against a float64 blend of the same lists the
// image of a 1080p frame of 1M is off by 4.0e-7 (2-norm), of the 4K orbit with its needles by 4.9e-6;
// with the tables in LDS that were here before it was 1.0e-6 and 8.9e-6.
//
// v_mfma_f32_32x32x16_bf16 multiplies 32 rows by 32 columns over 16 slots, of which lanes 0-31 supply
// slots 0-7 and lanes 32-63 slots 8-15, and lane l receives rows 8 i + 4 (l / 32) + j of column l % 32.
// Rows 8 i + 4 h + j, h = 0, 1, are Gaussian 4 i + j, with its coefficients in the slots of half h only
// and zeros in the others, and the slots of half h hold the coordinates of the strips of lanes 32 h ..
// 32 h + 31: so lane l receives all 16 Gaussians, in list order, at its own strip.  Two coefficients of
// three parts fill six slots of a half; five instructions make 16 values and 16 slopes per lane.
//
// The recurrence starts at the strip's first weight, so that one must not be flushed to zero while a
// later one matters.  Along the strip q_t = Q + cz (t - t0)^2 with Q = w + dx^2 (cy^2 - 4 cx cz) / (-4 cz).
// With cz in [-3, 0] and Q <= 20 it is not: q_0 < -126 means -cz t0^2 > 126 + Q, and then q_3 is below
// Q - (sqrt(126 + Q) - 3 sqrt(3))^2, 2^-27 or less; a rho_0 with a first weight above zero is below 2^42.  A
// semidefinite form, which fgs_preprocess makes up to roundings, has Q <= w and by the 0.3 it adds to the variances, in exact
// arithmetic, cz > -2.41.  From the 64 Gaussians with the first one beyond cz = -3 on, a list is walked with four
// exponentials per strip, of exponents summed up from the same value and slope (walk_chunks<.., true>); 64 with
// one among them that is out of what that takes too are blended by evaluating every exponent (walk_plain).  The
// two forms are loops behind each other: side by side in one loop they cost the first 20 to 60 spilled registers.
// A 4K frame of 3M with all its conics beyond -3: 900 us by walk_plain, 485 so (467 with exponents from tables over the
// tile); with one in a hundred beyond 430, 320 (335); with none 300.  1080p of 1M: 282, 160 (150); 218, 157 (150); 142.
// The same with 32x16 tiles: 700, 382 (760); 605, 461 (760); 443.
//
// What bounds the launch is the issue of vector instructions: 25 fp32 instructions (5 for the recurrence, 4 alpha T, 4 T -=,
// 12 for the colour sums) and two exponentials per Gaussian and wave, and 4 more for staging, stop tests and loop.
// The 4K frame of 3M takes some 107 cycles of its 2.1 GHz per Gaussian and 16x16 pixels: 1.486e9 evaluations in 285 us, where a loop of
// these instructions attains 6.2e12 a second, 240 us (5.2e12 with the two exponentials side by side; calibrate.hip).  With several waves on a
// SIMD v_mul_f32, v_add_f32 and v_sub_f32 with vector registers as all operands take 2.6 cycles, v_fma_f32 3.0, with a scalar operand
// 4.4 like comparisons, shifts and conversions, a v_exp_f32 8.4, and nothing issues beside it.  4K frame of 3M Gaussians 336 -> 280 us, 8K of
// 8M 762 -> 671, 1080p of 1M 147 -> 139, against a version that took the exponents from per-column and
// per-row tables in LDS (four exponentials, 32 vector instructions).  (Two waves per 16x16 pixels with
// two pixels per lane and staging shared over barriers: 357 us on the 4K frame.)
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

constexpr int kBatch = 16;                  // Gaussians per matrix product
constexpr int kChunk = kWave;               // Gaussians staged at a time, one per lane
constexpr int kStopBelow = 0x38d1b717;      // 0.0001f: a pixel with less transmittance left is opaque
constexpr float kMostExponent = 20.0f;      // of a Gaussian that the matrix product takes
// Curvature along the strip up to which exponents are summed up: value and slopes are rounded at some 200 times it, to
// 1e-3 at most (as from tables over the tile).
constexpr float kSharpest = 64.0f;
constexpr int kNeverStop = -2147483647 - 1;
// Exponents up to this one count as none above zero: T of kLeastInFront to 1 stays in there, and once below kStopBelow it stays
// below it, since a weight turns the sign of T with a factor of at most 2^0.01 - 1 < 0.007.
constexpr float kSlightlyAbove = 0.01f, kLeastInFront = -0.01f;

// An fp32 number as the sum of three bf16 numbers: eight bits of the significand each.
// (Each is the upper half of a float; the bits below are left to high_halves to drop.)
struct Parts {
    float hi, mid, lo;
};
__device__ __forceinline__ Parts parts_of(float x)
{
    Parts p;
    p.hi = x;
    p.mid = x - __uint_as_float(__float_as_uint(x) & 0xffff0000u);
    p.lo = p.mid - __uint_as_float(__float_as_uint(p.mid) & 0xffff0000u);
    return p;
}

// the upper halves of two floats, a's in the lower half of the word
__device__ __forceinline__ float high_halves(float a, float b)
{
    return __uint_as_float(__builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u));
}

// six slots: the parts of two coefficients
__device__ __forceinline__ float4 slots_of(const Parts& a, const Parts& b)
{
    return make_float4(high_halves(a.hi, b.hi), high_halves(a.mid, b.mid), high_halves(a.lo, b.lo), 0.0f);
}

// Keeps two values in one aligned pair of registers, `even` in its even one and `odd` in its odd one.  No instruction comes of it.
// v_fma_f32 and v_fmac_f32 read three registers, and where all three numbers are even, or all are odd, the instruction takes
// 4.6 cycles of a SIMD in place of 2.6 (loops of 32 on every combination of registers 8 to 23 and eight sums, five waves; v_mul, v_add and v_sub, with
// two operands, always 2.6).
__device__ __forceinline__ void paired(float& even, float& odd)
{
    typedef float Pair __attribute__((ext_vector_type(2)));
    Pair p = {even, odd};
    asm("" : "+v"(p));
    even = p.x; odd = p.y;
}

// What a lane keeps of the 64 x 4 pixels of a wave.
struct Pixels {
    float T[4], r[4], g[4], b[4];
};

__device__ __forceinline__ void pixel_of(int lane, int j, int* x, int* y)
{
    *x = lane & 15;
    *y = ((lane >> 4) << 2) + j;
}

// The colour sums C += (alpha T) c are a matrix product, pixels x Gaussians times Gaussians x
// channels, and go through v_mfma_f32_4x4x4_16b_f16: sixteen independent 4x4 products with an
// inner dimension of 4.  A block is four neighbouring lanes; row i of its A operand is lane i's
// pixel, its four f16 values that pixel's weights alpha T for four Gaussians; column j of B is
// channel j of those Gaussians' colours (the same in every block; column 3 is zero); lane j of the
// block accumulates, in fp32, channel j of the four lanes' pixels in its four result registers.
// A lane shades four pixels, so four Gaussians cost it four such instructions where the plain form
// costs 48 multiply-adds.  Weights and colours are rounded to f16 (to nearest), products and sums
// are fp32: the colour of a pixel differs from the all-fp32 sum by at most 2^-10 of itself.  The
// weights are scaled by 2^14 (added to the exponent, taken out again with the result), which keeps
// them in f16's normal range down to 4e-9.  T itself never leaves fp32.  This form is opt-in
// (FGS_BLEND_MATRIX_F16); the default forms the sums by fp32 multiply-add, as the reference does.
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef float float4_t __attribute__((ext_vector_type(4)));
constexpr float kWeightScaleLog2 = 14.0f;
constexpr float kWeightUnscale = 6.103515625e-05f;          // 2^-14
constexpr float kColourMax = 65504.0f;                      // largest f16: a colour beyond it is drawn as this

// A read that stays where it is written: the compiler neither sinks it to its first use nor drops
// it when the value turns out unused (volatile on the vector type keeps it one wide LDS read).
template <typename V>
__device__ __forceinline__ V lds_read(const char* p)
{
    typedef float Native __attribute__((ext_vector_type(sizeof(V) / sizeof(float))));
    const Native n = *(const volatile __attribute__((address_space(3))) Native*)p;
    V v;
    __builtin_memcpy(&v, &n, sizeof(V));
    return v;
}

// A store to LDS that stays where it is written.
__device__ __forceinline__ void lds_write(char* p, float v)
{
    *(volatile __attribute__((address_space(3))) float*)p = v;
}

__device__ __forceinline__ uint32_t pack_f16(float a, float b)
{
    const float2_t v = {a, b};
    const half2_t h = __builtin_convertvector(v, half2_t);       // v_cvt_pk_f16_f32, round to nearest
    return __builtin_bit_cast(uint32_t, h);
}

// A wave's colour sums: in the lane of the pixel (fp32), or in the layout of the matrix instruction.
template <bool kFp32>
struct Sums {
    float r[4], g[4], b[4];
};
template <>
struct Sums<false> {
    float4_t acc[4];
};

// LDS of a wave, in bytes: a record of five times six slots per staged Gaussian and one of zeros behind them,
// then per Gaussian (r, g, b, E), or with f16 operands its four f16 channels in groups of four
// Gaussians and E by itself.  (With f16 operands the sums also go back to their pixels through it.)
constexpr int kRecord = 5 * 16;
constexpr int kColours = (kChunk + 1) * kRecord;
constexpr int kRatios = kColours + 8 * kChunk;              // f16 operands only
constexpr int kStageFloats = (kColours + 16 * kChunk) / 4;

// Lane-constant part of the walk.
struct LaneRole {
    int lane;
    // this lane's columns of the right-hand matrices, two coordinates each: (1, X), (Y, X^2), (Y^2, XY)
    float right[3];
    // which record it supplies to the left-hand matrix: Gaussian 4 i + j for row 8 i + 4 h + j of its own
    // half h, the record of zeros for the rows of the other half
    int record_at, record_step;

    __device__ __forceinline__ void init(int lane_, float* stage)
    {
        lane = lane_;
        const float X = (float)((lane & 15) - 8), Y = (float)(4 * (lane >> 4) - 8);
        right[0] = high_halves(1.0f, X);
        right[1] = high_halves(Y, X * X);
        right[2] = high_halves(Y * Y, X * Y);
        const bool own = (lane >> 5) == ((lane >> 2) & 1);
        record_at = own ? (((lane >> 1) & 12) | (lane & 3)) * kRecord : kChunk * kRecord;
        record_step = own ? kBatch * kRecord : 0;
        if (lane < kRecord / 4) stage[kChunk * (kRecord / 4) + lane] = 0.0f;
    }
};

template <bool kFp32>
__device__ __forceinline__ void clear(float (&T)[4], Sums<kFp32>& sums)
{
    float one = 1.0f;
    asm volatile("" : "+v"(one));       // made here, not kept (in private memory, by then) from one job of a wave to the next
#pragma unroll
    for (int k = 0; k < 4; k++) {
        T[k] = one;
        if constexpr (kFp32) { sums.r[k] = 0.0f; sums.g[k] = 0.0f; sums.b[k] = 0.0f; }
        else sums.acc[k] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }
}

// Whether all 256 pixels have T < stop_below, by their bits, which order like the numbers (a negative T
// counts as opaque either way).  Mostly the first comparison settles it.
__device__ __forceinline__ bool all_stopped(const float (&T)[4], int stop_below)
{
    auto as_int = [](float t) { return (int)__float_as_uint(t); };
    if (ballot(as_int(T[1]) >= stop_below) != 0) return false;
    return ballot(max(max(as_int(T[0]), as_int(T[2])), as_int(T[3])) >= stop_below) == 0;
}

__device__ __forceinline__ float clamped_to_f16(float c)          // NaN stays NaN
{
    return c > kColourMax ? kColourMax : (c < -kColourMax ? -kColourMax : c);
}

__device__ __forceinline__ void accumulate_f16(Sums<false>& sums, const uint32_t (&packed)[4][2], float2 colours)
{
    const half4_t colour = __builtin_bit_cast(half4_t, colours);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const uint2 a = make_uint2(packed[k][0], packed[k][1]);
        sums.acc[k] = __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(half4_t, a), colour, sums.acc[k], 0, 0, 0);
    }
}

// The first cnt of the Gaussians that the lanes hold (lane i: the i-th), with every exponent evaluated as
// render.cu:42-45 writes it.  Returns how many were walked, ~that when the stop ended it.
template <bool kFp32>
__device__ __forceinline__ int walk_plain(float2 xy, float4 co, float4 rgb, int cnt, float left, float top, int stop_below,
                                                    float (&T)[4], Sums<kFp32>& sums)
{
    int lane = lane_id();
    asm volatile("" : "+v"(lane));      // as in write_square
    int x, y;
    pixel_of(lane, 0, &x, &y);
    for (int i = 0; i < cnt; i += 2) {
        uint32_t packed[4][2] = {};
        float w[2][4] = {};
        float c[2][3] = {};
#pragma unroll
        for (int half = 0; half < 2; half++) {
            const int src = i + half;
            if (src >= cnt) break;
            const float dx = bcast_f(xy.x, src) - (left + (float)x);
            const float cx = bcast_f(co.x, src), cy = bcast_f(co.y, src), cz = bcast_f(co.z, src), lw = bcast_f(co.w, src);
            c[half][0] = bcast_f(rgb.x, src); c[half][1] = bcast_f(rgb.y, src); c[half][2] = bcast_f(rgb.z, src);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float dy = bcast_f(xy.y, src) - (top + (float)(y + k));
                const float q = lw + cx * dx * dx + cz * dy * dy + cy * dx * dy;
                const float at = __builtin_amdgcn_exp2f(q) * T[k];
                if constexpr (kFp32) {
                    sums.r[k] += c[half][0] * at;
                    sums.g[k] += c[half][1] * at;
                    sums.b[k] += c[half][2] * at;
                    T[k] -= at;
                } else {
                    T[k] = __builtin_fmaf(at, -kWeightUnscale, T[k]);
                    w[half][k] = at;
                }
            }
        }
        if constexpr (!kFp32) {
            // two of the four Gaussians of a matrix instruction; this lane's channel of their colours
#pragma unroll
            for (int k = 0; k < 4; k++) packed[k][0] = pack_f16(w[0][k], w[1][k]);
            const int ch = lane & 3;
            float a = 0.0f, b = 0.0f;
#pragma unroll
            for (int m = 0; m < 3; m++)
                if (ch == m) { a = clamped_to_f16(c[0][m]); b = clamped_to_f16(c[1][m]); }
            accumulate_f16(sums, packed, make_float2(__uint_as_float(pack_f16(a, b)), 0.0f));
        }
        if (i + 1 < cnt && all_stopped(T, stop_below)) return ~(i + 2);
    }
    return cnt;
}

// What a wave holds of a list ahead of its walk: the attributes of the chunk that comes next, one Gaussian per lane, and
// the indices for the chunk behind it.  The list index is fetched two chunks ahead and the attributes one chunk ahead, so
// that no wave waits for an index only to start the loads that depend on it.  Positions past the end of the list are
// clamped to its last entry: those loads are valid and their result unused.  (Positions are unsigned: a list may end
// with pair 2^31 - 1.)
struct Ahead {
    float2 xy;
    float4 co, rgb;
    uint32_t index;
};

// walk_list below from its entry base on, in chunks of 64: to the first chunk that the recurrence does not take, or
// (kSteep) to the end.  Returns as walk_list does, or base of the chunk it ended in front of.
template <bool kFp32, bool kSteep, bool kRun>
__device__ __forceinline__ int walk_chunks(
    const LaneRole& role, float* stage,
    const uint32_t* __restrict__ point_list, int begin, int n,
    float left, float top,
    const float2* __restrict__ points_xy,
    const float4* __restrict__ rgb_depth,
    const float4* __restrict__ conic_opacity,
    float (&T)[4], Sums<kFp32>& sums, int stop_below, Ahead& next, int base, bool& above)
{
    const int lane = role.lane;
    char* const bytes = reinterpret_cast<char*>(stage);
    auto fetch = [&]() {
        next.xy = points_xy[next.index]; next.co = conic_opacity[next.index]; next.rgb = rgb_depth[next.index];
        next.index = point_list[min((uint32_t)begin + (uint32_t)base + 2u * kChunk + (uint32_t)lane, (uint32_t)begin + (uint32_t)n - 1u)];
    };
    for (; base < n; base += kChunk) {
        const int cnt = min(kChunk, n - base);
        float2 xy = next.xy;
        float4 co = next.co, rgb = next.rgb;
        asm volatile("" : "+v"(co.x));          // nothing of the checks below is made earlier: no spilled registers (8K frame 695 -> 686 us)
        // conic_opacity = (cx, cy, cz, w) in the units of the exponent (see fgs_preprocess).  With f16
        // weights log2 of the opacity is held below 2 so that no scaled weight leaves f16's range.
        if constexpr (!kFp32) co.w = (co.w > 1.99f ? 1.99f : co.w) + kWeightScaleLog2;
        const float ex = xy.x - (left + 8.0f), ey = xy.y - (top + 8.0f);
        const float bx = -__builtin_fmaf(2.0f * co.x, ex, co.y * ey), by = -__builtin_fmaf(2.0f * co.z, ey, co.y * ex);
        float c = __builtin_fmaf(ex, __builtin_fmaf(co.x, ex, co.y * ey), __builtin_fmaf(co.z * ey, ey, co.w));
        // Q over the columns of the square, multiplied out, and the other limits of the walk.  (These checks are made by every wave of
        // a tile: as comparisons one by one they cost a 1599x901 frame of 32x16 tiles 1.3 %.  A NaN that max drops makes one of
        // the sum.)
        const float limit = kSteep ? kSharpest : 3.0f;
        const float reach = __builtin_fabsf(ex) + 8.0f;         // of the square's columns from the centre
        const float beyond = __builtin_fmaf(__builtin_fmaf(co.y, co.y, -4.0f * co.x * co.z) * reach, reach, 4.0f * co.z * (kMostExponent - co.w));
        const bool fits = __builtin_fmaxf(__builtin_fmaxf(beyond, co.z), __builtin_fmaxf(-limit - co.z, co.w - kMostExponent)) <= 0.0f &&
                          __builtin_fabsf(c) + __builtin_fabsf(bx) + __builtin_fabsf(by) + __builtin_fabsf(co.x) < 1.0e9f;
        float over = 0.0f;
        if constexpr (kRun) {
            // Any exponent above kSlightlyAbove: over the columns, multiplied out by 4 cz < 0.  cz = 0, where over is 0 too unless
            // cy makes it more, is one; what does not fit is looked at below.
            const float w = kFp32 ? co.w : co.w - kWeightScaleLog2;
            over = __builtin_fmaf(__builtin_fmaf(co.y, co.y, -4.0f * co.x * co.z) * reach, reach, 4.0f * co.z * (kSlightlyAbove - w));
            above = above || ballot(!(__builtin_fmaxf(over, w - kSlightlyAbove) < 0.0f)) != 0;
        }
        if (ballot(!fits) != 0) {
            if constexpr (!kSteep) return base;
            if constexpr (kRun) above = above || ballot(!(over < 0.0f && co.z < 0.0f)) != 0;     // (NaN too)
            const int walked = walk_plain<kFp32>(xy, co, rgb, cnt, left, top, stop_below, T, sums);
            if (walked < 0) return ~(base + ~walked);
            fetch();
            continue;
        }
        if (cnt < kChunk) {                     // (a branch, not selects for every chunk)
            asm volatile("");
            if (lane >= cnt) {                  // a slot past the end of the list: every weight is zero, and so is
                c = -1.0e30f;                   // the colour, or the weight would make NaN of an infinite one
                rgb = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
        }
        const float ratio = kSteep ? 2.0f * co.z : __builtin_amdgcn_exp2f(2.0f * co.z);
        __builtin_amdgcn_wave_barrier();
        {
            const Parts pcz = parts_of(co.z), pcy = parts_of(co.y);
            float4* const record = reinterpret_cast<float4*>(bytes + lane * kRecord);
            record[0] = slots_of(parts_of(c), parts_of(bx));
            record[1] = slots_of(parts_of(by), parts_of(co.x));
            record[2] = slots_of(pcz, pcy);
            record[3] = slots_of(parts_of(by + co.z), pcy);
            const Parts twice = {2.0f * pcz.hi, 2.0f * pcz.mid, 2.0f * pcz.lo}, none = {0.0f, 0.0f, 0.0f};
            record[4] = slots_of(twice, none);
            if constexpr (kFp32) {
                *reinterpret_cast<float4*>(bytes + kColours + 16 * lane) = make_float4(rgb.x, rgb.y, rgb.z, ratio);
            } else {
                _Float16* const colour = reinterpret_cast<_Float16*>(bytes + kColours + 32 * (lane >> 2)) + (lane & 3);
                colour[0] = (_Float16)clamped_to_f16(rgb.x);
                colour[4] = (_Float16)clamped_to_f16(rgb.y);
                colour[8] = (_Float16)clamped_to_f16(rgb.z);
                colour[12] = (_Float16)0.0f;
                *reinterpret_cast<float*>(bytes + kRatios + 4 * lane) = ratio;
            }
        }
        __builtin_amdgcn_wave_barrier();
        fetch();

        const char* record = bytes + role.record_at;
        uint32_t colour_off = kColours + (kFp32 ? 0 : 8 * (lane & 3));
        asm volatile("" : "+v"(colour_off));            // a vector register: LDS addresses are not scalars
        const char* colour_at = bytes + colour_off;
        const char* ratio_at = bytes + kRatios;
#pragma unroll 1
        for (int from = 0; from < cnt; from += kBatch) {
            float16_t q, d;
            {
                bf16x8_t slots[5], right[3];        // the same two coordinates for the three parts
#pragma unroll
                for (int m = 0; m < 3; m++) {
                    float both = role.right[m];
                    asm volatile("" : "+v"(both));      // copied here and not kept in three registers throughout
                    right[m] = __builtin_bit_cast(bf16x8_t, make_float4(both, both, both, 0.0f));
                }
#pragma unroll
                for (int m = 0; m < 5; m++) slots[m] = __builtin_bit_cast(bf16x8_t, lds_read<float4>(record + 16 * m));
                float16_t zero;
#pragma unroll
                for (int i = 0; i < 16; i++) zero[i] = 0.0f;
                q = __builtin_amdgcn_mfma_f32_32x32x16_bf16(slots[0], right[0], zero, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(slots[3], right[0], zero, 0, 0, 0);
                q = __builtin_amdgcn_mfma_f32_32x32x16_bf16(slots[1], right[1], q, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(slots[4], right[1], d, 0, 0, 0);
                q = __builtin_amdgcn_mfma_f32_32x32x16_bf16(slots[2], right[2], q, 0, 0, 0);
            }
            const int left_over = cnt - from;
            int upto;
            bool stopped = false;
            // the weights of Gaussian j of the batch along the strip
            auto weights = [&](int j, float E, float (&alpha)[4]) {
                alpha[0] = __builtin_amdgcn_exp2f(q[j]);
                if constexpr (kSteep) {         // (E is the slope's step)
                    float at = q[j] + d[j], slope = d[j] + E;
                    alpha[1] = __builtin_amdgcn_exp2f(at);
                    at += slope; slope += E;
                    alpha[2] = __builtin_amdgcn_exp2f(at);
                    alpha[3] = __builtin_amdgcn_exp2f(at + slope);
                } else {
                    float rho = __builtin_amdgcn_exp2f(d[j]);
                    // (zero times anything is zero here: a slope beyond the range of fp32 belongs to a value of zero)
                    alpha[1] = mul_zero_wins(alpha[0], rho); rho *= E;
                    alpha[2] = mul_zero_wins(alpha[1], rho); rho *= E;
                    alpha[3] = mul_zero_wins(alpha[2], rho);
                }
            };
            if constexpr (kFp32) {
                // render.cu:46-52, operation for operation.  T -= at stays a subtraction: the product is there for the
                // colours anyway, and v_fma_f32 with a negated and a repeated operand takes the issue of about two
                // v_sub_f32 (4K frame of 3M 290 -> 283 us, 8K of 8M 693 -> 674, 1080p of 1M 141 -> 136; errors against
                // float64 the same to three digits).
                auto shade = [&](int j, const float4& u) {
                    float alpha[4], at[4];
                    weights(j, u.w, alpha);
                    // The sums of a strip's even pixels in even registers and their factor in an odd one, those of the odd pixels the other way
                    // round, so no multiply-add reads three registers of one kind (paired; five in twelve did): 4K frame of 3M 619 -> 597 thousand
                    // cycles, of which the power limit leaves half (2.06 -> 2.04 GHz).  Whole frames: 4K / 3M 624.6 -> 621.2 us, 8K / 8M 1400 ->
                    // 1393, 110M pairs 3432 -> 3424, 1599x901 in 32x16 tiles 183.8 -> 182.
#pragma unroll
                    for (int p = 0; p < 4; p += 2) {
                        at[p] = alpha[p] * T[p];
                        at[p + 1] = alpha[p + 1] * T[p + 1];
                        paired(at[p + 1], at[p]);
#pragma unroll
                        for (int k = p; k < p + 2; k++) {
                            sums.r[k] += u.x * at[k];
                            sums.g[k] += u.y * at[k];
                            sums.b[k] += u.z * at[k];
                            T[k] -= at[k];
                        }
                        paired(sums.r[p], sums.r[p + 1]);
                        paired(sums.g[p], sums.g[p + 1]);
                        paired(sums.b[p], sums.b[p + 1]);
                    }
                };
                auto colour = [&](int j) { return lds_read<float4>(colour_at + 16 * j); };
                // Gaussians go in pairs, the stop is tested after each pair; a colour is read while the
                // Gaussian ahead of it is shaded.  The second half of an odd tail (render.cu:486-487) is an
                // unused slot: its weights and its colour are zero.
#define FGS_PAIR(J)                                                                    \
                second = colour((J) + 1);                                                  \
                shade((J), first);                                                         \
                first = colour(((J) + 2) % kBatch);     /* past the batch: read and dropped */ \
                shade((J) + 1, second);                                                    \
                upto = (J) + 2;                                                            \
                if (upto >= left_over || all_stopped(T, stop_below)) break;
                static_assert(kBatch == 16, "the pairs below cover a batch of 16");
                float4 first = colour(0), second;
                do {
                    FGS_PAIR(0) FGS_PAIR(2) FGS_PAIR(4) FGS_PAIR(6) FGS_PAIR(8) FGS_PAIR(10) FGS_PAIR(12) FGS_PAIR(14)
                } while (0);
#undef FGS_PAIR
            } else {
                uint32_t packed[4][2];        // f16 weights of the group's Gaussians 0-1 and 2-3, per pixel
                float w0[4], w1[4];
                auto shade = [&](int j, float E, float (&w)[4]) {
                    float alpha[4];
                    weights(j, E, alpha);
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        w[k] = alpha[k] * T[k];
                        T[k] = __builtin_fmaf(w[k], -kWeightUnscale, T[k]);
                    }
                };
                auto pack = [&](int half) {
#pragma unroll
                    for (int k = 0; k < 4; k++) packed[k][half] = pack_f16(w0[k], w1[k]);
                };
                // a stop behind the first pair of a group: the second pair's weights are zero
#define FGS_GROUP(G)                                                                         \
                {                                                                            \
                    const float2 colours = lds_read<float2>(colour_at + 32 * (G));           \
                    const float4 E = lds_read<float4>(ratio_at + 16 * (G));                  \
                    shade(4 * (G), E.x, w0);                                                 \
                    shade(4 * (G) + 1, E.y, w1);                                             \
                    pack(0);                                                                 \
                    upto = 4 * (G) + 2;                                                      \
                    _Pragma("unroll") for (int k = 0; k < 4; k++) packed[k][1] = 0u;         \
                    if (upto < left_over && !all_stopped(T, stop_below)) {                   \
                        shade(4 * (G) + 2, E.z, w0);                                         \
                        shade(4 * (G) + 3, E.w, w1);                                         \
                        pack(1);                                                             \
                        upto = 4 * (G) + 4;                                                  \
                    }                                                                        \
                    accumulate_f16(sums, packed, colours);                                   \
                    if (upto >= left_over || all_stopped(T, stop_below)) break;              \
                }
                do { FGS_GROUP(0) FGS_GROUP(1) FGS_GROUP(2) FGS_GROUP(3) } while (0);
#undef FGS_GROUP
            }
            stopped = all_stopped(T, stop_below);
            if (stopped) return ~min(base + from + upto, n);
            record += role.record_step;
            colour_at += kFp32 ? 16 * kBatch : 8 * kBatch;
            ratio_at += 4 * kBatch;
        }
    }
    return n;
}

// One wave blends entries [begin, begin + n) of the sorted list into the 16x16 pixels whose first pixel
// is (left, top), front to back, on top of T and sums; begin must be an even distance from the start
// of the tile's list, so that the pairs are the reference's pairs.  The walk ends after the pair behind
// which all 256 pixels have T < stop_below (render.cu:394-408).  Returns the entries walked, or ~entries
// when that stop ended the walk.  stage: this wave's kStageFloats of LDS.
template <bool kFp32, bool kRun>
__device__ __forceinline__ int walk_list(
    const LaneRole& role, float* stage,
    const uint32_t* __restrict__ point_list, int begin, int n,
    float left, float top,
    const float2* __restrict__ points_xy,
    const float4* __restrict__ rgb_depth,
    const float4* __restrict__ conic_opacity,
    float (&T)[4], Sums<kFp32>& sums, int stop_below, bool& above)
{
    const int lane = role.lane;
    Ahead next = {};
    if (n > 0) {
        const uint32_t last = (uint32_t)begin + (uint32_t)n - 1u;
        const uint32_t g = point_list[min((uint32_t)begin + (uint32_t)lane, last)];
        next.index = point_list[min((uint32_t)begin + kChunk + (uint32_t)lane, last)];
        next.xy = points_xy[g]; next.co = conic_opacity[g]; next.rgb = rgb_depth[g];
    }
    const int walked = walk_chunks<kFp32, false, kRun>(role, stage, point_list, begin, n, left, top, points_xy, rgb_depth, conic_opacity,
                                                 T, sums, stop_below, next, 0, above);
    if (walked < 0 || walked >= n) return walked;
    return walk_chunks<kFp32, true, kRun>(role, stage, point_list, begin, n, left, top, points_xy, rgb_depth, conic_opacity,
                                    T, sums, stop_below, next, walked, above);
}

// The wave's pixels out of T and the colour sums.
template <bool kFp32>
__device__ __forceinline__ void finish(float* stage, const float (&T)[4], const Sums<kFp32>& sums, Pixels& px)
{
#pragma unroll
    for (int k = 0; k < 4; k++) px.T[k] = T[k];
    if constexpr (kFp32) {
#pragma unroll
        for (int k = 0; k < 4; k++) { px.r[k] = sums.r[k]; px.g[k] = sums.g[k]; px.b[k] = sums.b[k]; }
    } else {
        // Lane 4b+j holds channel j of the pixels of lanes 4b .. 4b+3: handed back through the
        // staging area (a block of 16 x 4 floats per four lanes, padded to 68 so that the stores of
        // the 32 lanes served together fall into different banks).
        const int lane = lane_id();
        __builtin_amdgcn_wave_barrier();
        char* const out = reinterpret_cast<char*>(stage) + 4 * ((lane >> 2) * 68 + (lane & 3));
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int r = 0; r < 4; r++) lds_write(out + 4 * (r * 16 + k * 4), sums.acc[k][r]);
        __builtin_amdgcn_wave_barrier();
        const char* const in = reinterpret_cast<const char*>(stage) + 4 * ((lane >> 2) * 68 + (lane & 3) * 16);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float4 c = lds_read<float4>(in + 16 * k);
            px.r[k] = c.x * kWeightUnscale;
            px.g[k] = c.y * kWeightUnscale;
            px.b[k] = c.z * kWeightUnscale;
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// render.cu:59-73; (left, top): first pixel of the wave's 16x16 square
__device__ __forceinline__ void write_square(
    int lane, int left, int top, int width, int height, const Pixels& px,
    float bg_r, float bg_g, float bg_b, uint8_t* __restrict__ out_u8, float* __restrict__ out_f32)
{
    asm volatile("" : "+v"(lane));      // what follows from it is computed here, not kept through the walk
#pragma unroll
    for (int k = 0; k < 4; k++) {
        int x, y;
        pixel_of(lane, k, &x, &y);
        x += left; y += top;
        if (x < width && y < height) {
            const size_t pid = (size_t)width * y + x;
            float t = px.T[k];
            if (t < 0.0001f) t = 0.0f;
            const float r = px.r[k] + t * bg_r, g = px.g[k] + t * bg_g, b = px.b[k] + t * bg_b;
            if (out_u8) {
                out_u8[3 * pid + 0] = encode_u8(r);
                out_u8[3 * pid + 1] = encode_u8(g);
                out_u8[3 * pid + 2] = encode_u8(b);
            }
            if (out_f32) {
                out_f32[3 * pid + 0] = r;
                out_f32[3 * pid + 1] = g;
                out_f32[3 * pid + 2] = b;
            }
        }
    }
}

#define FGS_BLEND_PARAMS                                                                         \
    const int2* __restrict__ ranges, const uint32_t* __restrict__ point_list,                   \
    int width, int height, int tiles_x, int tiles_y,                                            \
    const float2* __restrict__ points_xy, const float4* __restrict__ rgb_depth,                 \
    const float4* __restrict__ conic_opacity, float bg_r, float bg_g, float bg_b,               \
    uint8_t* __restrict__ out_u8, float* __restrict__ out_f32

template <bool kFp32>
constexpr int kBlendWaves = kFp32 ? 5 : 4;       // resident waves per SIMD

// One workgroup per tile, one wave per 16x16 square of it (1 for 16x16 tiles, 2 for 32x16, 4 for
// 32x32); the waves of a wide tile walk the same list and find its lines in their CU's cache.  (One
// wave for a whole 32x32 tile needs 64 registers for its colour sums, leaves two waves per SIMD, and
// a frame of 3600 such tiles ends with the longest lists on single waves: 1200 us for 1M Gaussians
// at 2560x1440 against 377 us; 32x16 tiles at 1599x901 384 against 217.)  The stop is the tile's, not the
// wave's: a wave that finds its own square stopped waits until all have, those that stopped
// earlier than the last one walk on to where it did, and the tile stops there if all are still opaque.
// Resident waves: 5 per SIMD is what 96 registers allow (4: the same time on the largest frames, 3 to 5 %
// more on the others; 6 spills).
template <int SX, int SY, bool kFp32>
__global__ __launch_bounds__(kWave * SX * SY) __attribute__((amdgpu_waves_per_eu(kBlendWaves<kFp32>, kBlendWaves<kFp32>))) void blend_kernel(FGS_BLEND_PARAMS,
    const LongLists* __restrict__ longer, LongLists* __restrict__ next_longer, int long_list, int long_per_shard)
{
    constexpr int kSquares = SX * SY;
    __shared__ __align__(16) float s_stage[kSquares][kStageFloats];
    __shared__ int s_walked[kSquares], s_stopped[kSquares];

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = kSquares == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    int tile_x, tile_y;
    const int long_lists = longer ? kLongShards * long_per_shard : 0;
    const bool first = (int)blockIdx.x < long_lists;
    if (first) {
        const uint32_t shard = blockIdx.x % kLongShards, at = blockIdx.x / kLongShards;
        if (at == 0 && threadIdx.x == 0) next_longer->count[shard] = 0;
        const uint32_t tile = longer->tiles[shard][at];
        if (at >= longer->count[shard] || tile >= (uint32_t)(tiles_x * tiles_y) || long_shard(tile) != shard) return;
        tile_x = (int)(tile % (uint32_t)tiles_x);
        tile_y = (int)(tile / (uint32_t)tiles_x);
    } else if (!tile_of_position((int)blockIdx.x - long_lists, tiles_x, tiles_y, &tile_x, &tile_y)) {
        return;
    }
    const uint32_t tile = (uint32_t)(tile_y * tiles_x + tile_x);
    const int2 range = ranges[tile];
    const int n = range.y - range.x;
    if (longer && !first && n >= long_list) {       // left to one of the first workgroups?
        const uint32_t shard = long_shard(tile), at = (uint32_t)lane;
        const bool listed = at < min(longer->count[shard], (uint32_t)long_per_shard) && longer->tiles[shard][at % kLongPerShard] == tile;
        if (ballot(listed) != 0) return;
    }
    // A launch ends when its longest list ends, and a wave that shares its SIMD equally with the
    // waves of short lists gets to its own end late: waves with long lists ask for a higher
    // issue priority.
    if (n > 1024) __builtin_amdgcn_s_setprio(3);
    else if (n > 512) __builtin_amdgcn_s_setprio(2);
    else if (n > 256) __builtin_amdgcn_s_setprio(1);

    LaneRole role;
    role.init(lane, s_stage[wave]);
    float T[4];
    Sums<kFp32> sums;
    clear<kFp32>(T, sums);
    const int left = (tile_x * SX + wave % SX) * 16, top = (tile_y * SY + wave / SX) * 16;
    int done = 0, upto = n;
    int stop_below = kStopBelow;
    for (;;) {
        bool above;
        const int walked = walk_list<kFp32, false>(role, s_stage[wave], point_list, range.x + done, upto - done, (float)left, (float)top,
                                                   points_xy, rgb_depth, conic_opacity, T, sums, stop_below, above);
        if (kSquares == 1) break;
        done += walked < 0 ? ~walked : walked;
        if (stop_below == kStopBelow) {
            if (lane == 0) s_walked[wave] = done;
            __syncthreads();
            upto = 0;
#pragma unroll
            for (int w = 0; w < kSquares; w++) upto = max(upto, s_walked[w]);
            upto = __builtin_amdgcn_readfirstlane(upto);
            stop_below = kNeverStop;        // to where the last one stopped
            if (done < upto) continue;
        }
        // All waves are at the same pair, the first one behind which the tile can stop.  A weight above 1
        // turns the sign of T: then a square that had stopped need not be opaque any more.
        if (upto >= n) break;
        const bool stopped = all_stopped(T, kStopBelow);
        if (lane == 0) s_stopped[wave] = stopped;
        __syncthreads();
        bool all = true;
#pragma unroll
        for (int w = 0; w < kSquares; w++) all = all && s_stopped[w] != 0;
        if (__builtin_amdgcn_readfirstlane(all)) break;
        upto = n;
        stop_below = kStopBelow;
    }
    Pixels px;
    finish<kFp32>(s_stage[wave], T, sums, px);
    write_square(lane, left, top, width, height, px, bg_r, bg_g, bg_b, out_u8, out_f32);
}

// Frames of at most kOrderCap tiles.  Such a frame is about resident at once, and a wave alone on its SIMD issues one
// instruction in seven cycles, 104 ns per entry, where five waves issue one in three: the launch lasted as long as its
// longest lists on single waves (32x16 tiles, 1599x901: 60 us of issue, 236 us for 2465 entries).  So the tiles are ranked by list
// length, the longest start first, and those that are long for this frame (tile_order_kernel) have a workgroup of kT teams, one wave per
// 16x16 square each, to themselves; all other tiles have a team each, without a word to the others of the workgroup
// (one wave per square: a wave for a whole 32x32 tile needs 64 registers for its colour sums).
//
// A long list is walked in rounds.  Its first kHead entries are walked by the first team, since what stops there (opaque
// content mostly does) shall cost the others nothing.  Then every team takes a run of the entries that follow, from T = 1, C = 0, and
// the owner folds them front to back, C += T C_run, T *= T_run.  A round is kRoundRuns runs, whatever the number of teams, so a
// list is cut alike in every frame; they are kHead entries long at first and twice as long with every round, so that what
// is walked past a stop stays a fraction of the list.  The tile's stop is looked for behind
// every run, from the products of T.  The run that has it is walked once more by the owner, on top of what was in front of it and with
// the stop tested behind every pair, so the image ends where the reference's walk ends.  (Weights do not exceed
// 1, so T only falls and a stop shows at the end of the run that has it; a run with an exponent above zero in it, which can
// turn the sign of T, is walked that way too, and so is a run behind T of some pixel above 1 or below
// kLeastInFront: there a run's own stop is not the tile's, and the tile's need not last to the end of the run.)
//
// Against a wave per square that shared (16x16 tiles only) from 768 entries on among the four tiles of a workgroup: 32x16 at 1599x901
// 237 -> 115 us, 32x32 at 2560x1440 1M 321 -> 277, at 640x512 1M 1873 -> 943; 16x16 1080p 1M 145 -> 126, 700k 104 -> 92, 1365x767 300k
// 80 -> 58, 1280x720 with long lists everywhere 224 -> 86, with short ones 30 -> 31, 256x192 300k 227 -> 181, 4K 32x32 city 789 -> 788,
// needles that make every tile opaque 45 -> 45 at 1080p and 33 -> 40 at 1024x700.  (What a round costs beside its walk is some
// 2 us; 15 with the owner's state in volatile private memory, whose loads wait for each other.)  Shared from a quarter or a half of the average on
// instead of three eighths: 1080p 141 and 132, 32x32 276 and 325; heads of 128 or 256 entries: 1080p 127 and 123, 1280x720 98
// and 148 (64: 121 and 98, all with rounds of as many runs as teams); rounds of four runs: 32x16 108, 1280x720 98, 256x192 206.
//
// Unranked (stream capture, no memory, all workgroups resident at once) every team has a tile and long lists are shared with the others of the workgroup, cut as
// they are with a table.  What a team has blended of its own tile waits in private memory meanwhile.
constexpr int kHead = 64, kMostRun = 512, kRoundRuns = 8;
// resident waves per SIMD: whole workgroups
template <bool kFp32>
constexpr int shared_waves(int of_workgroup) { return of_workgroup > 8 ? of_workgroup / 4 : kBlendWaves<kFp32>; }

template <int SX, int SY, int kT, bool kFp32>
__global__ __launch_bounds__(kWave * SX * SY * kT) __attribute__((amdgpu_waves_per_eu(shared_waves<kFp32>(SX * SY * kT), shared_waves<kFp32>(SX * SY * kT))))
void blend_kernel_shared(FGS_BLEND_PARAMS, const uint32_t* __restrict__ tile_order, int tiles_per_group, int simds)
{
    constexpr int kSquares = SX * SY, kWaves = kSquares * kT;
    constexpr int kHandOver = 4 * 4 * kWave;            // a run's result: 4 pixels x 4 floats per lane
    __shared__ __align__(16) float s_stage[kWaves][kStageFloats > kHandOver ? kStageFloats : kHandOver];
    __shared__ int s_walked[kWaves], s_stopped[kWaves], s_above[2][kT];
    __shared__ int s_tile[kT][4];                       // of every team: first pixel, first pair, pairs
    __shared__ int s_rest[kT];                          // 1: pairs left for all teams, 3: and T of the first run is outside

    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int team = wave / kSquares, square = wave % kSquares;
    static_assert(kLeastShared >= 2 * kHead, "a rest worth sharing behind the head");
    const int num_tiles = tiles_x * tiles_y, group = (int)blockIdx.x;
    // Ranked: the tiles with long lists have a workgroup each, tiles_per_group teams of the others have a tile, and nothing
    // is shared where a team without one has left.
    int rank = team * (int)gridDim.x + group, least, teams = kT;
    bool active = team < tiles_per_group;
    if (tile_order) {
        const int alone = (int)tile_order[kOrderCap];
        const int first = group < alone ? group : alone + (group - alone) * tiles_per_group;
        if (first >= num_tiles) return;
        if (group >= alone && team >= tiles_per_group) return;
        teams = group < alone ? kT : tiles_per_group;
        rank = first + team;
        active = group >= alone || team == 0;
        least = (int)tile_order[kOrderCap + 1];
    } else {
        least = least_shared(RangeLength{ranges}, num_tiles, kSquares, simds);
    }
    active = active && rank < num_tiles;
    int tile_x = 0, tile_y = 0;
    int2 range = make_int2(0, 0);
    if (active) {
        const int tile = tile_order ? (int)tile_order[rank] : rank;
        tile_x = tile % tiles_x;
        tile_y = tile / tiles_x;
        range = ranges[tile];
    }
    int n = range.y - range.x, begin = range.x;         // of the tile that is walked
    if (lane == 0 && square == 0) {
        s_tile[team][0] = tile_x * SX * 16;
        s_tile[team][1] = tile_y * SY * 16;
        s_tile[team][2] = begin;
        s_tile[team][3] = n;
        s_above[0][team] = 0;
        s_above[1][team] = 0;
        s_rest[team] = 0;
    }
    if (n > 256) __builtin_amdgcn_s_setprio(1);
    LaneRole role;
    role.init(lane, s_stage[wave]);
    __syncthreads();
    bool share = false;                                 // some list of the workgroup is long
#pragma unroll
    for (int t = 0; t < kT; t++) share = share || (t < teams && s_tile[t][3] >= least);
    share = teams == kT && __builtin_amdgcn_readfirstlane(share);

    const int square_x = square % SX * 16, square_y = square / SX * 16;
    int left = tile_x * SX * 16 + square_x, top = tile_y * SY * 16 + square_y;
    float T[4];
    Sums<kFp32> sums;
    clear<kFp32>(T, sums);
    // The wave's own square while it works on runs: in private memory (its address is given away), not in registers.
    float4_t kept[4];
    asm volatile("" : : "v"((__attribute__((address_space(5))) float4_t*)&kept[0]) : "memory");
    auto result = [&](float4_t (&p)[4]) {               // of the walk
        Pixels px;
        finish<kFp32>(s_stage[wave], T, sums, px);
#pragma unroll
        for (int k = 0; k < 4; k++) p[k] = float4_t{px.r[k], px.g[k], px.b[k], px.T[k]};
    };
    auto keep = [&](const float4_t (&p)[4]) {
#pragma unroll
        for (int k = 0; k < 4; k++) kept[k] = p[k];
        asm volatile("" : : : "memory");
    };
    auto recall = [&](float4_t (&p)[4]) {
#pragma unroll
        for (int k = 0; k < 4; k++) p[k] = kept[k];
    };
    // Whether a pixel's T is outside what a run may start from (see above).  It can be only behind entries that were walked
    // one after the other, and is looked at there: before every fold it was 2 % of the blend of frames of some thousand tiles.
    auto outside = [&]() {
        const float most = __builtin_fmaxf(__builtin_fmaxf(T[0], T[1]), __builtin_fmaxf(T[2], T[3]));
        const float fewest = __builtin_fminf(__builtin_fminf(T[0], T[1]), __builtin_fminf(T[2], T[3]));
        return ballot(most > 1.0f || fewest < kLeastInFront) != 0;
    };
    enum { kOwn, kRuns, kAgain };
    int mode = kOwn, v = -1;                            // v: the team whose tile is shared
    int end = share && n >= least ? kHead : n;           // of the walk of entries one after the other
    int from = 0, upto = end, stop_below = kStopBelow;
    int pos = 0, cap = 0, len = 0, left_runs = 0, step = 0;         // runs start at pos and are len long, at most cap; left_runs of a round
    for (;;) {
        bool above = false;
        int walked = 0;
        if (upto > from)
            walked = walk_list<kFp32, true>(role, s_stage[wave], point_list, begin + from, upto - from, (float)left, (float)top,
                                            points_xy, rgb_depth, conic_opacity, T, sums, stop_below, above);
        bool next_tile = false;
        if (mode == kRuns) {
            {
                float4_t p[4];
                result(p);
                float4_t* const mine = reinterpret_cast<float4_t*>(s_stage[wave]);
#pragma unroll
                for (int k = 0; k < 4; k++) mine[k * kWave + lane] = p[k];
            }
            if (above && lane == 0) s_above[step & 1][team] = 1;
            __syncthreads();
            if (team == v) {
                float t[4] = {kept[0][3], kept[1][3], kept[2][3], kept[3][3]};
                int mask = 0;
#pragma unroll
                for (int j = 0; j < kT; j++) {
                    const float4_t* const part = reinterpret_cast<const float4_t*>(s_stage[j * kSquares + square]);
#pragma unroll
                    for (int k = 0; k < 4; k++) t[k] *= part[k * kWave + lane][3];
                    if (all_stopped(t, kStopBelow)) mask |= 1 << j;
                }
                if (lane == 0) s_stopped[square] = mask;
            }
            __syncthreads();
            int mask = s_stopped[0];
#pragma unroll
            for (int q = 1; q < kSquares; q++) mask &= s_stopped[q];
#pragma unroll
            for (int j = 0; j < kT; j++) mask |= s_above[step & 1][j] != 0 ? 1 << j : 0;
            mask = __builtin_amdgcn_readfirstlane(mask);
            const int taken = mask ? __builtin_ctz(mask) : kT;
            if (team == v) {
                float4_t p[4];
                recall(p);
                for (int j = 0; j < taken; j++) {
                    const float4_t* const part = reinterpret_cast<const float4_t*>(s_stage[j * kSquares + square]);
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const float4_t run = part[k * kWave + lane];
                        const float t = p[k][3];
                        p[k] = float4_t{p[k][0] + t * run[0], p[k][1] + t * run[1], p[k][2] + t * run[2], t * run[3]};
                    }
                }
                keep(p);
            }
            step++;
            if (lane == 0 && square == 0) s_above[step & 1][team] = 0;
            const int runs = min(taken, left_runs);
            pos = min(n, pos + runs * len);
            left_runs -= runs;
            if (taken == kT) {
                next_tile = pos >= n;
            } else {
                // run `taken` has the tile's stop in it or weights above one: its team walks it
                mode = kAgain;
                clear<kFp32>(T, sums);
                from = pos;
                end = min(n, pos + len);
                upto = team == v ? end : pos;
                stop_below = kStopBelow;
                if (team == v) {
#pragma unroll
                    for (int k = 0; k < 4; k++) T[k] = kept[k][3];
                }
            }
            __syncthreads();                            // the parts have been read
            if (mode == kAgain) continue;
        } else {
            // entries one after the other
            from += walked < 0 ? ~walked : walked;
            bool stopped = walked < 0;
            const bool bystander = mode == kAgain && team != v;
            if (kSquares == 1) {
                if (mode == kOwn && !share) break;
                if (mode == kAgain) {
                    if (team == v && lane == 0) s_stopped[0] = stopped;
                    __syncthreads();
                    stopped = __builtin_amdgcn_readfirstlane(s_stopped[0]) != 0;
                }
            } else {
                // The stop is the tile's: a square that has stopped waits until all have, those that stopped earlier than the last
                // one walk on to where it did, and the tile stops there if all are still opaque (a weight above 1 turns
                // the sign of T: then a square that had stopped need not be opaque any more).
                const int first = (mode == kAgain ? v : team) * kSquares;      // the tile's waves
                if (stop_below == kStopBelow) {
                    if (lane == 0) s_walked[wave] = from;
                    __syncthreads();
                    int furthest = 0;
#pragma unroll
                    for (int q = 0; q < kSquares; q++) furthest = max(furthest, s_walked[first + q]);
                    upto = __builtin_amdgcn_readfirstlane(furthest);
                    if (bystander) from = upto;
                    stop_below = kNeverStop;
                    continue;
                }
                // 1: opaque, 2: at the end
                const bool opaque = all_stopped(T, kStopBelow);
                if (lane == 0) s_stopped[wave] = bystander ? 3 : (opaque ? 1 : 0) | (upto >= end ? 2 : 0);
                __syncthreads();
                int state = 3;
                bool unfinished = false;
#pragma unroll
                for (int t = 0; t < kT; t++) {
                    int of_team = 3;
#pragma unroll
                    for (int q = 0; q < kSquares; q++) of_team &= s_stopped[t * kSquares + q];
                    unfinished = unfinished || (t < teams && of_team == 0);
                    if (t * kSquares == first) state = of_team;
                }
                state = __builtin_amdgcn_readfirstlane(state);
                __syncthreads();                        // read before they are written again
                stopped = (state & 1) != 0;
                stop_below = kStopBelow;
                if (__builtin_amdgcn_readfirstlane(unfinished)) {
                    upto = state != 0 || bystander ? from : end;        // (a finished tile stays where it is)
                    continue;
                }
                if (mode == kOwn && !share) break;
            }
            if (mode == kOwn) {
                if (!stopped && n >= least) {
                    const int rest = outside() ? 3 : 1;
                    if (lane == 0) atomicOr(&s_rest[team], rest);
                }
                __syncthreads();
                int rests = 0;
#pragma unroll
                for (int t = 0; t < kT; t++) rests |= s_rest[t];
                if (__builtin_amdgcn_readfirstlane(rests) == 0) break;
                float4_t p[4];
                result(p);
                keep(p);
                next_tile = true;
            } else {
                if (team == v) {
                    float4_t p[4], before[4];
                    result(p);
                    recall(before);
#pragma unroll
                    for (int k = 0; k < 4; k++) p[k] += float4_t{before[k][0], before[k][1], before[k][2], 0.0f};
                    keep(p);
                    const bool serial = outside();
                    if (serial && lane == 0 && end < n) s_above[step & 1][0] = 1;        // as if the next run had weights above 1
                }
                pos = end;
                left_runs--;
                next_tile = stopped || end >= n;
                __syncthreads();                        // s_stopped has been read
            }
        }
        if (next_tile) {
            int rest = 0;
            while (++v < kT && (rest = __builtin_amdgcn_readfirstlane(s_rest[v])) == 0) {}
            if (v == kT) break;
            if ((rest & 2) != 0 && wave == 0 && lane == 0) s_above[step & 1][0] = 1;
            __builtin_amdgcn_s_setprio(3);
            left = __builtin_amdgcn_readfirstlane(s_tile[v][0]) + square_x;
            top = __builtin_amdgcn_readfirstlane(s_tile[v][1]) + square_y;
            begin = __builtin_amdgcn_readfirstlane(s_tile[v][2]);
            n = __builtin_amdgcn_readfirstlane(s_tile[v][3]);
            pos = kHead;
            cap = kHead / 2;
            left_runs = 0;
        }
        mode = kRuns;
        if (left_runs == 0) {
            left_runs = kRoundRuns;
            cap = min(2 * cap, kMostRun);
            len = min(cap, ((n - pos + kRoundRuns - 1) / kRoundRuns + 15) & ~15);
        }
        from = team < left_runs ? min(n, pos + team * len) : n;
        upto = min(n, from + len);
        stop_below = kSquares == 1 ? kStopBelow : kNeverStop;
        clear<kFp32>(T, sums);
    }
    float4_t p[4];
    if (v >= 0) recall(p);
    else result(p);
    Pixels px;
#pragma unroll
    for (int k = 0; k < 4; k++) { px.r[k] = p[k][0]; px.g[k] = p[k][1]; px.b[k] = p[k][2]; px.T[k] = p[k][3]; }
    if (active) write_square(lane, tile_x * SX * 16 + square_x, tile_y * SY * 16 + square_y, width, height, px, bg_r, bg_g, bg_b, out_u8, out_f32);
}
#undef FGS_BLEND_PARAMS

// How the colour sums are formed by the entry points that do not say (see fgs_set_colour_sums).
std::atomic<int> g_colour_sums{FGS_COLOUR_SUMS_FP32};

// The mode of one call: what its flags ask for, else the process default.
int colour_mode(int flags, int* mode, const char* who)
{
    if (flags & ~(FGS_BLEND_FP32 | FGS_BLEND_MATRIX_F16)) return fail(FGS_E_INVALID, "%s: unknown flags 0x%x", who, flags);
    if ((flags & FGS_BLEND_FP32) && (flags & FGS_BLEND_MATRIX_F16))
        return fail(FGS_E_INVALID, "%s: FGS_BLEND_FP32 and FGS_BLEND_MATRIX_F16 exclude each other", who);
    *mode = (flags & FGS_BLEND_FP32) ? FGS_COLOUR_SUMS_FP32
          : (flags & FGS_BLEND_MATRIX_F16) ? FGS_COLOUR_SUMS_MATRIX_F16 : g_colour_sums.load();
    return FGS_OK;
}

int check_tile(int block_x, int block_y, int* sx, int* sy, const char* who)
{
    if ((block_x == 16 && block_y == 16) || (block_x == 32 && block_y == 16) || (block_x == 32 && block_y == 32)) {
        *sx = block_x / 16;
        *sy = block_y / 16;
        return FGS_OK;
    }
    return fail(FGS_E_INVALID, "%s: tile %dx%d unsupported (16x16, 32x16, 32x32)", who, block_x, block_y);
}

// A frame of at most kOrderCap tiles is about resident at once: its tiles are ranked by the length of
// their lists, the longest start first, and the long ones are shared out.  In a
// larger frame the short lists at any time fill in behind the long ones, and neighbouring tiles
// finding each other's lines in the L2 counts for more.
bool is_ranked(int tiles_x, int tiles_y) { return (long long)tiles_x * tiles_y <= kOrderCap; }

// Pairs from which on tile_ranges_sampled_kernel is the faster one, whatever the number of tiles and however unevenly the pairs
// lie in them (its second trip to memory costs 1.3 us): 1.4M pairs 4.1 us by every key and 5.4 by samples, 1.7M 4.4 and 5.7,
// 3.3M 6.0 and 5.3, 4.0M 7.2 and 5.8.
constexpr int kSampledPairs = 3 << 20;

// The table of the long lists of a frame whose tiles are not ranked; no list where there is none.
struct LongTable {
    LongLists *list = nullptr, *next = nullptr;
    int least = 0;
    int per_shard = kLongPerShard / 2;
    OrderTable* taken_from = nullptr;       // whose turn ends when a blend that clears `next` is enqueued
};

// A list is long for its frame if it has a seventh of the entries that a SIMD has on average: it takes 166 ns per entry beside others
// where a SIMD takes 50, so half of the launch.
// Only frames of kLongTiles tiles and more have such lists often enough (8K / 8M Gaussians, 129 600 tiles: ranges and blend 675 -> 625 us, 3 of the
// ranges' 23 for the listing; 6620x4058 / 29.6M pairs and 4797x3666 / 15.5M, where none ends late: 1 % more; before the listing cost that little:
// 57 600 tiles blend 444 -> 441 us and ranges 16.5 -> 19.1, 32 400 319 -> 320 and 12.3 -> 16.8), and none where a seventh is more than
// kLongMost entries: lists that long are opaque long before their end (110M pairs: 477 -> 479 and 88 -> 128).
constexpr int kLongTiles = 1 << 16, kLongLeast = 1024, kLongMost = 8192;
static_assert(kLongLeast > kRangeRuns * kWave, "a tile that tile_ranges_sampled_kernel lists goes on behind the wave's runs");
int long_table(hipStream_t stream, int num_rendered, int block_x, int block_y, int width, int height, LongTable* out, std::unique_lock<std::mutex>* enqueue)
{
    const int tiles_x = (width + block_x - 1) / block_x, tiles_y = (height + block_y - 1) / block_y;
    if ((long long)tiles_x * tiles_y < kLongTiles || num_rendered < kSampledPairs) return FGS_OK;        // (ranges marked from every key list none)
    int device = 0, cus = 0;
    FGS_HIP_TRY(hipGetDevice(&device));
    FGS_HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
    const long long seventh = (long long)num_rendered * (block_x / 16) * (block_y / 16) / (4 * cus) / 7;
    if (seventh > kLongMost) return FGS_OK;
    uint32_t* ranks = nullptr;
    OrderTable* entry = nullptr;
    int rc = tile_order_table(stream, &ranks, enqueue, &entry);
    if (rc != FGS_OK || !ranks) return rc;
    LongLists* const both = (LongLists*)(ranks + kOrderCap + 2);
    out->list = both + entry->turn;
    out->next = both + (entry->turn ^ 1);
    out->taken_from = entry;
    out->least = (int)std::max(seventh, (long long)kLongLeast);
    return FGS_OK;
}

// render.cu:556-563: zero the ranges, then mark where each tile starts and ends
int ranges_impl(int block_x, int block_y, int num_rendered, int width, int height,
                const uint64_t* keys_sorted, int* ranges, const LongTable& longer, void* stream, const char* who)
{
    if (num_rendered < 0) return fail(FGS_E_INVALID, "%s: num_rendered = %d is negative", who, num_rendered);
    if (width <= 0 || height <= 0 || block_x <= 0 || block_y <= 0)
        return fail(FGS_E_INVALID, "%s: width/height/block must be positive", who);
    if (!ranges || (num_rendered > 0 && !keys_sorted)) return fail(FGS_E_INVALID, "%s: null buffer", who);
    if (((uintptr_t)keys_sorted | (uintptr_t)ranges) % 8 != 0)
        return fail(FGS_E_INVALID, "%s: keys and ranges must be 8-byte aligned", who);
    const int tiles_x = (width + block_x - 1) / block_x, tiles_y = (height + block_y - 1) / block_y;
    const size_t num_tiles = (size_t)tiles_x * tiles_y;
    hipStream_t st = (hipStream_t)stream;
    const size_t words = num_tiles * 2;
    size_t fill_blocks = (words + 1023) / 1024;
    if (fill_blocks > 1024) fill_blocks = 1024;
    if (num_rendered == 0)
        hipLaunchKernelGGL(fill_i32_kernel, dim3((unsigned)fill_blocks), dim3(256), 0, st, ranges, words, 0);
    else if (num_rendered >= kSampledPairs)
        hipLaunchKernelGGL(longer.list ? tile_ranges_sampled_kernel<true> : tile_ranges_sampled_kernel<false>,
                           dim3((unsigned)(((size_t)num_rendered + 4 * kRangeRuns * kWave - 1) / (4 * kRangeRuns * kWave))),
                           dim3(256), 0, st, num_rendered, keys_sorted, (int2*)ranges,
                           (uint32_t)(num_tiles > 0xffffffffu ? 0xffffffffu : num_tiles), longer.list, longer.least);
    else
        hipLaunchKernelGGL(tile_ranges_kernel,
                           dim3((unsigned)(((size_t)num_rendered + 256 * kRangesPerThread - 1) / (256 * kRangesPerThread))),
                           dim3(256), 0, st,
                           num_rendered, keys_sorted, (int2*)ranges,
                           (uint32_t)(num_tiles > 0xffffffffu ? 0xffffffffu : num_tiles));
    return check_hip(hipGetLastError(), who);
}

// Teams of a workgroup of blend_kernel_shared, a divisor of kRoundRuns.  More of them where there are few tiles: 192 with
// 1811 entries on average 208 us by 4, 183 by 8; 475 with 760 152, 112; 950 with 1320 184, 149.  32x32 tiles: 247 with 4372 1137 by 2,
// 975 by 4.
int teams_of(int sx, int sy, int num_tiles, int cus)
{
    if (sx == 1 && sy == 1) return num_tiles > 4 * cus ? 4 : 8;
    if (sx == 2 && sy == 2) return num_tiles > cus ? 2 : 4;
    return 4;
}

// What a blend takes, checked before anything is launched for it.
int check_blend(int block_x, int block_y, int width, int height, const float* points_xy, const float* rgb_depth, const float* conic_opacity,
                const int* ranges, const float* bg, const uint8_t* out_u8, const float* out_f32, int flags, int* sx, int* sy, int* mode, const char* who)
{
    int rc = check_tile(block_x, block_y, sx, sy, who);
    if (rc != FGS_OK) return rc;
    rc = colour_mode(flags, mode, who);
    if (rc != FGS_OK) return rc;
    if (width <= 0 || height <= 0) return fail(FGS_E_INVALID, "%s: width/height must be positive", who);
    if (!ranges || !bg || (!out_u8 && !out_f32)) return fail(FGS_E_INVALID, "%s: null ranges, bg_color or output", who);
    if (((uintptr_t)rgb_depth | (uintptr_t)conic_opacity) % 16 != 0 ||
        ((uintptr_t)points_xy | (uintptr_t)ranges) % 8 != 0)
        return fail(FGS_E_INVALID, "%s: rgb_depth/conic_opacity must be 16-byte aligned, points_xy/ranges 8-byte aligned", who);
    if (positions_of((width + block_x - 1) / block_x, (height + block_y - 1) / block_y) > 0x7fffffffLL - kLongShards * kLongPerShard)
        return fail(FGS_E_INVALID, "%s: image too large", who);
    return FGS_OK;
}

// How the blend of a ranked frame is launched.
struct SharedGrid {
    int cus = 0, teams = 0, resident = 0;       // teams of a workgroup, workgroups that are resident at once
};
int shared_grid(int sx, int sy, int num_tiles, bool fp32, SharedGrid* out)
{
    int device = 0;
    FGS_HIP_TRY(hipGetDevice(&device));
    FGS_HIP_TRY(hipDeviceGetAttribute(&out->cus, hipDeviceAttributeMultiprocessorCount, device));
    out->teams = teams_of(sx, sy, num_tiles, out->cus);
    out->resident = out->cus * std::max(1, 4 * (fp32 ? kBlendWaves<true> : kBlendWaves<false>) / (sx * sy * out->teams));
    return FGS_OK;
}

// render.cu:566-575
// ranked: the table of ranks of a frame that is ranked already, whose lock the caller holds, or null.
// rank: a blend by itself (fgs_blend) is two launches, the ranking and the blend.  Behind the ranges of the same call (fgs_render)
// a frame whose workgroups are all resident at once even with one tile each goes unranked, since nothing starts later than
// anything else there; the image is the same bits.  256x192 / 2.8k pairs 11.1 -> 8.7 us, 348k pairs 181 -> 178, 400x300 / 362k
// 110 -> 107, opaque needles 110 -> 117, 700x600 in 32x32 tiles 114 -> 112.
int blend_impl(bool rank, uint32_t* ranked, const LongTable& longer, int block_x, int block_y, int width, int height,
               const float* points_xy, const float* rgb_depth, const float* conic_opacity,
               const uint32_t* values_sorted, const int* ranges, const float bg[3],
               uint8_t* out_u8, float* out_f32, int flags, void* stream, const char* who)
{
    int sx = 0, sy = 0, mode = 0;
    int rc = check_blend(block_x, block_y, width, height, points_xy, rgb_depth, conic_opacity, ranges, bg, out_u8, out_f32, flags, &sx, &sy, &mode, who);
    if (rc != FGS_OK) return rc;
    const int tiles_x = (width + block_x - 1) / block_x, tiles_y = (height + block_y - 1) / block_y;
    hipStream_t st = (hipStream_t)stream;
    // one workgroup per tile of the image padded to whole blocks of tiles, blocks padded to a multiple of 8
    const long long groups = positions_of(tiles_x, tiles_y);
    const int num_tiles = tiles_x * tiles_y;
    const bool fp32 = mode == FGS_COLOUR_SUMS_FP32;
#define FGS_BLEND_ARGS (const int2*)ranges, values_sorted, width, height, tiles_x, tiles_y,                     \
                       (const float2*)points_xy, (const float4*)rgb_depth, (const float4*)conic_opacity,        \
                       bg[0], bg[1], bg[2], out_u8, out_f32
    if (!is_ranked(tiles_x, tiles_y)) {
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)(groups + (longer.list ? kLongShards * longer.per_shard : 0))), dim3(kWave * sx * sy), 0, st, FGS_BLEND_ARGS,
                               (const LongLists*)longer.list, longer.next, longer.least, longer.per_shard);
        };
        if (sx == 1 && sy == 1) launch(fp32 ? blend_kernel<1, 1, true> : blend_kernel<1, 1, false>);
        else if (sx == 2 && sy == 1) launch(fp32 ? blend_kernel<2, 1, true> : blend_kernel<2, 1, false>);
        else launch(fp32 ? blend_kernel<2, 2, true> : blend_kernel<2, 2, false>);
        rc = check_hip(hipGetLastError(), who);
        if (rc == FGS_OK && longer.taken_from) longer.taken_from->turn ^= 1;
        return rc;
    }
    SharedGrid grid;
    rc = shared_grid(sx, sy, num_tiles, fp32, &grid);
    if (rc != FGS_OK) return rc;
    const int cus = grid.cus, teams = grid.teams, waves = sx * sy * teams, resident = grid.resident;
    uint32_t* tile_order = ranked;
    std::unique_lock<std::mutex> enqueue;       // from the ranking to the blend that reads it
    if (!ranked && (rank || num_tiles > resident)) {
        rc = tile_order_table(st, &tile_order, &enqueue);
        if (rc != FGS_OK) return rc;
    }
    if (tile_order && !ranked)
        hipLaunchKernelGGL(tile_order_kernel, dim3(1), dim3(1024), 0, st, (const int2*)ranges, num_tiles, tile_order, sx * sy, 4 * cus);
    auto launch = [&](auto kernel) {
        const int per_group = num_tiles <= resident ? 1 : teams;
        hipLaunchKernelGGL(kernel, dim3((unsigned)(tile_order ? num_tiles : (num_tiles + per_group - 1) / per_group)),
                           dim3(kWave * waves), 0, st, FGS_BLEND_ARGS, (const uint32_t*)tile_order, per_group, 4 * cus);
    };
    if (sx == 1 && sy == 1) {
        if (teams == 8) launch(fp32 ? blend_kernel_shared<1, 1, 8, true> : blend_kernel_shared<1, 1, 8, false>);
        else launch(fp32 ? blend_kernel_shared<1, 1, 4, true> : blend_kernel_shared<1, 1, 4, false>);
    } else if (sx == 2 && sy == 1) {
        launch(fp32 ? blend_kernel_shared<2, 1, 4, true> : blend_kernel_shared<2, 1, 4, false>);
    } else {
        if (teams == 4) launch(fp32 ? blend_kernel_shared<2, 2, 4, true> : blend_kernel_shared<2, 2, 4, false>);
        else launch(fp32 ? blend_kernel_shared<2, 2, 2, true> : blend_kernel_shared<2, 2, 2, false>);
    }
#undef FGS_BLEND_ARGS
    return check_hip(hipGetLastError(), who);
}

int render_impl(int block_x, int block_y, int num_rendered, int width, int height,
                const float* points_xy, const float* rgb_depth, const float* conic_opacity,
                const uint64_t* keys_sorted, const uint32_t* values_sorted,
                int* ranges, const float bg[3], uint8_t* out_u8, float* out_f32, int flags, void* stream, const char* who)
{
    int sx = 0, sy = 0, mode = 0;
    int rc = check_blend(block_x, block_y, width, height, points_xy, rgb_depth, conic_opacity, ranges, bg, out_u8, out_f32, flags, &sx, &sy, &mode, who);
    if (rc != FGS_OK) return rc;                // before anything is launched
    if (num_rendered > 0 && (!points_xy || !rgb_depth || !conic_opacity || !keys_sorted || !values_sorted))
        return fail(FGS_E_INVALID, "%s: null buffer", who);
    LongTable longer;
    std::unique_lock<std::mutex> enqueue;       // from the launch that lists them to the blend that reads the table
    rc = long_table((hipStream_t)stream, num_rendered, block_x, block_y, width, height, &longer, &enqueue);
    if (rc != FGS_OK) return rc;
    rc = ranges_impl(block_x, block_y, num_rendered, width, height, keys_sorted, ranges, longer, stream, who);
    if (rc != FGS_OK) return rc;
    return blend_impl(false, nullptr, longer, block_x, block_y, width, height, points_xy, rgb_depth, conic_opacity, values_sorted, ranges,
                      bg, out_u8, out_f32, flags, stream, who);
}

// Sort and render of one frame.  The sort knows where every tile's pairs stand: its segment launches write the ranges and list the long lists,
// and a workgroup of the scatter ranks the tiles of a small frame, so the launches that would find all this in the sorted keys are left out (720p / 0.2M
// pairs: two of ten, 9 us of 77).  Where the sort has no such table (one pair, more than 2^18 tile ids) they follow it as in render_impl.
int sort_render_impl(int block_x, int block_y, int num_rendered, int width, int height, char* list_sorting_space, size_t sorting_size,
                     const uint64_t* keys_unsorted, const uint32_t* values_unsorted, uint64_t* keys_sorted, uint32_t* values_sorted,
                     const float* points_xy, const float* rgb_depth, const float* conic_opacity, int* ranges, const float bg[3],
                     uint8_t* out_u8, float* out_f32, int flags, void* stream, const char* who)
{
    int sx = 0, sy = 0, mode = 0;
    int rc = check_blend(block_x, block_y, width, height, points_xy, rgb_depth, conic_opacity, ranges, bg, out_u8, out_f32, flags, &sx, &sy, &mode, who);
    if (rc != FGS_OK) return rc;
    if (num_rendered > 0 && (!points_xy || !rgb_depth || !conic_opacity)) return fail(FGS_E_INVALID, "%s: null buffer", who);
    // (a call that is refused has asked the runtime for nothing)
    rc = check_sort(num_rendered, width, height, block_x, block_y, list_sorting_space, sorting_size, keys_unsorted, values_unsorted,
                    keys_sorted, values_sorted, who);
    if (rc != FGS_OK) return rc;
    const int tiles_x = (width + block_x - 1) / block_x, tiles_y = (height + block_y - 1) / block_y, num_tiles = tiles_x * tiles_y;
    LongTable longer;
    std::unique_lock<std::mutex> enqueue, ranking;      // from the launch that writes a table to the blend that reads it
    rc = long_table((hipStream_t)stream, num_rendered, block_x, block_y, width, height, &longer, &enqueue);
    if (rc != FGS_OK) return rc;
    FrameTables frame = { { (int2*)ranges, longer.list, (uint32_t)num_tiles, longer.least }, { nullptr, num_tiles, sx * sy, 0 } };
    if (num_rendered > 0 && is_ranked(tiles_x, tiles_y)) {
        SharedGrid grid;
        rc = shared_grid(sx, sy, num_tiles, mode == FGS_COLOUR_SUMS_FP32, &grid);
        if (rc != FGS_OK) return rc;
        frame.ranking.simds = 4 * grid.cus;
        if (num_tiles > grid.resident) {
            rc = tile_order_table((hipStream_t)stream, &frame.ranking.order, &ranking);
            if (rc != FGS_OK) return rc;
        }
    }
    rc = sort_impl(num_rendered, width, height, block_x, block_y, list_sorting_space, sorting_size, keys_unsorted, values_unsorted,
                   keys_sorted, values_sorted, &frame, stream, who);
    if (rc != FGS_OK) return rc;
    // The segment launch comes by the tiles in their order, and with half of the places the last ones of a horizon found none: frames of 763 and 793 long
    // lists (8K / 8M, 6620x4058 / 6M) take 1.00 and 0.98 of the time behind a launch of their own with half of the places, 0.988 and 0.93 with all.
    if (frame.notes.longer) longer.per_shard = kLongPerShard;
    if (!frame.notes.ranges) {
        rc = ranges_impl(block_x, block_y, num_rendered, width, height, keys_sorted, ranges, longer, stream, who);
        if (rc != FGS_OK) return rc;
    }
    if (!frame.ranking.order && ranking.owns_lock()) ranking.unlock();          // (the blend ranks by itself)
    return blend_impl(false, frame.ranking.order, longer, block_x, block_y, width, height, points_xy, rgb_depth, conic_opacity, values_sorted, ranges,
                      bg, out_u8, out_f32, flags, stream, who);
}

} // namespace
} // namespace fgs

#define FGS_DEFINE_RENDER(NAME, BX, BY)                                                                      \
    extern "C" int NAME(int num_rendered, int width, int height,                                             \
                        const float* points_xy, const float* rgb_depth, const float* conic_opacity,          \
                        const uint64_t* gaussian_keys_sorted, const uint32_t* gaussian_values_sorted,        \
                        int* ranges, const float bg_color[3], uint8_t* out_color, void* stream)              \
    {                                                                                                        \
        if (!out_color) return fgs::fail(FGS_E_INVALID, #NAME ": null out_color");                           \
        return fgs::render_impl(BX, BY, num_rendered, width, height, points_xy, rgb_depth, conic_opacity,    \
                                gaussian_keys_sorted, gaussian_values_sorted, ranges, bg_color, out_color,   \
                                nullptr, 0, stream, #NAME);                                                  \
    }

FGS_DEFINE_RENDER(fgs_render_16x16, 16, 16)
FGS_DEFINE_RENDER(fgs_render_32x16, 32, 16)
FGS_DEFINE_RENDER(fgs_render_32x32, 32, 32)

extern "C" int fgs_render_f32(int block_x, int block_y, int num_rendered, int width, int height,
                              const float* points_xy, const float* rgb_depth, const float* conic_opacity,
                              const uint64_t* gaussian_keys_sorted, const uint32_t* gaussian_values_sorted,
                              int* ranges, const float bg_color[3], uint8_t* out_color_u8, float* out_color_f32,
                              void* stream)
{
    return fgs::render_impl(block_x, block_y, num_rendered, width, height, points_xy, rgb_depth,
                            conic_opacity, gaussian_keys_sorted, gaussian_values_sorted, ranges, bg_color,
                            out_color_u8, out_color_f32, 0, stream, "fgs_render_f32");
}

extern "C" int fgs_render_ex(int block_x, int block_y, int num_rendered, int width, int height,
                             const float* points_xy, const float* rgb_depth, const float* conic_opacity,
                             const uint64_t* gaussian_keys_sorted, const uint32_t* gaussian_values_sorted,
                             int* ranges, const float bg_color[3], uint8_t* out_color_u8, float* out_color_f32,
                             int flags, void* stream)
{
    return fgs::render_impl(block_x, block_y, num_rendered, width, height, points_xy, rgb_depth,
                            conic_opacity, gaussian_keys_sorted, gaussian_values_sorted, ranges, bg_color,
                            out_color_u8, out_color_f32, flags, stream, "fgs_render_ex");
}

extern "C" int fgs_sort_render(int block_x, int block_y, int num_rendered, int width, int height,
                               char* list_sorting_space, size_t sorting_size,
                               const uint64_t* gaussian_keys_unsorted, const uint32_t* gaussian_values_unsorted,
                               uint64_t* gaussian_keys_sorted, uint32_t* gaussian_values_sorted,
                               const float* points_xy, const float* rgb_depth, const float* conic_opacity,
                               int* ranges, const float bg_color[3], uint8_t* out_color_u8, float* out_color_f32,
                               int flags, void* stream)
{
    return fgs::sort_render_impl(block_x, block_y, num_rendered, width, height, list_sorting_space, sorting_size, gaussian_keys_unsorted,
                                 gaussian_values_unsorted, gaussian_keys_sorted, gaussian_values_sorted, points_xy, rgb_depth, conic_opacity,
                                 ranges, bg_color, out_color_u8, out_color_f32, flags, stream, "fgs_sort_render");
}

extern "C" int fgs_set_colour_sums(int mode)
{
    if (mode != FGS_COLOUR_SUMS_MATRIX_F16 && mode != FGS_COLOUR_SUMS_FP32) {
        fgs::fail(FGS_E_INVALID, "fgs_set_colour_sums: mode %d unknown", mode);
        return -1;
    }
    return fgs::g_colour_sums.exchange(mode);
}

extern "C" const char* fgs_blend_kernel_name(int block_x, int block_y, int width, int height, int flags)
{
    using namespace fgs;
    int sx = 0, sy = 0, mode = 0;
    if (check_tile(block_x, block_y, &sx, &sy, "fgs_blend_kernel_name") != FGS_OK || width <= 0 || height <= 0) return "";
    if (colour_mode(flags, &mode, "fgs_blend_kernel_name") != FGS_OK) return "";
    const bool ranked = is_ranked((width + block_x - 1) / block_x, (height + block_y - 1) / block_y);
    const bool fp32 = mode == FGS_COLOUR_SUMS_FP32;
#define FGS_NAME(name) (fp32 ? name "true>" : name "false>")
    if (ranked) {
        const int tiles = ((width + block_x - 1) / block_x) * ((height + block_y - 1) / block_y);
        int device = 0, cus = 0;
        if (hipGetDevice(&device) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) {
            (void)hipGetLastError();
            cus = 256;          // no device: what an MI355X would launch
        }
        const int teams = teams_of(sx, sy, tiles, cus);
        if (sx == 1 && sy == 1)
            return teams == 8 ? FGS_NAME("tile_order_kernel + blend_kernel_shared<1, 1, 8, ") : FGS_NAME("tile_order_kernel + blend_kernel_shared<1, 1, 4, ");
        if (sx == 2 && sy == 1) return FGS_NAME("tile_order_kernel + blend_kernel_shared<2, 1, 4, ");
        return teams == 4 ? FGS_NAME("tile_order_kernel + blend_kernel_shared<2, 2, 4, ") : FGS_NAME("tile_order_kernel + blend_kernel_shared<2, 2, 2, ");
    }
    if (sx == 1 && sy == 1) return FGS_NAME("blend_kernel<1, 1, ");
    if (sx == 2 && sy == 1) return FGS_NAME("blend_kernel<2, 1, ");
    return FGS_NAME("blend_kernel<2, 2, ");
#undef FGS_NAME
}

extern "C" int fgs_tile_ranges(int block_x, int block_y, int num_rendered, int width, int height,
                               const uint64_t* gaussian_keys_sorted, int* ranges, void* stream)
{
    return fgs::ranges_impl(block_x, block_y, num_rendered, width, height, gaussian_keys_sorted, ranges, fgs::LongTable(), stream,
                            "fgs_tile_ranges");
}

extern "C" int fgs_blend(int block_x, int block_y, int width, int height,
                         const float* points_xy, const float* rgb_depth, const float* conic_opacity,
                         const uint32_t* gaussian_values_sorted, const int* ranges, const float bg_color[3],
                         uint8_t* out_color_u8, float* out_color_f32, void* stream)
{
    return fgs::blend_impl(true, nullptr, fgs::LongTable(), block_x, block_y, width, height, points_xy, rgb_depth, conic_opacity,
                           gaussian_values_sorted, ranges, bg_color, out_color_u8, out_color_f32, 0, stream, "fgs_blend");
}

extern "C" int fgs_blend_ex(int block_x, int block_y, int width, int height,
                            const float* points_xy, const float* rgb_depth, const float* conic_opacity,
                            const uint32_t* gaussian_values_sorted, const int* ranges, const float bg_color[3],
                            uint8_t* out_color_u8, float* out_color_f32, int flags, void* stream)
{
    return fgs::blend_impl(true, nullptr, fgs::LongTable(), block_x, block_y, width, height, points_xy, rgb_depth, conic_opacity,
                           gaussian_values_sorted, ranges, bg_color, out_color_u8, out_color_f32, flags, stream, "fgs_blend_ex");
}

