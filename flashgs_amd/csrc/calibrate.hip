// Microbenchmarks that measure what this GPU attains on the three resources the rasterizer's
// rooflines are priced against: streaming memory traffic, the issue of vector instructions.  Built
// into its own small library (libflashgs_calibrate.so): measurement aid, not part of the
// rasterizer.  Every function runs on `stream`, times its kernel with HIP events and returns the
// result through `out`; return value 0 or a hipError_t code.
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace {

constexpr int kThreads = 256;

__global__ __launch_bounds__(kThreads) void copy_kernel(const float4* __restrict__ src, float4* __restrict__ dst, size_t n)
{
    size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * kThreads;
    for (; i < n; i += stride) dst[i] = src[i];
}

__global__ __launch_bounds__(kThreads) void read_kernel(const float4* __restrict__ src, float* __restrict__ sink, size_t n)
{
    size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * kThreads;
    float acc = 0.f;
    for (; i < n; i += stride) {
        const float4 v = src[i];
        acc += v.x + v.y + v.z + v.w;
    }
    if (acc == 12345.678f) *sink = acc;      // never true for the fill value; keeps the loads alive
}

// Loops of one kind of instruction on eight registers in turn, or of what blend_kernel issues for a list entry.
// %8 and %9 are vector registers, %10 is a scalar one.
#define FGS_FMA(x) "v_fma_f32 " x ", " x ", %8, %9\n\t"
#define FGS_MUL(x) "v_mul_f32 " x ", " x ", %8\n\t"
#define FGS_ADD(x) "v_add_f32 " x ", " x ", %8\n\t"
#define FGS_SUB(x) "v_sub_f32 " x ", " x ", %8\n\t"
#define FGS_FMA_SCALAR(x) "v_fma_f32 " x ", " x ", %10, %9\n\t"
#define FGS_MUL_SCALAR(x) "v_mul_f32 " x ", %10, " x "\n\t"
#define FGS_FMA_REPEATED(x) "v_fma_f32 " x ", -%8, " x ", " x "\n\t"
#define FGS_SHIFT(x) "v_lshlrev_b32 " x ", 1, " x "\n\t"
#define FGS_CMP(x) "v_cmp_gt_f32 vcc, " x ", %8\n\t"
#define FGS_EXP(x) "v_exp_f32 " x ", " x "\n\t"
#define FGS_FMAC(x) "v_fmac_f32 " x ", %8, %9\n\t"
#define FGS_EIGHT(m) m("%0") m("%1") m("%2") m("%3") m("%4") m("%5") m("%6") m("%7")
#define FGS_48(m) FGS_EIGHT(m) FGS_EIGHT(m) FGS_EIGHT(m) FGS_EIGHT(m) FGS_EIGHT(m) FGS_EIGHT(m)
// 25 multiplications, subtractions and multiply-adds, and two comparisons and two shifts for the rest
#define FGS_ENTRY FGS_MUL("%2") FGS_MUL("%3") FGS_MUL("%4") FGS_MUL("%5") FGS_MUL("%6") FGS_MUL("%7") FGS_SUB("%0") FGS_MUL("%1") FGS_SUB("%2") \
    FGS_MUL("%3") FGS_SUB("%4") FGS_MUL("%5") FGS_SUB("%6") FGS_EIGHT(FGS_FMAC) FGS_FMAC("%0") FGS_FMAC("%1") FGS_FMAC("%2") FGS_FMAC("%3") \
    FGS_CMP("%4") FGS_SHIFT("%5") FGS_CMP("%6") FGS_SHIFT("%7")

enum { kFma, kMul, kAdd, kSub, kFmaScalar, kMulScalar, kFmaRepeated, kShift, kCmp, kExp, kEntry, kEntryApart, kModes };
constexpr int kPerIteration[kModes] = {48, 48, 48, 48, 48, 48, 48, 48, 48, 48, 1, 1};         // instructions, or entries

template <int kMode>
__global__ __launch_bounds__(kThreads) void issue_kernel(float* __restrict__ sink, int iters, float s)
{
    float x0 = threadIdx.x, x1 = x0 + 1, x2 = x0 + 2, x3 = x0 + 3, x4 = x0 + 4, x5 = x0 + 5, x6 = x0 + 6, x7 = x0 + 7, a = x0 * s, b = x0 * s + 1.0f;
#define FGS_LOOP(body) \
    for (int i = 0; i < iters; i++) \
        asm volatile(body : "+v"(x0), "+v"(x1), "+v"(x2), "+v"(x3), "+v"(x4), "+v"(x5), "+v"(x6), "+v"(x7) : "v"(a), "v"(b), "s"(s) : "vcc")
    if constexpr (kMode == kFma) FGS_LOOP(FGS_48(FGS_FMA));
    if constexpr (kMode == kMul) FGS_LOOP(FGS_48(FGS_MUL));
    if constexpr (kMode == kAdd) FGS_LOOP(FGS_48(FGS_ADD));
    if constexpr (kMode == kSub) FGS_LOOP(FGS_48(FGS_SUB));
    if constexpr (kMode == kFmaScalar) FGS_LOOP(FGS_48(FGS_FMA_SCALAR));
    if constexpr (kMode == kMulScalar) FGS_LOOP(FGS_48(FGS_MUL_SCALAR));
    if constexpr (kMode == kFmaRepeated) FGS_LOOP(FGS_48(FGS_FMA_REPEATED));
    if constexpr (kMode == kShift) FGS_LOOP(FGS_48(FGS_SHIFT));
    if constexpr (kMode == kCmp) FGS_LOOP(FGS_48(FGS_CMP));
    if constexpr (kMode == kExp) FGS_LOOP(FGS_48(FGS_EXP));
    if constexpr (kMode == kEntry) FGS_LOOP(FGS_EXP("%0") FGS_EXP("%1") FGS_ENTRY);
    if constexpr (kMode == kEntryApart) FGS_LOOP(FGS_EXP("%0") "s_nop 0\n\t" FGS_EXP("%1") "s_nop 0\n\t" FGS_ENTRY);
#undef FGS_LOOP
    const float r = x0 + x1 + x2 + x3 + x4 + x5 + x6 + x7;
    if (r == 12345.678f) *sink = r;             // keeps the registers alive
}

template <typename Launch>
int timed(hipStream_t st, int reps, double* ms, Launch launch)
{
    hipEvent_t e0, e1;
    hipError_t rc = hipEventCreate(&e0);
    if (rc != hipSuccess) return (int)rc;
    rc = hipEventCreate(&e1);
    if (rc != hipSuccess) return (int)rc;
    launch();                                   // warm-up
    (void)hipEventRecord(e0, st);
    for (int r = 0; r < reps; r++) launch();
    (void)hipEventRecord(e1, st);
    rc = hipEventSynchronize(e1);
    float t = 0.f;
    if (rc == hipSuccess) rc = hipEventElapsedTime(&t, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc == hipSuccess) rc = hipGetLastError();
    *ms = (double)t / reps;
    return (int)rc;
}

} // namespace

// Bytes per second moved by a device-to-device copy of `bytes` bytes (read + write counted).
extern "C" int fgs_cal_copy(const void* src, void* dst, size_t bytes, double* bytes_per_s, void* stream)
{
    hipStream_t st = (hipStream_t)stream;
    const size_t n = bytes / sizeof(float4);
    double ms = 0;
    const int rc = timed(st, 10, &ms, [&] {
        hipLaunchKernelGGL(copy_kernel, dim3(256 * 32), dim3(kThreads), 0, st, (const float4*)src, (float4*)dst, n);
    });
    *bytes_per_s = 2.0 * (double)(n * sizeof(float4)) / (ms * 1e-3);
    return rc;
}

// Bytes per second read by a streaming reduction over `bytes` bytes.
extern "C" int fgs_cal_read(const void* src, float* sink, size_t bytes, double* bytes_per_s, void* stream)
{
    hipStream_t st = (hipStream_t)stream;
    const size_t n = bytes / sizeof(float4);
    double ms = 0;
    const int rc = timed(st, 10, &ms, [&] {
        hipLaunchKernelGGL(read_kernel, dim3(256 * 32), dim3(kThreads), 0, st, (const float4*)src, sink, n);
    });
    *bytes_per_s = (double)(n * sizeof(float4)) / (ms * 1e-3);
    return rc;
}

// Wave64 instructions (or, modes 10 and 11, list entries) per second times 64 lanes, summed over the chip, with `waves` resident
// waves per SIMD: 0 to 3 fma, mul, add, sub with all operands in vector registers, 4 and 5 fma and mul with a scalar
// one, 6 fma with a negated and a repeated operand, 7 shift, 8 comparison, 9 exponential, 10 the instructions of a blend's list
// entry, 11 the same with its exponentials apart.
extern "C" int fgs_cal_issue(int mode, int waves, float* sink, double* lane_ops_per_s, void* stream)
{
    if (mode < 0 || mode >= kModes || waves < 1 || waves > 8) return (int)hipErrorInvalidValue;
    hipStream_t st = (hipStream_t)stream;
    int device = 0, cus = 0;
    hipError_t rc = hipGetDevice(&device);
    if (rc == hipSuccess) rc = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
    if (rc != hipSuccess) return (int)rc;
    typedef void (*Kernel)(float*, int, float);
    static const Kernel kernels[kModes] = {issue_kernel<0>, issue_kernel<1>, issue_kernel<2>, issue_kernel<3>, issue_kernel<4>, issue_kernel<5>,
                                           issue_kernel<6>, issue_kernel<7>, issue_kernel<8>, issue_kernel<9>, issue_kernel<10>, issue_kernel<11>};
    const int iters = 4096, blocks = cus * waves;          // a wave on each SIMD of a CU per workgroup
    double ms = 0;
    const int status = timed(st, 3, &ms, [&] { hipLaunchKernelGGL(kernels[mode], dim3(blocks), dim3(kThreads), 0, st, sink, iters, 1e-6f); });
    *lane_ops_per_s = (double)blocks * kThreads * iters * kPerIteration[mode] / (ms * 1e-3);
    return status;
}
