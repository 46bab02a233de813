// hip_forward.hip — gfx950 kernels and the C ABI of spingalett_hip.h.
//
// This translation unit holds every HIP runtime call and the smaller kernels; the large families of template kernels are
// compiled beside it, a part per hip_part.hip (hip_instances.inl lists which), from the .inl files of hip_kernels.h:
//   sp_decode         element decoders (bit-exact with Serialize.c:45-85,195-297)
//   hip_gemv.inl      sp_gemv*: 1..4 samples (FP32 weights: up to 64): vector kernels, FP32-grade arithmetic; integer
//                     weights as exact integer dot products on the INT8 matrix cores (sp_gemv_i8mfma)
//   hip_skinny.inl    sp_skinny16[_kw]: 5..256 samples, or layers with <= 64 outputs: one operand streamed once
//                     through registers into 16-bit MFMAs, the thin one in LDS (_kw: thin side of <= 8 rows, K split
//                     inside the workgroup)
//   hip_gemm16.inl    sp_gemm16_big / sp_gemm16: larger batches: LDS-tiled dequant-to-16-bit MFMA GEMM, fused epilogue
//   hip_gemm32.inl    FP32 weights beyond four samples: FP32 MFMA GEMMs of small layers, unaligned rows, large weights
//   hip_tile32.inl    sp_gemm32_f32: the FP32 MFMA GEMM of the other layers and of training's backward
//   hip_gemm32_parts.inl  sp_gemm32_bf16_parts: large FP32 forward products on BF16 parts
//   sp_softmax_rows   per-sample softmax (Activation.c:5-21)
//   sp_eval_*         loss and argmax of a labelled batch (SIMD.c:522-552, Training.c:421-435)
//   hip_train.inl     the batched training step (included at the end)
//   hip_train_tiny.inl  nets of one compute unit's size: whole trainings in one launch
// Host side (device state per net, kernel selection, the sphip_* entry points) follows the kernels.
// Weights stay in their serialized form on the device; row-major [out][in]
// (Private.h:16), element i of an INT4 array in nibble i&1 of byte i/2, element
// i of an INT2 array at bits 2(i%4) of byte i/4 (Serialize.c:148-152,181-183).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <type_traits>
#include <vector>

#include "hip_kernels.h"
#include "sp_train_tiny.h"
#include "spingalett_hip.h"

using namespace sphip_kernels;

#define SP_KERNEL(...) extern template __global__ void __VA_ARGS__;
namespace sphip_kernels {
#include "hip_instances.inl"
}  // namespace sphip_kernels
#undef SP_KERNEL

namespace {

// ---------------------------------------------------------------------------
// small helpers
// ---------------------------------------------------------------------------
size_t fmt_bytes(int f, uint64_t n)
{
    return (size_t)((n * (uint64_t)fmt_bits(f) + 7u) / 8u);
}

// divisor d of the integer formats: w = (q / d) * max   (Serialize.c:233,258,285)
float fmt_divisor(int f) { return f == I8 ? 127.0f : f == I4 ? 7.0f : 1.0f; }

// folded scale used by the arithmetic kernels: w = q * scale
float fmt_scale(int f, float max_val)
{
    if (f == F32 || f == F16 || f == BF16) return 1.0f;
    if (!(max_val > 0.0f)) return 0.0f;            // Serialize.c:231-236: zeros
    return (float)((double)max_val / (double)fmt_divisor(f));
}

thread_local char g_err[512] = "";

int fail_msg(const char *msg)
{
    snprintf(g_err, sizeof g_err, "%s", msg);
    return 1;
}

int fail_hip(const char *what, hipError_t e)
{
    snprintf(g_err, sizeof g_err, "%s: %s", what, hipGetErrorString(e));
    return 1;
}

#define HCHECK(expr)                                              \
    do {                                                          \
        hipError_t e_ = (expr);                                   \
        if (e_ != hipSuccess) return fail_hip(#expr, e_);         \
    } while (0)

// The two events of a timed region; destroyed on every way out of the function that holds them.
struct TimingEvents {
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int create()
    {
        HCHECK(hipEventCreate(&e0));
        HCHECK(hipEventCreate(&e1));
        return 0;
    }
    ~TimingEvents()
    {
        if (e0) (void)hipEventDestroy(e0);
        if (e1) (void)hipEventDestroy(e1);
    }
};

hipStream_t g_stream = nullptr;
// Routing state of the calling thread.  The launch_* functions below decide which kernel a layer takes and launch it;
// with `dry` set they only decide (nothing is enqueued), which is how sphip_layer_kernel_name answers without side
// effects.  `name` receives the main kernel of the layer routed last.
struct RouteState {
    bool dry = false;
    const char *name = "";
    uint32_t halves = 1;            // 2: split activations (SPHIP_SPLIT_ACTIVATIONS), every layer goes through partial sums
};
thread_local RouteState tl_route;
constexpr uint32_t kGemvStageBytes = 64u * 1024u;   // LDS budget of one stage of the integer GEMV

std::mutex g_init_mutex;

// Workspace of sphip_forward_noalloc: one fixed array per GPU, held until the process ends.  Host code never uses the
// array's name as an address: g_scratch_ptr[device] is what hipGetSymbolAddress returned with that device current.
constexpr size_t kScratchBytes = SPHIP_NOALLOC_SCRATCH_BYTES;
constexpr size_t kScratchRoom = kScratchBytes + (64u << 10);       // a row of padded widths where the widths themselves fit
constexpr int kScratchDevices = 16;
static __device__ __align__(256) unsigned char scratch[kScratchRoom];
unsigned char *g_scratch_ptr[kScratchDevices] = {};

// address of the scratch array on the current device (looked up once per device); caller holds g_init_mutex
int scratch_lookup(unsigned char **out)
{
    int dev = 0;
    HCHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kScratchDevices) return fail_msg("sphip: device index beyond the scratch table");
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        HCHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return fail_msg("sphip: hipGetSymbolAddress returned no address for the scratch array");
        g_scratch_ptr[dev] = static_cast<unsigned char *>(p);
    }
    *out = g_scratch_ptr[dev];
    return 0;
}

// One stream per process (default priority), created at first use; safe to call from several threads.
int ensure_stream()
{
    std::lock_guard<std::mutex> lock(g_init_mutex);
    if (g_stream) return 0;
    int cnt = 0;
    HCHECK(hipGetDeviceCount(&cnt));
    if (cnt <= 0) return fail_msg("no HIP device");
    HCHECK(hipSetDevice(0));
    unsigned char *sp = nullptr;
    if (scratch_lookup(&sp)) return 1;
    HCHECK(hipStreamCreateWithFlags(&g_stream, hipStreamNonBlocking));
    return 0;
}

// ---------------------------------------------------------------------------
// decode kernel — the device form of read_array_compressed
// ---------------------------------------------------------------------------
// lut[q + bias] = fl((float)q / d) computed on the host in IEEE arithmetic, so the
// strict result fl(lut * max) does not depend on the device's division.
struct DecodeParams {
    const uint8_t *codes;
    float *out;
    uint64_t n;
    float max_val;       // scale from the file
    float rel_scale;     // fl(max * fl(1/d))  (mode 1)
    int mode;            // 0 strict, 1 release
    uint32_t cols, pcols;  // elements of a row, and of a row as it lies (padded_width)
    float lut[256];
};

template <int FMT>
__global__ __launch_bounds__(256) void sp_decode(const DecodeParams p)
{
    uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (i >= p.n) return;
    const uint64_t at = p.cols == p.pcols ? i : i / p.cols * p.pcols + i % p.cols;
    float v;
    if constexpr (FMT == F32 || FMT == F16 || FMT == BF16) {
        v = elem_value<FMT>(p.codes, at);
    } else {
        if (!(p.max_val > 0.0f)) {
            v = 0.0f;
        } else {
            int q = int_code<FMT>(p.codes, at);
            if (FMT == I2) v = __fmul_rn((float)q, p.max_val);                    // Serialize.c:285
            else if (p.mode == 1) v = __fmul_rn((float)q, p.rel_scale);
            else v = __fmul_rn(p.lut[q + (FMT == I8 ? 128 : 8)], p.max_val);      // Serialize.c:233,258
        }
    }
    p.out[i] = v;
}

// ---------------------------------------------------------------------------
// softmax over rows (Activation.c:5-21); one wave per row
// ---------------------------------------------------------------------------
// put(i, value i) for the row at p, by the lanes of one wave
template <class Put>
__device__ __forceinline__ void softmax_row(const float *__restrict__ p, uint32_t width, int lane, Put &&put)
{
    constexpr int R = 16;                       // rows up to 1024 wide stay in registers: one batch of loads
    if (width <= (uint32_t)R * kWave) {
        float v[R];
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const uint32_t i = (uint32_t)j * kWave + (uint32_t)lane;
            const float t = p[i < width ? i : 0u];
            v[j] = i < width ? t : -3.402823466e+38f;
        }
        float m = v[0];
#pragma unroll
        for (int j = 1; j < R; ++j) m = fmaxf(m, v[j]);
        m = wave_max(m);
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const uint32_t i = (uint32_t)j * kWave + (uint32_t)lane;
            v[j] = i < width ? expf(v[j] - m) : 0.0f;
            s += v[j];
        }
        s = wave_sum(s);
        const float inv = s > 0.0f ? 1.0f / s : 1.0f;
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const uint32_t i = (uint32_t)j * kWave + (uint32_t)lane;
            if (i < width) put(i, v[j] * inv);
        }
        return;
    }
    float m = -3.402823466e+38f;
    for (uint32_t i = lane; i < width; i += kWave) m = fmaxf(m, p[i]);
    m = wave_max(m);
    float s = 0.0f;
    for (uint32_t i = lane; i < width; i += kWave) s += expf(p[i] - m);
    s = wave_sum(s);
    const float inv = s > 0.0f ? 1.0f / s : 1.0f;
    for (uint32_t i = lane; i < width; i += kWave) put(i, expf(p[i] - m) * inv);
}

// out_kind: 0 FP32, 1 BF16, 2 FP16, 3 split FP16 (hi, and (v - hi) 2^11 rows * width elements further on)
__global__ __launch_bounds__(256) void sp_softmax_rows(const float *__restrict__ in, void *__restrict__ out,
                                                       int out_kind, uint32_t rows, uint32_t width)
{
    const int lane = threadIdx.x & 63;
    const uint32_t row = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (row >= rows) return;
    softmax_row(in + (size_t)row * width, width, lane, [&](uint32_t i, float v) {
        const size_t o = (size_t)row * width + i;
        if (out_kind == 0) reinterpret_cast<float *>(out)[o] = v;
        else if (out_kind == 1) reinterpret_cast<uint16_t *>(out)[o] = f32_to_bf16_rne(v);
        else if (out_kind == 2) reinterpret_cast<uint16_t *>(out)[o] = f32_to_f16_sat(v);
        else {
            const uint16_t hi = f32_to_f16_sat(v);
            _Float16 hh;
            __builtin_memcpy(&hh, &hi, 2);
            reinterpret_cast<uint16_t *>(out)[o] = hi;
            reinterpret_cast<uint16_t *>(out)[(size_t)rows * width + o] = f32_to_f16_sat((v - (float)hh) * 2048.0f);
        }
    });
}

// Softmax of rows of any sums: of the partial sums [part][rows][N] of a layer whose K was split over the grid (those of split
// activations' second matrix, from `splits` on, times 2^-11; biases added here), in one launch with their addition, or of
// logits.  NWV waves to a row, 4 PER values a thread, all in registers.  Written by the reduction and read again by a launch of its
// own, the logits of a split layer cost 4 us, and a wave alone with a row of more than 1024 walks it value by value (whole
// nets, before -> with it, us: 4096 x 1000 INT4 at 16 / 64 samples 15.6 / 18.2 -> 12.1 / 14.5, FP32 at 64 20.2 -> 16.8, 8192 x 4000
// FP16 at 600 116 -> 79.8).  A wave to a row up to 256 outputs, with which four waves have nothing to do (1500 x 100 FP32 at 2000 samples
// 26.4 before, 28.5 with four, 23.5 with one), and of many rows up to 768 (64 x 400 INT2 with split activations at 8192 samples 31.5,
// with four 36.2; x 513 36.7 and 40.1, at 2000 19.1 and 18.3; x 1000 at 4000 35.0 and 31.2).  A thread's place for 64 values where 20
// are needed costs registers and a sixth of the time (64 x 4097 FP16 at 8192 samples 130 before, 253 with 64 of them all gone
// through, 117 without those beyond the row, 106 with 32).  Finished logits take it beyond 1024 outputs: 512 x 3000 FP16 at 1 / 64 /
// 8192 samples 27.8 / 40.5 / 124 -> 8.7 / 12.2 / 97.
struct SoftSums {
    const float *ws;
    uint32_t splits, parts, rows, N;
    LayerArgs L;
    void *out;
    int kind;                // as sp_softmax_rows
    int logits;              // ws holds one set of finished logits
};
constexpr uint32_t kSoftSumsMost = 16384u;

// Whether a layer's partial sums meet in this launch: beyond 1024 outputs, a few rows' workgroups would add the parts of a row one
// after the other (added by a reduction of their own, which spreads them over the chip, and here, us: 8192 x 4097 FP16 at 16 / 64 / 256
// samples 27.7 / 33.4 / 63.1 and 33.3 / 39.0 / 66.7, 8192 x 2000 INT2 with split activations at 16 23.4 and 27.1, 2048 x 6000 at 16 /
// 3000 23.3 / 256 and 30.8 / 234).
bool soft_sums_pay(uint32_t rows, uint32_t N) { return N <= 1024u || (N <= kSoftSumsMost && rows >= 512u); }

template <int PER, bool VEC, int NWV>
__global__ __launch_bounds__(256) void sp_sum_softmax(const SoftSums a)
{
    __shared__ float red[2][4];
    const uint32_t t = NWV == 1 ? threadIdx.x & 63u : threadIdx.x, N = a.N;
    const uint32_t row = NWV == 1 ? blockIdx.x * 4u + (threadIdx.x >> 6) : blockIdx.x;
    if (row >= a.rows) return;                             // (whole waves; NWV == 4: none)
    const uint64_t total = (uint64_t)a.rows * N, first = (uint64_t)row * N;
    float v[PER][4], top = -3.402823466e+38f, sum = 0.0f;
    // value e of group g: outputs 4 (t + T g) + e, or t + T (4 g + e) where rows are not whole float4s; groups beyond the row are
    // left out (uniform)
    constexpr uint32_t T = 64u * NWV;
    auto at = [&](int g, int e) { return VEC ? 4u * (t + T * g) + e : t + T * (4u * g + e); };
    auto live = [&](int g) { return 4u * T * g < N; };
#pragma unroll
    for (int g = 0; g < PER; ++g) {
        if (!live(g)) continue;
        float low[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (VEC) {
            const uint32_t n = at(g, 0);
            float4 s, l;
            add_parts(reinterpret_cast<const float4 *>(a.ws + first + (n < N ? n : 0u)), total / 4u, a.splits, a.parts, s, l);
            v[g][0] = s.x; v[g][1] = s.y; v[g][2] = s.z; v[g][3] = s.w;
            low[0] = l.x; low[1] = l.y; low[2] = l.z; low[3] = l.w;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[g][e] = 0.0f;
            const float *src[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) src[e] = a.ws + first + (at(g, e) < N ? at(g, e) : 0u);
            for (uint32_t p0 = 0; p0 < a.parts; p0 += 4u) {              // (four parts on their way, as add_parts)
                float x[4][4];
#pragma unroll
                for (uint32_t i = 0; i < 4u; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[i][e] = src[e][(p0 + i < a.parts ? p0 + i : p0) * total];
#pragma unroll
                for (uint32_t i = 0; i < 4u; ++i) {
                    if (p0 + i >= a.parts) continue;
#pragma unroll
                    for (int e = 0; e < 4; ++e) (p0 + i < a.splits ? v[g][e] : low[e]) += x[i][e];
                }
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t n = at(g, e);
            if (!a.logits) {
                const float bias = elem_value_rt(a.L.bias_fmt, a.L.bias, n < N ? n : 0u) * a.L.bscale;
                v[g][e] = fmaf(fmaf(low[e], kLoScale, v[g][e]), a.L.wscale, bias);
            }
            v[g][e] = n < N ? v[g][e] : -3.402823466e+38f;
            top = fmaxf(top, v[g][e]);
        }
    }
    top = wave_max(top);
    if constexpr (NWV == 4) {
        if ((t & 63u) == 0) red[0][t >> 6] = top;
        __syncthreads();
        top = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));
    }
#pragma unroll
    for (int g = 0; g < PER; ++g) {
        if (!live(g)) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[g][e] = at(g, e) < N ? expf(v[g][e] - top) : 0.0f;
            sum += v[g][e];
        }
    }
    sum = wave_sum(sum);
    if constexpr (NWV == 4) {
        if ((t & 63u) == 0) red[1][t >> 6] = sum;
        __syncthreads();
        sum = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
    }
    const float inv = sum > 0.0f ? 1.0f / sum : 1.0f;
#pragma unroll
    for (int g = 0; g < PER; ++g) {
        if (!live(g)) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t n = at(g, e);
            if (n >= N) continue;
            const uint64_t o = first + n;
            const float y = v[g][e] * inv;
            if (a.kind == 0) {
                reinterpret_cast<float *>(a.out)[o] = y;
            } else if (a.kind == 1) {
                reinterpret_cast<uint16_t *>(a.out)[o] = f32_to_bf16_rne(y);
            } else if (a.kind == 2) {
                reinterpret_cast<uint16_t *>(a.out)[o] = f32_to_f16_sat(y);
            } else {
                uint16_t hi, lo;
                split_f16(y, hi, lo);
                reinterpret_cast<uint16_t *>(a.out)[o] = hi;
                reinterpret_cast<uint16_t *>(a.out)[total + o] = lo;
            }
        }
    }
}

void launch_sum_softmax(const SoftSums &a)
{
    const bool vec = a.N % 4u == 0 && (reinterpret_cast<uintptr_t>(a.ws) & 15u) == 0;
    auto go = [&](auto per_c, auto nwv_c) {
        constexpr int PER = decltype(per_c)::value, NWV = decltype(nwv_c)::value;
        const uint32_t grid = NWV == 1 ? (a.rows + 3u) / 4u : a.rows;
        if (vec) sp_sum_softmax<PER, true, NWV><<<grid, 256, 0, g_stream>>>(a);
        else sp_sum_softmax<PER, false, NWV><<<grid, 256, 0, g_stream>>>(a);
    };
    using std::integral_constant;
    if (a.N <= 256u) go(integral_constant<int, 1>{}, integral_constant<int, 1>{});
    else if (a.N <= 512u && a.rows >= 2048u) go(integral_constant<int, 2>{}, integral_constant<int, 1>{});
    else if (a.N <= 768u && a.rows >= 4096u) go(integral_constant<int, 3>{}, integral_constant<int, 1>{});
    else if (a.N <= 1024u) go(integral_constant<int, 1>{}, integral_constant<int, 4>{});
    else if (a.N <= 4096u) go(integral_constant<int, 4>{}, integral_constant<int, 4>{});
    else if (a.N <= 8192u) go(integral_constant<int, 8>{}, integral_constant<int, 4>{});
    else go(integral_constant<int, 16>{}, integral_constant<int, 4>{});
}

// rows of finished logits; up to 1024 of them a wave holds in registers (sp_softmax_rows)
void launch_softmax(const float *logits, void *out, int kind, uint32_t rows, uint32_t N)
{
    if (N > 1024u && N <= kSoftSumsMost) launch_sum_softmax({logits, 1, 1, rows, N, LayerArgs{}, out, kind, 1});
    else sp_softmax_rows<<<(rows + 3) / 4, 256, 0, g_stream>>>(logits, out, kind, rows, N);
}

// FP32 -> 16-bit activations for the first GEMM layer
template <bool F16T>
__global__ __launch_bounds__(256) void sp_cvt16(const float *__restrict__ in, uint16_t *__restrict__ out, uint64_t n)
{
    uint64_t i = ((uint64_t)blockIdx.x * 256u + threadIdx.x) * 4u;
    if (i + 4 <= n) {
        float4 v = *reinterpret_cast<const float4 *>(in + i);
        uint2 o;
        o.x = (uint32_t)f32_to_t16<F16T>(v.x) | ((uint32_t)f32_to_t16<F16T>(v.y) << 16);
        o.y = (uint32_t)f32_to_t16<F16T>(v.z) | ((uint32_t)f32_to_t16<F16T>(v.w) << 16);
        *reinterpret_cast<uint2 *>(out + i) = o;
    } else {
        for (; i < n; ++i) out[i] = f32_to_t16<F16T>(in[i]);
    }
}

// FP32 -> the two FP16 matrices of a split activation: hi = the value rounded to FP16, and (value - hi) 2^11, n
// elements further on (the difference is exact in FP32; infinities and NaNs live in hi alone)
__global__ __launch_bounds__(256) void sp_cvt16_split(const float *__restrict__ in, uint16_t *__restrict__ out, uint64_t n)
{
    auto one = [](float v, uint16_t &hi, uint16_t &lo) {
        hi = f32_to_f16_sat(v);
        _Float16 hh;
        __builtin_memcpy(&hh, &hi, 2);
        const float rest = (v - (float)hh) * 2048.0f;
        lo = (rest == rest && fabsf(rest) != __builtin_inff()) ? f32_to_f16_sat(rest) : (uint16_t)0;
    };
    uint64_t i = ((uint64_t)blockIdx.x * 256u + threadIdx.x) * 4u;
    if (i + 4 <= n && (n & 3u) == 0) {                 // (n a multiple of four keeps the second matrix 8-byte aligned)
        const float4 v = *reinterpret_cast<const float4 *>(in + i);
        uint16_t h[4], l[4];
        one(v.x, h[0], l[0]); one(v.y, h[1], l[1]); one(v.z, h[2], l[2]); one(v.w, h[3], l[3]);
        *reinterpret_cast<uint2 *>(out + i) = make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
        *reinterpret_cast<uint2 *>(out + n + i) = make_uint2((uint32_t)l[0] | ((uint32_t)l[1] << 16), (uint32_t)l[2] | ((uint32_t)l[3] << 16));
    } else {
        for (uint64_t e = i; e < n && e < i + 4; ++e) one(in[e], out[e], out[n + e]);
    }
}

// largest bit pattern of |w| among the finite BF16 values of an array
__global__ __launch_bounds__(256) void sp_absmax_bf16(const uint16_t *__restrict__ w, uint64_t n, uint32_t *__restrict__ out)
{
    uint32_t m = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256u) {
        const uint32_t a = w[i] & 0x7FFFu;
        if (a < 0x7F80u && a > m) m = a;
    }
    for (int off = 32; off; off >>= 1) {
        const uint32_t o = (uint32_t)__shfl_xor((int)m, off);
        m = o > m ? o : m;
    }
    if ((threadIdx.x & 63) == 0 && m) atomicMax(out, m);
}

// BF16 -> FP16 of w * 2^shift (the shift puts the array's largest magnitude just below FP16's largest power of two,
// so only values 2^-29 of it and smaller leave the normal range); round to nearest even, exact for every value whose
// scaled magnitude is at least 2^-14, since BF16 has fewer significant bits than FP16
__global__ __launch_bounds__(256) void sp_bf16_to_f16(const uint16_t *__restrict__ w, uint16_t *__restrict__ out, uint64_t n, int shift)
{
    const uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (i < n) out[i] = f32_to_f16_sat(ldexpf(__uint_as_float((uint32_t)w[i] << 16), shift));
}

#include "hip_gemm32.inl"
#include "hip_tile32.inl"
#include "hip_gemm32_parts.inl"

// ---------------------------------------------------------------------------
// FP32 weights on the 16-bit matrix cores (split mode of an FP32 net beyond 64 samples).  With FP16 parts
// w 2^shift = wh + wl and x = xh + xl 2^-11,
//     2^shift sum x w = sum xh wh + sum xl (wh 2^-11) + sum xh wl        (xl wl, 2^-22 of it, is dropped),
// three FP16 products into one FP32 accumulator, i.e. one product over 3 Kp with the parts side by side along k:
// activations [xh | xl | xh], weights [wh | wh 2^-11 | wl]; Kp = K rounded up to 8 elements, padded with zeros.
// The shift brings the array's largest magnitude into [2^14, 2^15), so wl and wh 2^-11 keep their bits except for
// weights 2^-12 of the largest and smaller, whose error is 2^-24 of the largest.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void sp_cat3_x(const float *__restrict__ x, uint16_t *__restrict__ out, uint32_t n, uint32_t K,
                                                 uint32_t Kp, int vec)
{
    const uint32_t groups = Kp / 8u;                      // one thread per 8 consecutive k of a row
    const uint64_t id = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (id >= (uint64_t)n * groups) return;
    const uint32_t r = (uint32_t)(id / groups), k0 = (uint32_t)(id % groups) * 8u;
    const float *src = x + (size_t)r * K + k0;
    float v[8];
    if (vec && k0 + 8u <= K) {
        const float4 a = *reinterpret_cast<const float4 *>(src), b = *reinterpret_cast<const float4 *>(src + 4);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = k0 + e < K ? src[e] : 0.0f;
    }
    uint32_t hi[4], lo[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        uint16_t h0, l0, h1, l1;
        split_f16(v[2 * e], h0, l0);
        split_f16(v[2 * e + 1], h1, l1);
        hi[e] = (uint32_t)h0 | ((uint32_t)h1 << 16);
        lo[e] = (uint32_t)l0 | ((uint32_t)l1 << 16);
    }
    uint16_t *row = out + (size_t)r * 3u * Kp + k0;
    const uint4 H = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    *reinterpret_cast<uint4 *>(row) = H;
    *reinterpret_cast<uint4 *>(row + Kp) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    *reinterpret_cast<uint4 *>(row + 2u * Kp) = H;
}

// largest bit pattern of |w| among the finite values of an FP32 array
__global__ __launch_bounds__(256) void sp_absmax_f32(const float *__restrict__ w, uint64_t n, uint32_t *__restrict__ out)
{
    uint32_t m = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256u) {
        const uint32_t a = __float_as_uint(w[i]) & 0x7FFFFFFFu;
        if (a < 0x7F800000u && a > m) m = a;
    }
    for (int off = 32; off; off >>= 1) {
        const uint32_t o = (uint32_t)__shfl_xor((int)m, off);
        m = o > m ? o : m;
    }
    if ((threadIdx.x & 63) == 0 && m) atomicMax(out, m);
}

// one thread per weight: the three FP16 parts of w 2^shift, into the row's three sections; the padding is zeroed by
// the threads of the row's last elements
__global__ __launch_bounds__(256) void sp_cat3_w(const float *__restrict__ w, uint16_t *__restrict__ out, uint32_t N, uint32_t K,
                                                 uint32_t Kp, int shift)
{
    const uint64_t id = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (id >= (uint64_t)N * Kp) return;
    const uint32_t r = (uint32_t)(id / Kp), k = (uint32_t)(id % Kp);
    uint16_t h = 0, hs = 0, l = 0;
    if (k < K) {
        const float v = ldexpf(w[(size_t)r * K + k], shift);
        h = f32_to_f16_sat(v);
        _Float16 hh;
        __builtin_memcpy(&hh, &h, 2);
        const float rest = v - (float)hh;                     // exact in FP32
        l = (rest == rest && fabsf(rest) != __builtin_inff()) ? f32_to_f16_sat(rest) : (uint16_t)0;
        hs = f32_to_f16_sat((float)hh * (1.0f / 2048.0f));
    }
    uint16_t *row = out + (size_t)r * 3u * Kp + k;
    row[0] = h;
    row[Kp] = hs;
    row[2u * Kp] = l;
}

// ---------------------------------------------------------------------------
// padded layers (padded_width)
// ---------------------------------------------------------------------------
// [rows][cols] elements of BITS bits into [prows][pcols], zeros around; a thread makes one 32-bit word.  Packed elements
// run on across row ends, in the source and (behind a hidden softmax, whose width stays) in the destination.  Once per
// upload.
template <int BITS>
__global__ __launch_bounds__(256) void sp_pad_rows(const uint8_t *__restrict__ in, uint32_t *__restrict__ out, uint32_t rows, uint32_t cols,
                                                   uint32_t pcols, uint64_t words)
{
    constexpr uint32_t EPW = 32 / BITS;
    const uint64_t id = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (id >= words) return;
    const uint64_t e0 = id * EPW;
    uint32_t r = (uint32_t)(e0 / pcols), c = (uint32_t)(e0 % pcols), v = 0;
#pragma unroll
    for (uint32_t e = 0; e < EPW; ++e, ++c) {
        if (c == pcols) { c = 0; ++r; }
        if (r >= rows || c >= cols) continue;
        const uint64_t i = (uint64_t)r * cols + c;
        if constexpr (BITS == 16) v |= (uint32_t)reinterpret_cast<const uint16_t *>(in)[i] << (16u * e);
        else v |= ((uint32_t)in[i * BITS / 8u] >> (i % (8u / BITS) * BITS) & ((1u << BITS) - 1u)) << (BITS * e);
    }
    out[id] = v;
}

// The caller's rows of K floats as rows of Kp (a multiple of 4), zeros behind; KIND 0 FP32, 1 BF16, 2 FP16, 3 split FP16
// (sp_cvt16_split's two matrices).  A thread makes four elements of a row.
template <int KIND>
__global__ __launch_bounds__(256) void sp_pad_input(const float *__restrict__ x, void *__restrict__ out, uint32_t n, uint32_t K, uint32_t Kp)
{
    const uint64_t id = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    const uint32_t quads = Kp / 4u, r = (uint32_t)(id / quads), k = (uint32_t)(id % quads) * 4u;
    if (r >= n) return;
    float v[4];
#pragma unroll
    for (uint32_t e = 0; e < 4u; ++e) v[e] = k + e < K ? x[(size_t)r * K + k + e] : 0.0f;
    const size_t o = (size_t)r * Kp + k;
    if constexpr (KIND == 0) {
        *reinterpret_cast<float4 *>(reinterpret_cast<float *>(out) + o) = make_float4(v[0], v[1], v[2], v[3]);
        return;
    }
    uint16_t h[4], l[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if constexpr (KIND == 3) split_f16(v[e], h[e], l[e]);
        else h[e] = f32_to_t16<KIND == 2>(v[e]);
    }
    uint16_t *p = reinterpret_cast<uint16_t *>(out);
    *reinterpret_cast<uint2 *>(p + o) = make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
    if constexpr (KIND == 3)
        *reinterpret_cast<uint2 *>(p + (size_t)n * Kp + o) = make_uint2((uint32_t)l[0] | ((uint32_t)l[1] << 16), (uint32_t)l[2] | ((uint32_t)l[3] << 16));
}

__global__ __launch_bounds__(256) void sp_fill0(float *p, uint64_t cnt)
{
    const uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (i < cnt) p[i] = 0.0f;
}

// ---------------------------------------------------------------------------
// small copies (host staging of single-sample forwards)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void sp_copy32(const float *__restrict__ src, float *__restrict__ dst, uint64_t n)
{
    const uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

// gathers up to 16 layer slots (16-byte aligned starts) into the dense neurons layout
struct PackArgs {
    const float *src;
    float *dst;
    uint32_t count;
    uint32_t src_off[16], dst_off[16], len[16];
};

__global__ __launch_bounds__(256) void sp_pack_layers(const PackArgs a)
{
    const uint32_t s = blockIdx.y;
    if (s >= a.count) return;
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < a.len[s]; i += gridDim.x * 256u)
        a.dst[a.dst_off[s] + i] = a.src[a.src_off[s] + i];
}

// The end of a single-sample forward in one launch of one workgroup: the softmax of the last layer, if it has one, the
// gathering of up to 16 layer slots into pinned host memory, and the sequence number that the host polls (sp_signal_host).
// Three launches before, each of which begins when the one before has ended: 784-512-1000-10 INT8 30.4 -> 27.2 us a call.  Up
// to 3840 values are one round of loads of one workgroup; with more of them a second round costs what a launch does, and a
// net without a softmax saves one only (INT2 nets of 4440 values 30.7 -> 33.1 us, of 4535 27.6 -> 29.2), so longer nets keep the
// three.
struct GatherArgs {
    PackArgs p;
    uint32_t total;        // values to gather
    const float *logits;   // of the last layer, whose softmax is the last slot; nullptr: no softmax here
    uint32_t *flag;
    uint32_t seq;
};
constexpr uint32_t kGatherMost = 3840u;

__global__ __launch_bounds__(1024) void sp_gather_host(const GatherArgs a)
{
    const uint32_t t = threadIdx.x, last = a.p.count - 1u;
    const uint32_t end = a.logits ? a.p.dst_off[last] : a.total;
    if (t >= 960u) {
        // the last wave
        if (a.logits)
            softmax_row(a.logits, a.p.len[last], (int)(t - 960u), [&](uint32_t i, float v) { a.p.dst[end + i] = v; });
    } else {
        for (uint32_t base = 0; base < end; base += 4u * 960u) {
            float v[4];
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j) {
                const uint32_t i = base + j * 960u + t;
                uint32_t at = 0;
                for (uint32_t s = 0; s < a.p.count; ++s)
                    if (i >= a.p.dst_off[s]) at = a.p.src_off[s] + (i - a.p.dst_off[s]);
                v[j] = i < end ? a.p.src[at] : 0.0f;
            }
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j) {
                const uint32_t i = base + j * 960u + t;
                if (i < end) a.p.dst[i] = v[j];
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // this wave's values are written ...
    __syncthreads();                                        // ... and everybody's
    if (t == 0) __hip_atomic_store(a.flag, a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The last launch of a single-sample forward: a sequence number into pinned host memory, system scope, behind the
// kernel boundary that made the gathered activations visible.  The host polls the word instead of asking the runtime
// to wait for the stream.
__global__ __launch_bounds__(64) void sp_signal_host(uint32_t *flag, uint32_t seq)
{
    if (threadIdx.x == 0) __hip_atomic_store(flag, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------------------------------------------------------------------
// evaluation of a batch of outputs (compute_sample_loss, SIMD.c:522-552;
// batch_compute_loss, Training.c:421-435): one wave per sample
// ---------------------------------------------------------------------------
struct EvalArgs {
    const float *y;        // [n][width] outputs
    const float *target;   // [n][width]
    float *loss;           // [n] per-sample loss
    uint32_t *pred;        // [n] index of the first largest output
    uint32_t *hit;         // [n] 1 when the target's first largest entry has the same index
    uint32_t n, width;
    int loss_func;         // 0 sum of squared differences, 1 cross-entropy
    int sigmoid_out;       // cross-entropy in its binary form (output layer is a sigmoid)
};

__global__ __launch_bounds__(256) void sp_eval_rows(const EvalArgs a)
{
    const int lane = threadIdx.x & 63;
    const uint32_t row = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (row >= a.n) return;
    const float *o = a.y + (size_t)row * a.width, *tg = a.target + (size_t)row * a.width;
    const float eps = 1e-9f;
    float acc = 0.0f;
    float bo = -__builtin_inff(), bt = -__builtin_inff();
    uint32_t io = 0xFFFFFFFFu, it = 0xFFFFFFFFu;
    for (uint32_t k = lane; k < a.width; k += kWave) {
        const float ov = o[k], tv = tg[k];
        if (a.loss_func == 0) {
            const float d = ov - tv;
            acc += d * d;
        } else if (a.sigmoid_out) {
            float c = ov < eps ? eps : ov;
            c = c > 1.0f - eps ? 1.0f - eps : c;
            acc -= tv * logf(c) + (1.0f - tv) * logf(1.0f - c);
        } else {
            const float c = ov < eps ? eps : ov;
            acc -= tv * logf(c);
        }
        if (ov > bo || io == 0xFFFFFFFFu) { bo = ov; io = k; }
        if (tv > bt || it == 0xFFFFFFFFu) { bt = tv; it = k; }
    }
    acc = wave_sum(acc);
    // first largest element: larger value wins, equal values keep the lower index
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        const float vo = __shfl_xor(bo, s, kWave), vt = __shfl_xor(bt, s, kWave);
        const uint32_t jo = __shfl_xor(io, s, kWave), jt = __shfl_xor(it, s, kWave);
        if (jo != 0xFFFFFFFFu && (io == 0xFFFFFFFFu || vo > bo || (vo == bo && jo < io))) { bo = vo; io = jo; }
        if (jt != 0xFFFFFFFFu && (it == 0xFFFFFFFFu || vt > bt || (vt == bt && jt < it))) { bt = vt; it = jt; }
    }
    if (lane == 0) {
        a.loss[row] = acc;
        a.pred[row] = io;
        a.hit[row] = io == it ? 1u : 0u;
    }
}

// one workgroup: total loss (added in FP64) and number of hits
__global__ __launch_bounds__(1024) void sp_eval_total(const float *loss, const uint32_t *hit, uint32_t n, double *out_loss,
                                                      uint32_t *out_hits)
{
    __shared__ double s_l[16];
    __shared__ uint32_t s_h[16];
    double l = 0.0;
    uint32_t h = 0;
    for (uint32_t i = threadIdx.x; i < n; i += 1024u) { l += (double)loss[i]; h += hit[i]; }
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) { l += __shfl_xor(l, s, kWave); h += __shfl_xor(h, s, kWave); }
    if ((threadIdx.x & 63) == 0) { s_l[threadIdx.x >> 6] = l; s_h[threadIdx.x >> 6] = h; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double tl = 0.0;
        uint32_t th = 0;
        for (int w = 0; w < 16; ++w) { tl += s_l[w]; th += s_h[w]; }
        *out_loss = tl;
        *out_hits = th;
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
struct DevArray {
    uint8_t *base = nullptr;       // inside sphip_net::arrays, at a multiple of 256 bytes
    size_t bytes = 0;
    uint64_t count = 0;
    uint64_t laid = 0;             // elements that lie at base: the uploaded ones, and zeros around them (padded_width)
    float max_val = 0.0f;
    bool uploaded = false;
    uint16_t *codes16 = nullptr;   // weights of a layer with few outputs: unscaled codes as FP16 (made on demand)
    bool codes16_valid = false;
    uint16_t *wide16 = nullptr;    // BF16 weight arrays: the weights times 2^wide_shift as FP16 (made at upload)
    bool wide16_valid = false;
    int wide_shift = 0;
    uint16_t *cat3 = nullptr;      // FP32 weight arrays in split mode: [out][3 Kp] FP16 parts of w 2^cat3_shift (made on demand)
    bool cat3_valid = false;
    int cat3_shift = 0;
};

struct sphip_train_state;

// Device memory a forward needs beyond the net's arrays, its input and its output.  A net owns one, grown on demand by
// reserve(); sphip_forward_noalloc lays one out inside the library's fixed scratch array instead.
struct Workspace {
    void *buf[2];                  // ping-pong activation buffers, n x widest layer x 4 bytes each
    uint8_t *aq;                   // digit planes of the current layer input (two-launch form of the integer GEMV) ...
    float *aq_inv;                 // ... their scales ...
    int *aq_dsum;                  // ... and digit sums
    float *soft_tmp;               // FP32 logits of a softmax layer
    float *split_ws;               // partial sums of K splits
    uint64_t split_cap;            // ... and how many floats it holds
    uint16_t *const *codes16;      // [layers-1]: FP16 copy of the codes of an integer layer with few outputs, or nullptr
    uint16_t *cat;                 // split mode of an FP32 net: the three-part FP16 form of the current layer's input
};

struct sphip_net {
    uint32_t layers = 0;
    std::vector<uint32_t> topo;
    std::vector<uint8_t> act;
    int prec = 0;
    std::vector<DevArray> W, B;    // [layers-1] as uploaded, zeros behind them up to the padded outputs
    // Widths whose weight rows would not be whole 16-byte units run padded with zero weights (padded_width); PW are the
    // weights of the layers whose inputs that touches.  They lie on the device instead of W (base == nullptr there), but
    // for the first layer, whose uploaded rows the vector kernels multiply with the caller's.
    std::vector<uint32_t> ptopo;
    std::vector<DevArray> PW;
    uint8_t *arrays = nullptr;     // the one allocation behind every base
    uint8_t *pad_stage = nullptr;  // ... and behind them the room through which uploaded rows reach PW
    size_t pad_stage_bytes = 0;

    DevArray &w(uint32_t l) { return PW[l].base ? PW[l] : W[l]; }                    // what a forward multiplies with
    const DevArray &w(uint32_t l) const { return PW[l].base ? PW[l] : W[l]; }
    // workspace, grown on demand
    uint64_t cap_elems = 0;        // capacity of each ping-pong buffer in FP32 elements
    void *buf[2] = {nullptr, nullptr};
    uint8_t *aq = nullptr;         // digit planes of the current layer input (integer GEMV)
    float *aq_inv = nullptr;
    int *aq_dsum = nullptr;
    uint32_t aq_valid_layer = 0, aq_valid_n = 0;   // which layer input the planes describe (layer-only timing)
    uint32_t aq_cap_n = 0;
    float *soft_tmp = nullptr;     // FP32 logits of a softmax layer
    uint64_t soft_cap = 0;
    float *layers_buf = nullptr;   // all activations of a single-sample forward, each layer at a 16-byte aligned slot
    std::vector<uint32_t> slot_off;  // start of each layer's slot (floats)
    uint64_t slots_total = 0;
    float *pin_in = nullptr, *pin_out = nullptr;   // pinned host staging of small inputs / outputs
    uint32_t *pin_flag = nullptr;  // pinned word the last launch of a single-sample forward writes its sequence number to
    uint32_t flag_seq = 0;
    uint64_t pin_in_cap = 0, pin_out_cap = 0;
    float *stage_x = nullptr;      // device staging of host inputs / outputs
    float *stage_y = nullptr;
    uint64_t stage_x_cap = 0, stage_y_cap = 0;
    uint32_t max_width = 0;
    uint64_t total_neurons = 0;
    float *split_ws = nullptr;     // partial sums of the K splits of the thin-operand kernel
    uint64_t split_cap = 0;
    float *eval_buf = nullptr;     // evaluation: outputs, staged targets, per-sample loss / prediction / hit, totals
    uint64_t eval_cap = 0;
    sphip_train_state *train = nullptr;   // gradients, optimizer moments, kept activations (training only)
    std::vector<uint16_t *> codes16_ptrs; // [layers-1] what Workspace::codes16 points at for the net's own workspace
    uint16_t *cat_buf = nullptr;   // split mode of an FP32 net: three-part FP16 layer input
    uint64_t cat_cap = 0;          // ... in elements

    Workspace workspace() const
    {
        return Workspace{{buf[0], buf[1]}, aq, aq_inv, aq_dsum, soft_tmp, split_ws, split_cap, codes16_ptrs.data(), cat_buf};
    }
};

namespace {

void train_free(sphip_net *net);

// R_CAT3: FP32 weights, the larger layers as three FP16 products (cat3_layer, sp_cat3_x, sp_cat3_w), FP32 activations
// between the layers
enum Regime { R_GEMV, R_GEMM16, R_GEMM32, R_CAT3 };

// FP32 weights: the vector kernel up to four samples, like every other format; beyond that the FP32 matrix-core kernel
// with its K splits is the faster one, although the vector kernel takes eight samples per pass over the weights
// (784-512-1000-10 at 5 / 8 / 64 samples: 27 / 34 / 245 us against 27 / 30 / 31 us; three 4096-wide layers 97 / 124 / 960
// against 84 / 84 / 83 us; at four samples 16 against 29 and 42 against 85 us).
constexpr uint32_t kF32VectorMax = 4;

Regime pick_regime(const sphip_net *net, uint32_t n, uint32_t flags)
{
    if ((flags & SPHIP_FORCE_GEMV) && n <= 64) return R_GEMV;
    if (net->prec == F32 && (flags & SPHIP_SPLIT_ACTIVATIONS) && n > kF32VectorMax) return R_CAT3;
    if (flags & SPHIP_FORCE_GEMM) return net->prec == F32 ? R_GEMM32 : R_GEMM16;
    if (net->prec == F32) return n <= kF32VectorMax ? R_GEMV : R_GEMM32;
    return n <= 4 ? R_GEMV : R_GEMM16;
}

// Width a layer runs with.  Rows of weights that are not whole 16-byte units can only be read element by element or word
// by word, and every tile of such a layer waits for those loads (1030-1531-777-33 FP16 at 1333 samples: 107 us for each
// of three layers, 9 to 15 padded).  So an input or hidden layer of such a width gets neurons without weights up to
// the next whole unit (wide ones up to a multiple of 64, whole cache lines): zero rows and zero biases on the producing
// side, zero columns on the consuming side.  The kernels store something finite for a padded neuron whatever its inputs
// are (layer_sum), so that it adds nothing behind infinities and NaNs either.  Not the output layer, whose rows are the
// caller's, and not a hidden softmax, whose sum runs over its real neurons.
// Integer rows of eight codes' multiples (1000 INT8 codes) have kernels of their own, which are as good on small layers
// and take the input as it is; hidden widths of that kind are padded in front of half a million weights and more, where
// the streaming and DMA kernels, which want 16-byte rows, are the better ones, and so are inputs wider than what the small kernel
// takes (one layer, as they are -> padded, us: 4104 x 3000 INT8 at 16 / 300 samples 35 / 44.5 -> 13.1 / 37.5, 9040 x 2576 INT2 at 16 61
// -> 13.9; rows that are no whole words ran code by code: 11864 x 5968 INT2 at 16 / 1590 166 / 3029 -> 18 / 286).  FP32 rows stay as
// they are.
uint32_t padded_width(int fmt, uint32_t w, uint32_t next, bool hidden)
{
    if (fmt == F32) return w;
    const uint32_t unit = fmt_bits(fmt) == 16 ? 8u : 128u / (uint32_t)fmt_bits(fmt);
    if (w % unit == 0) return w;
    if (w % 8u == 0 && !((hidden || w > 2048u) && (uint64_t)w * next > (512u << 10))) return w;
    const uint32_t to = w >= 256u ? 64u : unit;
    return (w + to - 1u) / to * to;
}

// raw: its inputs unpadded (the first layer on the vector kernels, which take the caller's rows as they are); its outputs
// are padded all the same
LayerArgs make_layer_args(const sphip_net *net, uint32_t l /*1-based layer*/, bool raw = false)
{
    LayerArgs L{};
    const DevArray &w = raw ? net->W[l - 1] : net->w(l - 1), &b = net->B[l - 1];
    L.w = w.base;
    L.bias = b.base;
    L.wscale = fmt_scale(net->prec, net->W[l - 1].max_val);
    L.bscale = fmt_scale(net->prec, net->B[l - 1].max_val);
    L.bias_fmt = net->prec;
    L.act = net->act[l - 1] == A_SOFTMAX ? A_NONE : net->act[l - 1];
    L.N = net->ptopo[l];
    L.pad = (uint16_t)(net->ptopo[l] - net->topo[l]);                          // (at most 63)
    L.K = raw ? net->topo[l - 1] : net->ptopo[l - 1];
    return L;
}

bool rows_aligned(int fmt, uint32_t K) { return ((uint64_t)K * (uint64_t)fmt_bits(fmt)) % 128u == 0; }

// Whether the vector kernels read a first layer's weights as they were uploaded, next to the caller's rows.  Not where those
// rows are no whole words, which leaves only the kernel that reads code by code, a wave to a row (1.5 us per 1000 codes, FP16 4.5),
// and are long enough to pay for the launch that pads the input (one sample, as they are -> padded, us: 1531 x 777 FP16 8.9 -> 6.8,
// BF16 5.2 -> 6.5, 4099 x 600 FP16 19.7 -> 8.0, BF16 9.5 -> 8.0, INT8 9.1 -> 9.0, INT4 9.2 -> 7.2, INT2 8.8 -> 7.2, 9002 x 100 INT8 17.2
// -> 13.6, 7297 x 8070 FP16 80 -> 21, INT4 42 -> 16; 3001 x 600 INT8 7.2 -> 7.9; at four samples 4099 x 600 BF16 10.9 -> 11.4, 4097 x
// 9000 46.9 -> 23.5).  Padded rows stay in FP32 arithmetic, a word of codes a lane, whose decoding costs at three and four samples what the
// wider loads bring in INT2 (12287 x 2048 25.3 -> 28.2; thin layers, a workgroup to a row, 24.4 -> 10.8) and in shorter rows of
// INT8 (5003 x 1100 12.0 -> 13.0, 7297 x 1100 16.3 -> 16.6, 9002 x 1100 19.3 -> 19.2, 4099 x 8070 24.6 -> 22.6).
bool raw_rows(int fmt, uint32_t K, uint32_t N, uint32_t n)
{
    if (fmt == F32 || rows_aligned(fmt, K)) return true;
    const uint64_t row_bits = (uint64_t)K * (uint64_t)fmt_bits(fmt);
    if (fmt_bits(fmt) == 16) {
        if (K < (fmt == F16 ? 1280u : n > 2u && N < 2048u ? 5000u : 4096u)) return true;
        return row_bits % 32u == 0 && N <= 64u && row_bits / 32u >= 256u;
    }
    if (K < 4096u || row_bits % 32u == 0) return true;
    return n > 2u && N > 64u && (fmt == I2 || (fmt == I8 && N < 4096u && K < 7168u));
}

template <int FMT>
void launch_gemv_fmt(const LayerArgs &L, const float *x, float *y, uint32_t n, bool padded = false)
{
    const bool aligned = rows_aligned(FMT, L.K) && (L.K % 4u == 0);
    // integer rows of whole words: a word per lane when 16-byte chunks would leave most of a wave idle (rows of at
    // most 16 chunks) or do not apply (rows that are not whole 16-byte units)
    bool words = false;
    uint32_t lpr = 64;
    if constexpr (FMT == I8 || FMT == I4 || FMT == I2) {
        const uint64_t row_bits = (uint64_t)L.K * fmt_bits(FMT);
        // ... and for rows that are whole units by padding only (12000 -> 5200 -> 467 INT4 at four samples: 45 us, the chunks
        // 52), and for layers of at most 64 outputs, whose rows the 16-byte kernel would give to 32 waves or fewer:
        // there a row of 256 words and more spans a whole workgroup (8192 -> 10 INT4 at four samples: 20 -> 11 us)
        words = row_bits % 32u == 0 && (!aligned || padded || row_bits <= 16u * 128u || L.N <= 64u) && (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
        const uint32_t wpr = (uint32_t)(row_bits / 32u);
        while (lpr > 1u && lpr / 2u >= wpr) lpr /= 2u;
        if (L.N <= 64u && wpr >= 256u) lpr = 256u;
    } else {
        // FP32 and 16-bit weights: only the thin layers with long rows (a workgroup per row instead of a wave per two)
        const uint64_t row_bits = (uint64_t)L.K * fmt_bits(FMT);
        if (L.N <= 64u && row_bits % 32u == 0 && row_bits / 32u >= 256u) { words = true; lpr = 256u; }
    }
    tl_route.name = words ? "sp_gemv_words" : aligned ? "sp_gemv" : "sp_gemv_generic";
    if (tl_route.dry) return;
    for (uint32_t b0 = 0; b0 < n; b0 += 8) {
        const int nb = (int)(n - b0 < 8 ? n - b0 : 8);
        const float *xb = x + (size_t)b0 * L.K;
        float *yb = y + (size_t)b0 * L.N;
        {
            if (words) {
                const uint32_t rows_per_wg = 256u / lpr, grid = (L.N + rows_per_wg - 1) / rows_per_wg;
                if (nb == 1) sp_gemv_words<FMT, 1><<<grid, 256, 0, g_stream>>>(L, xb, yb, nb, lpr);
                else if (nb == 2) sp_gemv_words<FMT, 2><<<grid, 256, 0, g_stream>>>(L, xb, yb, nb, lpr);
                else if (nb <= 4) sp_gemv_words<FMT, 4><<<grid, 256, 0, g_stream>>>(L, xb, yb, nb, lpr);
                else sp_gemv_words<FMT, 8><<<grid, 256, 0, g_stream>>>(L, xb, yb, nb, lpr);
                continue;
            }
        }
        if (aligned) {
            constexpr int R = 2;
            const uint32_t waves = (L.N + R - 1) / R, grid = (waves + 3) / 4;
            if (nb == 1) sp_gemv<FMT, 1, R><<<grid, 256, 0, g_stream>>>(L, xb, yb, nb);
            else if (nb == 2) sp_gemv<FMT, 2, R><<<grid, 256, 0, g_stream>>>(L, xb, yb, nb);
            else if (nb <= 4) sp_gemv<FMT, 4, R><<<grid, 256, 0, g_stream>>>(L, xb, yb, nb);
            else sp_gemv<FMT, 8, R><<<grid, 256, 0, g_stream>>>(L, xb, yb, nb);
        } else {
            const uint32_t grid = (L.N + 3) / 4;
            if (nb == 1) sp_gemv_generic<FMT, 1><<<grid, 256, 0, g_stream>>>(L, xb, yb, nb);
            else if (nb <= 4) sp_gemv_generic<FMT, 4><<<grid, 256, 0, g_stream>>>(L, xb, yb, nb);
            else sp_gemv_generic<FMT, 8><<<grid, 256, 0, g_stream>>>(L, xb, yb, nb);
        }
    }
}

template <int FMT, int MT, int FQ = 0>
void launch_gemv_i8_mt(const GemvI8Args &a, uint32_t grid_x, uint32_t threads, size_t lds)
{
    if (tl_route.dry) return;
    auto kern = sp_gemv_i8mfma<FMT, MT, FQ>;
    static bool once = ((void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 156 * 1024), true);
    (void)once;
    kern<<<grid_x, threads, lds, g_stream>>>(a);
}

// Integer formats with 16-byte aligned rows go to the INT8 matrix cores:
// one quantise launch for the layer's input, then the GEMV proper.
template <int FMT>
bool launch_gemv_i8(const Workspace &wk, const LayerArgs &L, const float *x, float *y, uint32_t n, bool main_only)
{
    constexpr int KL = I8Fmt<FMT>::KL;
    // (reserve() gives every integer net its digit-plane buffers for up to 64 samples before anything is launched)
    if (!rows_aligned(FMT, L.K) || L.K < (uint32_t)KL || (!wk.aq && !tl_route.dry)) return false;
    // Small layers: this kernel's fixed phases (quantising the activations, the barrier, the K-share reduction) cost
    // more than they save, and the vector kernel, whose time goes with codes x samples, is faster: 512 x 784 INT8
    // 2.7 against 5.4 us at one sample and 4.4 against 7.3 us at four, 2048 x 2048 4.5 against 6.4 us at one; equal
    // from about 4 M code-sample products (INT2, whose decode costs more vector instructions: half that).
    if ((uint64_t)L.N * L.K * n <= (FMT == I2 ? (2ull << 20) : (4ull << 20))) return false;
    // layers of at most 64 outputs are four row groups at most: the vector kernel with a workgroup per row is quicker
    // (16384 -> 64 INT4 at four samples: 38 us here)
    if (L.N <= 64u && n <= 4u) return false;
    if (reinterpret_cast<uintptr_t>(x) & 15u) return false;   // the quantiser reads float4
    const int need = (int)(n + 3) / 4;
    const int MT = need <= 1 ? 1 : need <= 2 ? 2 : need <= 3 ? 3 : need <= 4 ? 4 : need <= 6 ? 6 : need <= 8 ? 8 : need <= 12 ? 12 : 16;
    GemvI8Args a{};
    a.L = L; a.x = x; a.y = y; a.nb = (int)n;
    a.aq = wk.aq; a.inv = wk.aq_inv; a.dsum = wk.aq_dsum;
    // waves of a workgroup: rw row groups (sharing the digit planes) x ks K shares
    const uint32_t wave_rows = (L.N + 15) / 16;
    const uint32_t kblocks = (L.K + KL - 1) / KL;
    const uint32_t blk_bytes = (uint32_t)I8Fmt<FMT>::NMF * 4u * n * 48u;
    const uint32_t budget = kGemvStageBytes;
    const uint32_t max_waves = MT > 4 ? 4u : 16u;             // register budget of the wide tiles
    // up to four samples: the GEMV workgroups quantise the activations themselves
    const bool fused = MT == 1;
    // self-quantising form: K shares of whole 128-byte lines in fetch groups of two blocks up to 64 MiB of weights,
    // of single blocks in groups of four beyond (gemv_i8_specialised has the measurements)
    const bool line_shares = fused && (uint64_t)L.N * L.K * I8Fmt<FMT>::bits / 8u <= (64ull << 20);
    const uint32_t G = line_shares ? 2u : 4u;                  // blocks per fetch group
    const uint32_t ks_cap = 2048u / (G * KL);                  // a scale chunk is a whole number of fetch groups
                                                               // and at most 2048 codes (one wave's batch of loads)
    uint32_t rw, ks;
    if (fused) {
        // about eight waves per compute unit in all; eight-wave workgroups unless that leaves fewer
        // workgroups than compute units
        ks = 2048u / wave_rows;
        ks = ks >= 8u ? 8u : ks >= 4u ? 4u : ks >= 2u ? 2u : 1u;
        if (ks > ks_cap) ks = ks_cap;
        rw = 8u / ks;
        while (rw > 1 && wave_rows / rw < 256u) rw >>= 1;
    } else {
        // the planes cost 3 n bytes per column and workgroup, the weights 2 bits-per-code bytes per
        // column and row group: more row groups per workgroup as n grows or the codes shrink
        rw = (3u * n + (uint32_t)I8Fmt<FMT>::bits - 1) / (uint32_t)I8Fmt<FMT>::bits;
        rw = rw >= 4 ? 4u : rw >= 2 ? 2u : 1u;
        while (rw > 1 && wave_rows / rw < 512u) rw >>= 1;      // keep the grid at least twice the chip
        ks = max_waves / rw > 8u ? 8u : max_waves / rw;
        if (ks > ks_cap) ks = ks_cap;
    }
    // one fetch group (G blocks of every K share) must fit the row, the stage budget and one scale chunk
    while (ks > 1 && (kblocks < G * ks || G * ks * blk_bytes > budget)) ks >>= 1;
    const uint32_t group_blocks = G * ks;
    // scale chunk: about 2048 codes, a whole number of fetch groups, and small enough for one LDS stage
    uint32_t kc_blocks = 2048u / KL;
    if (kc_blocks > budget / blk_bytes) kc_blocks = budget / blk_bytes;
    kc_blocks = kc_blocks / group_blocks * group_blocks;
    if (kc_blocks == 0) kc_blocks = group_blocks;
    a.kc = kc_blocks * KL;
    a.nchunks = (kblocks + kc_blocks - 1) / kc_blocks;
    a.meta_bytes = a.nchunks * n * 16u;
    if ((uint64_t)kc_blocks * blk_bytes + a.meta_bytes > 156u * 1024u) return false;
    const uint32_t nblocks = a.nchunks * kc_blocks;
    a.rw = rw;
    a.ks = ks;
    const uint32_t waves = rw * ks;
    const uint32_t grid = (wave_rows + rw - 1) / rw;
    const size_t red_bytes = (size_t)waves * MT * 64u * sizeof(float);
    tl_route.name = "sp_gemv_i8mfma";
    if (fused) {
        // digit planes in LDS: all of K in one buffer if that takes at most 120 KB, else two buffers of whole scale
        // chunks (at most 60 KB each) that the quant waves fill in turn
        uint32_t stage = nblocks;
        size_t lds = (size_t)nblocks * blk_bytes;
        if (lds > 120u * 1024u) {
            stage = (60u * 1024u / blk_bytes) / kc_blocks * kc_blocks;
            if (stage == 0) stage = kc_blocks;
            lds = 2u * (size_t)stage * blk_bytes;
        }
        a.stage_blocks = stage;
        if (lds < red_bytes) lds = red_bytes;
        lds += a.meta_bytes;
        // a K so long that two buffers and the scale records no longer fit: the vector kernel takes the layer
        if (lds > 156u * 1024u) return false;
        // one quant wave per (scale chunk, sample) of the first stage, at most eight.  (Cutting a chunk into slices so
        // that eight waves quantise a K of fewer chunks, the slices' maxima meeting in LDS, was measured: 0.7-0.9 us
        // slower per layer on 8192-wide INT2 / INT8 layers.)
        const uint32_t units = (stage / kc_blocks < a.nchunks ? stage / kc_blocks : a.nchunks) * n;
        a.qw = units < 8u ? units : 8u;
        if (line_shares) launch_gemv_i8_mt<FMT, 1, 1>(a, grid, (waves + a.qw) * 64, lds);
        else launch_gemv_i8_mt<FMT, 1, 2>(a, grid, (waves + a.qw) * 64, lds);
        return true;
    }
    // LDS stage: everything if it fits the budget, else whole scale chunks
    uint32_t stage = nblocks;
    if ((uint64_t)nblocks * blk_bytes > budget) {
        stage = (budget / blk_bytes) / kc_blocks * kc_blocks;
        if (stage == 0) stage = kc_blocks;
    }
    a.stage_blocks = stage;
    size_t lds = (size_t)stage * blk_bytes;
    if (lds < red_bytes) lds = red_bytes;
    lds += a.meta_bytes;
    if (!main_only && !tl_route.dry) sp_quant_x<FMT><<<(a.nchunks * n + 3u) / 4u, 256, 0, g_stream>>>(a);
    switch (MT) {
    case 1:  launch_gemv_i8_mt<FMT, 1>(a, grid, waves * 64, lds); break;
    case 2:  launch_gemv_i8_mt<FMT, 2>(a, grid, waves * 64, lds); break;
    case 3:  launch_gemv_i8_mt<FMT, 3>(a, grid, waves * 64, lds); break;
    case 4:  launch_gemv_i8_mt<FMT, 4>(a, grid, waves * 64, lds); break;
    case 6:  launch_gemv_i8_mt<FMT, 6>(a, grid, waves * 64, lds); break;
    case 8:  launch_gemv_i8_mt<FMT, 8>(a, grid, waves * 64, lds); break;
    case 12: launch_gemv_i8_mt<FMT, 12>(a, grid, waves * 64, lds); break;
    default: launch_gemv_i8_mt<FMT, 16>(a, grid, waves * 64, lds); break;
    }
    return true;
}

// padded: rows that are whole units by padding only.  They take the FP32 kernels, as they would unpadded: the integer
// matrix cores see an activation with 22 bits of its chunk's largest, FP32 has 24 of its own.
void launch_gemv(int prec, const Workspace &wk, const LayerArgs &L, const float *x, float *y, uint32_t n, bool main_only,
                 bool padded = false)
{
    switch (prec) {
    case F32:  launch_gemv_fmt<F32>(L, x, y, n); break;
    case F16:  launch_gemv_fmt<F16>(L, x, y, n); break;
    case BF16: launch_gemv_fmt<BF16>(L, x, y, n); break;
    case I8:   if (padded || !launch_gemv_i8<I8>(wk, L, x, y, n, main_only)) launch_gemv_fmt<I8>(L, x, y, n, padded); break;
    case I4:   if (padded || !launch_gemv_i8<I4>(wk, L, x, y, n, main_only)) launch_gemv_fmt<I4>(L, x, y, n, padded); break;
    default:   if (padded || !launch_gemv_i8<I2>(wk, L, x, y, n, main_only)) launch_gemv_fmt<I2>(L, x, y, n, padded); break;
    }
}

// Rows of a tile of the big GEMM.  128 x 256 tiles instead of partly filled or too few 256 x 256 ones: up to 128
// samples always (a single row of tiles), and for 16-bit weights, which reach LDS by DMA, whenever 256-row tiles
// would be fewer than 192 (8192 x 8192 BF16 at 256 / 512 / 1024 samples 48.5 / 85.0 / 132 against 58.0 / 85.9 / 144 us, 4096 x
// 4096 at 1024 samples 53.7 against 59.3: twice the tiles, half the K splits or none; but sums of 8192 into 2048 outputs at 768
// samples 58.7 against 53.5).  Integer weights are unpacked once per tile: half the rows per unpacked tile cost more than the
// tiles bring (8192 x 8192 INT2 at 512 samples 91.4 against 86.1 us, INT8 at 1024 samples 155 against 149).  With enough
// 256 x 256 tiles the smaller tile is no faster (8192-wide layers from 1536 samples).
uint32_t gemm16_tile_rows(int fmt, uint32_t M, uint32_t N)
{
    if (M <= 128u) return 128u;
    if (fmt_bits(fmt) != 16) return 256u;
    // ... and 128-row tiles are at most one per compute unit (more of them run in two rounds; where the line lay for the kernel
    // of eight waves, 8192 x 8192 at 1100 samples 242 against 225 us, and for this one not measured but there, 202 against 221)
    const uint32_t cols = (N + 255u) / 256u;
    return ((M + 255u) / 256u) * cols < 192u && ((M + 127u) / 128u) * cols <= 256u ? 128u : 256u;
}

// K splits of the tile GEMM when its tiles would leave compute units idle: from K = 4096 on (16-bit weights, which reach
// LDS by DMA: 3072), at least eight K tiles each.  Below, the single-stage kernel's small tiles fill the chip in one launch and
// no partial sums travel (forward of one layer, conversion of the input included, K split here against single stage: 1024 x 2048
// x 2048 FP16 31.0 against 25.5 us, at K = 3072 128 x 4096 21.7 against 26.5 and 1024 x 2048 even, 512 x 2048 x 4096 30.5 against
// 36.2, 256 x 8192 x 8192 49 against 84; INT8 1024 x 2048 x 3072 42.5 against 36.9, x 4096 47.8 against 45.9, INT4 600 x 4096 x
// 3584 59 against 50)
uint32_t gemm16_splits(int fmt, uint32_t M, uint32_t N, uint32_t K, uint32_t *kper)
{
    const uint32_t bm = gemm16_tile_rows(fmt, M, N);
    const uint32_t tiles = ((M + bm - 1) / bm) * ((N + 255u) / 256u), ktiles = (K + 63u) / 64u;
    *kper = 0;
    if (tiles >= 192u || ktiles < (fmt_bits(fmt) == 16 ? 48u : 64u)) return 1;
    uint32_t splits = (256u + tiles - 1) / tiles;
    if (splits > 8u) splits = 8u;
    if (splits > ktiles / 8u) splits = ktiles / 8u;
    if (splits <= 1u) return 1;
    const uint32_t per = (ktiles + splits - 1) / splits;
    *kper = per * 64u;
    return (ktiles + per - 1) / per;
}

// Longest K at which the single-stage kernel is the better one instead of 256 x 256 tiles.  A large tile has a compute unit to
// itself, one wave per SIMD, so that the matrix cores idle during its epilogue and the last round is mostly empty; several of
// the single-stage kernel's smaller workgroups share a compute unit and one's epilogue runs beside another's products.  The
// sigmoids or tanhs of a large tile take 17 us.  Large tiles / single-stage, input conversion and a head of 16 included, tanh (a
// sigmoid within 4 % of it), us:
//                      of the rounds   FP16                                          INT8
//   8192 x 8192        all     512 204 / 187   768 229 / 225  1024 253 / 267    1024 258 / 255  1536 310 / 334
//   15144 x 6416       0.83   1536 623 / 536  2048 720 / 655  3072 926 / 926    2048 761 / 630  3072 993 / 872
//   8192 x 4736        0.77   1024 179 / 166  1536 214 / 217  2048 248 / 269    1536 223 / 212  2048 260 / 264
//   4567 x 8192        0.74   1024 187 / 164  1536 220 / 209  2048 246 / 257    2048 266 / 247  3072 339 / 334
//   4567 x 4736        0.65   1024 124 / 110  1536 146 / 144  2048 168 / 169    2048 178 / 164
//   4605 x 4128        0.57    512 102 /  72  1024 121 /  97                    1024 128 /  97
//   4096 x 4096        one     256  59 /  54   512  65 /  65   768  72 /  78     512  66 /  65   768  72 /  76
// (Below six tenths it pays for longer than the lines there, which tests of both kernels' epilogues stand on.)
// Without a transcendental function a quarter of the rounds has to be idle, and the codes packed: leaky ReLU INT8 4567 x 4736 x
// 256 56 / 50, x 512 69 / 65, x 1024 94 / 96; 4567 x 8192 x 448 94 / 90, x 768 116 / 119; FP16 62 / 63 and 89 / 96 at 448.
uint32_t gemm16_shared_limit(int fmt, int act, uint32_t big_tiles, uint64_t outputs)
{
    const bool wide = fmt_bits(fmt) == 16;
    const uint32_t slots = (big_tiles + 255u) / 256u * 256u;
    if (act == A_TANH || act == A_SIGMOID) {
        const uint64_t tenth = (uint64_t)slots * 65536u / 10u;
        if (big_tiles <= 256u) return 512u;
        if (outputs > 9u * tenth) return wide ? 768u : 1024u;
        if (outputs < 6u * tenth) return wide ? 512u : 1024u;
        return wide ? 1536u : 2048u;
    }
    return wide || big_tiles <= 256u || 10u * slots < 13u * big_tiles ? 0u : 512u;
}

// K splits of the single-stage kernel for rows that are not whole 16-byte units (always 64 x 64 tiles, element-wise
// loads): few samples give it a handful of workgroups, each walking all of K with nothing in flight (1030 x 777 at
// 64 samples: 17 workgroups, 80 us).  Whole K tiles per split, about two workgroups per compute unit.
uint32_t gemm16_ragged_splits(uint32_t M, uint32_t N, uint32_t K, uint32_t *kper)
{
    const uint32_t tiles = ((M + 63u) / 64u) * ((N + 63u) / 64u), ktiles = (K + 63u) / 64u;
    *kper = 0;
    if (tiles >= 256u || ktiles < 2u) return 1;
    uint32_t splits = (512u + tiles - 1) / tiles;
    if (splits > 16u) splits = 16u;
    if (splits > ktiles) splits = ktiles;
    const uint32_t per = (ktiles + splits - 1) / splits;
    *kper = per * 64u;
    return (ktiles + per - 1) / per;
}

// K splits of the single-stage kernel for the other rows.  A tile walks its sums one K tile behind the other with a single one in
// flight, 0.7 us each of 128, so a layer of few tiles and long sums waits on that chain, the chip nearly empty.  Up to a tile
// per compute unit, two workgroups on each, at least four K tiles a part.  Forward of one layer, unsplit / split, us:
//            samples x outputs   INT8 at K 1024    2048        3072        8192        FP16 at K 3072   8192
//              260 x 100            8.6 /  8.6                 25.9 / 13.3 58.4 / 17.7   24.2 / 13.4   53.2 / 17.7
//             1000 x 250           13.6 / 13.6   22.0 / 22.1   31.5 / 20.4 67.4 / 27.8   30.7 / 20.0   63.1 / 28.5
//             2000 x 130           17.1 / 17.0   22.7 / 18.2   30.8 / 21.4 69.6 / 36.9   29.3 / 21.3   64.3 / 37.1
//             6500 x  73           18.6 / 18.7   30.2 / 27.7   41.9 / 37.1  106 / 86     41.0 / 37.3    102 / 86
// The partial sums and their launch cost 3 us and 4.4 a million, so the more outputs, the longer the sums for which that pays (INT8,
// us):
//            samples x outputs      K 1280        1536          1792          2048          2304          2560          3072
//             5000 x  75         20.0 / 19.0   22.3 / 19.9   24.6 / 21.6   27.6 / 23.4   29.7 / 25.0
//             1600 x 256                       17.5 / 17.2   20.0 / 18.1   21.8 / 19.3   24.1 / 19.7
//             2000 x 250         16.0 / 16.5   18.2 / 18.1   20.1 / 18.5   22.2 / 18.9   24.2 / 19.3
//             1024 x 512         14.4 / 15.6   16.3 / 17.2   18.2 / 18.0   20.0 / 19.4   21.9 / 20.5
//             1000 x 640         14.5 / 16.8   16.2 / 17.9   18.2 / 19.2   19.9 / 21.4   22.0 / 21.3   24.3 / 21.9   28.4 / 23.7
//             1000 x 1000        14.9 / 19.2   16.9 / 20.5   18.7 / 21.6   20.5 / 22.1   23.2 / 22.6   25.3 / 23.6   29.0 / 25.8
//             INT4               14.6 / 18.7   16.7 / 20.2   18.4 / 21.4   19.9 / 22.7   22.2 / 24.4   24.1 / 25.5   (at 2688 25.1 / 25.6)
// From 257 tiles on it loses below K = 3000 and gains little above: 2000 x 640 at K = 1024 16.4 / 22.8, 2048 26.1 / 26.5, 3584
// 38.6 / 36.7; 1300 x 1250 at 1024 17.8 / 26.5, 3584 39.9 / 42.9.  1024 workgroups are no faster (1000 x 250 at 8192 30.4), 256
// lose at large batches (2000 x 130 at 8192 41.3), and parts of two K tiles cost short sums (1000 x 640 at 1024 17.7 / 19.7).
uint32_t gemm16_single_splits(uint32_t M, uint32_t N, uint32_t K, uint32_t *kper)
{
    const uint32_t tiles = ((M + 63u) / 64u) * ((N + 63u) / 64u), ktiles = (K + 127u) / 128u;
    *kper = 0;
    if (tiles > 256u) return 1;
    const uint32_t outputs = M * N;                                          // (a million at most)
    if (K < (outputs <= 430000u ? 1024u : outputs <= 530000u ? 1792u : outputs <= 700000u ? 2560u : 2816u)) return 1;
    uint32_t splits = (512u + tiles - 1) / tiles;
    if (splits > 16u) splits = 16u;
    if (splits > K / 512u) splits = K / 512u;
    if (splits <= 1u) return 1;
    const uint32_t per = (ktiles + splits - 1) / splits;
    *kper = per * 128u;
    return (ktiles + per - 1) / per;
}

// Whether the single-stage kernel is the better one where the 256 x 256 tiles of integer codes would be split over K: up to K = 4608,
// and longer ones of more than two of its tiles a compute unit whose workgroups would leave most of a second round idle.  Inputs of
// such widths took it before they ran padded (unpadded / padded on large tiles / padded here, 4104 x 1030 INT4 at 700 / 1500 / 4000
// samples 40 / 44 / 31, 44 / 53 / 45, 88 / 112 / 91 us; 6024 x 1030 at 4000 125 / 140 / 129; tiles / here, 4104 x 2050 at 1000 70 / 55,
// x 3000 at 2500 116 / 120; 8200 x 1500 at 2500 130 / 135; 6024 x 770 at 4000, in one round, 96 / 110).
bool gemm16_split_wasted(uint32_t M, uint32_t N, uint32_t K, uint32_t workgroups)
{
    if (K <= 4608u) return true;
    const uint64_t tiles = (uint64_t)((M + 63u) / 64u) * ((N + 63u) / 64u);
    return K <= 8192u && tiles > 512u && 2u * ((workgroups + 255u) / 256u * 256u) >= 3u * workgroups;
}

// What the thin-operand kernel needs beyond the layer itself
struct ThinCtx {
    const uint16_t *w16;   // [N][K] 16-bit weights (raw 16-bit formats, or FP16 codes) when N <= 64, else nullptr
    float *ws;             // split-K workspace
    uint64_t ws_floats;
    bool x_f32;            // A is still the caller's FP32 input (the layer is one gemm16_small_layer() accepts)
    void *soft_out;        // softmax layer: where the normalised outputs go if the layer's kernel can do it itself ...
    int soft_kind;         // ... as 0 FP32, 1 BF16, 2 FP16, 3 FP16 in two halves (not by sp_skinny16_kw_head, which has no place for the second)
    bool *soft_done;       // ... and whether it did
    bool padded_in;        // the first layer, with the caller's rows padded (padded_width)
};

struct ThinPlan {
    bool use;
    bool mode_b;
    bool kw;               // thin operand of <= 8 rows: K split among the waves of a workgroup (sp_skinny16_kw)
    int nw;                // waves per workgroup in that case (4 or 8)
    bool head;             // few outputs: sp_skinny16_kw_head
    int nt;                // sixteens of outputs in that case
    uint32_t R, NC;        // streamed rows, thin rows
    int rt, ct;
    int nwv;               // waves per workgroup of sp_skinny16_regs
    bool regs;             // sp_skinny16_regs instead of sp_skinny16
    int st;                // sixteens of samples per workgroup of sp_skinny16 and sp_skinny16_kw_head
    uint32_t splits, kper, row_blocks, cblocks;
};

// Largest batch the weight-streaming kernel takes before the tiled GEMM does better (which runs from 65 samples up, a
// partly filled row of 256 x 256 tiles).  Measured per layer, streaming against tiles, at 128 and 192 samples:
// 8192 x 8192 BF16 57 / 107 against 48 / 57 us (tiles from 65 samples: 54 against 43 us there); 8192 x 8192 INT8 36 / 66
// against 41 / 54 us and 16384 x 16384 INT8 108 / 175 against 119 / 145 us (tiles from 129); 16384 x 16384 INT4 82 / 141
// against 104 / 143 us, 4096 x 16384 INT4 34 / 54 against 52 / 71 us, 8192 x 8192 INT2 29 / 44 against 40 / 52 us (streaming
// up to 256).  The fewer bytes a code has, the longer re-reading the weights per block of 64 samples pays.
// Layers of a few megabytes stay with the streaming kernel up to 256 samples, where the tiles would be a handful.  Sums of up to
// 1024 leave it at 65: the tiles take them without a K split (8192 x 784 INT8 at 128 samples 20 -> 13 us).
uint32_t thin_max_samples(int fmt, uint32_t N, uint32_t K)
{
    if (K <= 1024u) return 64u;
    if ((uint64_t)N * K * (uint64_t)fmt_bits(fmt) / 8u <= (8ull << 20)) return 256u;
    return fmt_bits(fmt) == 16 ? 64u : fmt == I8 ? 128u : 256u;
}

// codes of K in a chunk of sp_skinny16 (ThinFmt)
uint32_t thin_chunk(int fmt) { return fmt == I4 || fmt == I2 ? ThinFmt<I4>::BK : ThinFmt<I8>::BK; }
static_assert(ThinFmt<I2>::BK == ThinFmt<I4>::BK && ThinFmt<F16>::BK == ThinFmt<I8>::BK && ThinFmt<BF16>::BK == ThinFmt<I8>::BK, "thin_chunk");

// K splits of sp_skinny16: what costs least by the times measured for it (us): a chunk on st sixteens of samples, or its weights
// at the rate at which the chip reads them; the start and end of a workgroup, of which a compute unit holds one; the second
// launch that adds the parts.  At most most_sums of them: what the caller's workspace holds.
uint32_t thin_splits(int fmt, int st, uint32_t wgs, uint32_t chunks, uint64_t outputs, uint64_t most_sums)
{
    const bool narrow = fmt == I2 || fmt == I4;
    const float products = narrow ? 0.55f + 0.20f * st : 0.35f + 0.11f * st;
    const float bytes = 16.0f * (float)thin_chunk(fmt) * (float)fmt_bits(fmt);           // 128 rows of a chunk
    uint32_t best = 1;
    float least = 0.0f;
    for (uint32_t s = 1; s <= 16u && (s == 1u || (2u * s <= chunks && s * outputs <= most_sums)); ++s) {
        const float at_once = wgs * s < 256u ? (float)(wgs * s) : 256.0f;
        const float chunk = fmaxf(products, at_once * bytes / 5.5e6f);
        const float t = (float)((wgs * s + 255u) / 256u) * ((float)((chunks + s - 1) / s) * chunk + 3.5f) +
                        (s > 1u ? 3.2f + (float)s * (float)outputs * 1e-6f : 0.0f);
        if (s == 1u || t < least) {
            best = s;
            least = t;
        }
    }
    return best;
}

// mode_b streams 16-bit activations (fmt = the activation type), mode a the weights.  most_sums: thin_splits().  halves: activation
// matrices.
ThinPlan plan_thin(int fmt, uint32_t M, uint32_t N, uint32_t K, uint64_t most_sums = ~0ull, uint32_t halves = 1)
{
    ThinPlan p{};
    // Few outputs: sp_skinny16_kw_head, one launch.  Against sp_skinny16_regs and its reduction (more than 16 outputs; us, FP16):
    // 1024 x 20 at 16 / 1000 / 16384 samples 12.8 / 15.5 / 42.4 -> 7.6 / 8.7 / 27.6, 1536 x 48 14.5 / 18.4 / 56.6 -> 12.5 / 14.4 /
    // 43.6.  Its eight waves are all the K split there is for more than 16 outputs, and a workgroup reads all weights for its samples:
    // few samples of longer sums into many outputs are left to the split (2048 x 50 at 16 samples 12.7 against 13.1, at 256 18.4
    // against 16.5; 3072 x 32 at 16 samples 12.0 against 13.0, x 20 11.9 against 11.6, with split activations 15.8 against 16.1;
    // 3072 x 40 at 64 16.4 against 17.3, at 1000 21.7 against 20.4).  Up to 16 outputs K is cut over the grid as well where the samples
    // are few, in parts of 1024 from 3072 on (x 16 at K = 4096, 16 / 64 / 1000 samples 11.8 / 12.1 / 15.7 whole, 9.2 / 9.9 / 14.5 in
    // four; with split activations 15.8 / 16.1 / 20.7 and 10.0 / 11.2 / 16.8, x 1 12.6 / 13.0 / 17.4 and 9.3 / 10.3 / 15.6), up to eight
    // of them (x 16 at 16384 and 64 samples 14.4, in four 16.3); up to eight outputs of unsplit activations, or of as few samples, in parts of
    // 2048 beyond 4096, below which the second launch costs what they bring (x 8 at 4096 and 64 samples 10.8 whole, 11.3 in four).  From 129
    // workgroups on no longer (x 16 at 4096 and 4096 samples 25.9 whole, 28.9 in two), but for rows of split activations that L2 does
    // not hold (x 10 at 16384 and 4096 samples 178 and 163).  Two sixteens of samples a workgroup where there are enough to fill the
    // chip with them (1024 x 33 at 8192 samples 23.4 -> 20.9, at 4096 16.5 -> 17.2), not with one of outputs (1000 x 10 at 8192
    // samples 15.3 -> 16.7 in workgroups of 64).
    const int nt = N <= 16u ? 1 : N <= 32u ? 2 : 4;
    if (N <= 64 && K % 8u == 0 && M >= 1 &&
        (nt == 1 || (K * nt <= 6144u && (halves == 2u || N * K <= (84u << 10))) || (K <= 2048u && M >= 128u) || (K <= 3072u && M >= 1000u))) {
        p.use = p.mode_b = p.head = true; p.R = M; p.NC = N;
        p.nt = nt;
        p.st = p.nt > 1 && M >= 8192u ? 2 : 1;
        p.cblocks = 1;
        p.row_blocks = (M + 16u * p.st - 1u) / (16u * p.st);
        const uint32_t steps = (K + 31u) / 32u;
        const bool fine = nt == 1 && (N > 8u || (halves == 2u && M > 8u));
        uint32_t splits = K > 4096u ? K / 2048u : 1u;
        if (fine && K >= 3072u && splits < 8u) splits = K / 1024u < 8u ? K / 1024u : 8u;
        const uint32_t room = (halves == 2u && K >= 16384u ? 512u : 256u) / p.row_blocks;
        if (splits > room) splits = room;
        if (splits > 16u) splits = 16u;
        if (splits > most_sums / ((uint64_t)M * N)) splits = (uint32_t)(most_sums / ((uint64_t)M * N));
        if (splits < 1u) splits = 1u;
        const uint32_t per = (steps + splits - 1u) / splits;
        p.kper = per * 32u;
        p.splits = (steps + per - 1u) / per;
        return p;
    } else if (N <= 64 && K % 8u == 0 && M >= 1) {
        p.use = true; p.mode_b = true; p.R = M; p.NC = N;
    } else if (M >= 16u && (uint64_t)N * K <= (128u << 10)) {
        // a layer of a few hundred rows and columns gives this kernel two or three workgroups, each fetching the whole
        // thin operand before it starts: the single-stage tile kernel is quicker from 16 samples on (eight 256 x 256
        // layers at 64 samples: 51 against 73-79 us in every format)
        return p;
    } else if (M <= thin_max_samples(fmt, N, K) && rows_aligned(fmt, K) && K % 8u == 0) {
        p.use = true; p.mode_b = false; p.R = N; p.NC = M;
    } else {
        return p;
    }
    const int sfmt = p.mode_b ? F16 : fmt;
    // the kernel addresses both operands with 32-bit lane offsets
    if ((uint64_t)p.R * K * (uint64_t)fmt_bits(sfmt) / 8u >= (1ull << 32) || (uint64_t)p.NC * K * 2u >= (1ull << 32)) {
        p.use = false;
        return p;
    }
    const uint32_t bkc = sfmt == I8 ? 128u : (sfmt == I4 || sfmt == I2) ? 256u : 64u;
    // K split inside the workgroup (sp_skinny16_kw) for thin operands of at most 8 rows.  Every wave then fetches its
    // own thin chunks (four times the thin traffic, from L2), which pays where the second launch of the split-K path
    // weighs more: measured faster for INT8 at every size tried, for INT4 / INT2 up to 64 MB and for 16-bit operands
    // up to 32 MB of streamed bytes, slower beyond (16384 x 16384 INT4 at 8 samples: 40 us against 34 us).
    const uint64_t streamed_bytes = (uint64_t)p.R * K * (uint64_t)fmt_bits(sfmt) / 8u;
    const bool kw_pays = sfmt == I8 || streamed_bytes <= ((sfmt == I4 || sfmt == I2) ? (64ull << 20) : (32ull << 20));
    if (p.NC <= 8u && kw_pays) {
        // one workgroup per 32 streamed rows, its four waves share K; K is split across workgroups as well only
        // when the rows alone do not fill the chip
        p.kw = true;
        p.rt = p.ct = 1;
        p.cblocks = 1;
        p.row_blocks = (p.R + 31u) / 32u;
        const uint32_t chunks = (K + bkc - 1) / bkc;
        // 6144 to 12287 streamed rows: eight waves per workgroup instead of a K split across two workgroups
        p.nw = (p.row_blocks >= 192u && p.row_blocks < 384u && chunks >= 16u) ? 8 : 4;
        uint32_t splits = p.row_blocks >= 192u ? 1u : (512u + p.row_blocks - 1) / p.row_blocks;
        if (splits > 16u) splits = 16u;
        if (splits > chunks / 4u) splits = chunks / 4u;
        if (splits < 1u) splits = 1u;
        const uint32_t cps = (chunks + splits - 1) / splits;
        p.kper = cps * bkc;
        p.splits = (chunks + cps - 1) / cps;
        return p;
    }
    // sp_skinny16: workgroups of 128 rows by up to 64 samples.  More of them than compute units with several blocks of samples
    // would read the samples' chunks from L2 twice as often as the 256 rows of sp_skinny16_regs do (INT2 at 256 samples:
    // 16384 x 2048 35 against 27 us, 16384 x 8192 84 against 70; at 100 samples 16384 x 8192 48.5 against 45.7, but x 4096 29.6
    // against 31.8).  Exactly as many as compute units, which is 8065 to 8192 rows at 193 to 256 samples, from K = 8192 on:
    // 8192 x 8192 INT2 44.3 against 42.5, INT4 45.3 against 47.6, 8192 x 16384 76 against 68 and 80 against 79; fewer never.
    const uint32_t blocks = (p.R + 127u) / 128u * ((p.NC + 63u) / 64u);
    p.regs = p.mode_b || ((fmt == I4 || fmt == I2) && p.NC > 64u && (blocks > 256u || (blocks == 256u && K >= 8192u)));
    if (!p.regs) {
        p.cblocks = (p.NC + 63u) / 64u;
        p.st = (int)(((p.NC + p.cblocks - 1u) / p.cblocks + 15u) / 16u);
        p.row_blocks = (p.R + 127u) / 128u;
        const uint32_t bk = thin_chunk(fmt), chunks = (K + bk - 1) / bk;
        p.splits = thin_splits(fmt, p.st, p.row_blocks * p.cblocks, chunks, (uint64_t)p.NC * p.R, most_sums);
        const uint32_t cps = (chunks + p.splits - 1) / p.splits;
        p.kper = cps * bk;
        p.splits = (chunks + cps - 1) / cps;
        return p;
    }
    p.ct = p.NC <= 32 ? 1 : 2;
    p.cblocks = (p.NC + 32u * p.ct - 1) / (32u * p.ct);
    // Waves per workgroup, and the number of workgroups the K split aims at.  Every workgroup fetches the thin block
    // of its K share once, so eight waves (256 streamed rows) halve that traffic; they pay from 16384 streamed rows, and
    // with several blocks of thin rows (8192 x 8192 INT2 at 256 samples 45 against 53 us, 8100 rows 42.6 against 50.2), four
    // waves stay better on smaller layers (8192 x 8192 INT8 at 64 samples 27.3 against 29.0 us).  One workgroup per compute unit is the target:
    // twice as many K splits write twice the partial sums (16384 x 16384 INT4 at 64 samples 67 us, 8192 x 8192 INT8
    // 38 us), half as many leave compute units idle (74 us).  Two row tiles per wave were slower wherever tried.
    p.rt = 1;
    p.nwv = (p.R >= 16384u || p.cblocks > 1u) ? 8 : 4;
    const uint32_t target = 256u;
    p.row_blocks = (p.R + 32u * p.nwv * p.rt - 1) / (32u * p.nwv * p.rt);
    const uint32_t chunks = (K + bkc - 1) / bkc;
    const uint32_t wgs = p.row_blocks * p.cblocks;
    uint32_t splits = (target + wgs - 1) / wgs;
    if (splits > 16u) splits = 16u;
    if (splits > chunks / 2u) splits = chunks / 2u;
    if (splits < 1u) splits = 1u;
    const uint32_t cps = (chunks + splits - 1) / splits;
    p.kper = cps * bkc;
    p.splits = (chunks + cps - 1) / cps;
    return p;
}

template <int SFMT, bool F16T, int RT, int CT, int NWV = 4>
void launch_thin_inst(const SkinnyArgs &a, const ThinPlan &p)
{
    if (tl_route.dry) return;
    constexpr size_t lds = 2 * 32 * CT * SkinnyFmt<SFMT>::PITCH;
    auto kern = sp_skinny16_regs<SFMT, F16T, RT, CT, NWV>;
    static bool once = ((void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), true);
    (void)once;
    const uint32_t gx = p.cblocks > 1 ? (p.row_blocks + 7u) / 8u * 8u * p.cblocks : p.row_blocks;
    kern<<<dim3(gx, p.splits * a.halves, 1), 64 * NWV, lds, g_stream>>>(a);
}

template <int FMT, bool F16T, int ST>
void launch_thin_dma(const SkinnyArgs &a, const ThinPlan &p)
{
    if (tl_route.dry) return;
    constexpr size_t lds = ThinFmt<FMT>::template Tile<ST>::LDS;
    auto kern = sp_skinny16<FMT, F16T, ST>;
    static bool once = ((void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), true);
    (void)once;
    const uint32_t gx = p.cblocks > 1 ? (p.row_blocks + 7u) / 8u * 8u * p.cblocks : p.row_blocks;
    kern<<<dim3(gx, p.splits * a.halves, 1), 512, lds, g_stream>>>(a);
}

template <int SFMT, bool F16T, int NW>
void launch_thin_kw(const SkinnyArgs &a, const ThinPlan &p)
{
    if (tl_route.dry) return;
    constexpr size_t lds = (size_t)NW * 2 * 8 * SkinnyFmt<SFMT>::PITCH + (size_t)NW * 4 * 64 * sizeof(float);
    auto kern = sp_skinny16_kw<SFMT, F16T, NW>;
    static bool once = ((void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), true);
    (void)once;
    kern<<<dim3(p.row_blocks, p.splits * a.halves, 1), 64 * NW, lds, g_stream>>>(a);
}

template <bool F16T, int HALVES>
void launch_thin_head(const SkinnyArgs &a, const ThinPlan &p)
{
    if (tl_route.dry) return;
    const dim3 grid(p.row_blocks, p.splits);
    if (p.nt == 1) sp_skinny16_kw_head<F16T, 1, 1, HALVES><<<grid, 512, 0, g_stream>>>(a);
    else if (p.nt == 2 && p.st == 1) sp_skinny16_kw_head<F16T, 2, 1, HALVES><<<grid, 512, 0, g_stream>>>(a);
    else if (p.nt == 2) sp_skinny16_kw_head<F16T, 2, 2, HALVES><<<grid, 512, 0, g_stream>>>(a);
    else if (p.st == 1) sp_skinny16_kw_head<F16T, 4, 1, HALVES><<<grid, 512, 0, g_stream>>>(a);
    else sp_skinny16_kw_head<F16T, 4, 2, HALVES><<<grid, 512, 0, g_stream>>>(a);
}

template <int SFMT, bool F16T>
void launch_thin(SkinnyArgs a, const ThinPlan &p)
{
    if (p.splits == 1 && (a.halves == 1 || p.head)) a.ws = nullptr;
    a.ksplits = p.splits;
    a.parts = p.head ? p.splits : p.splits * a.halves;
    if (p.head) {
        if constexpr (F16T) {
            if (a.halves == 2) launch_thin_head<true, 2>(a, p);
            else launch_thin_head<true, 1>(a, p);
        } else {
            launch_thin_head<false, 1>(a, p);
        }
    } else if (p.kw) {
        if (p.nw == 8) launch_thin_kw<SFMT, F16T, 8>(a, p);
        else launch_thin_kw<SFMT, F16T, 4>(a, p);
    } else if (!p.regs) {
        if (p.st == 1) launch_thin_dma<SFMT, F16T, 1>(a, p);
        else if (p.st == 2) launch_thin_dma<SFMT, F16T, 2>(a, p);
        else if (p.st == 3) launch_thin_dma<SFMT, F16T, 3>(a, p);
        else launch_thin_dma<SFMT, F16T, 4>(a, p);
    } else if constexpr (SFMT == I4 || SFMT == I2) {
        launch_thin_inst<SFMT, F16T, 1, 2, 8>(a, p);
    } else if constexpr (SFMT == F16 || SFMT == BF16) {
        if (p.nwv == 8) {
            if (p.ct == 2) launch_thin_inst<SFMT, F16T, 1, 2, 8>(a, p); else launch_thin_inst<SFMT, F16T, 1, 1, 8>(a, p);
        } else {
            if (p.ct == 2) launch_thin_inst<SFMT, F16T, 1, 2>(a, p); else launch_thin_inst<SFMT, F16T, 1, 1>(a, p);
        }
    }
    if (a.ws && a.soft_out && !tl_route.dry) {
        launch_sum_softmax({a.ws, p.splits, a.parts, a.NC, a.R, a.L, a.soft_out, a.soft_kind, 0});
    } else if (a.ws && !tl_route.dry) {
        const uint64_t total = (uint64_t)a.NC * a.R;
        // four rows per thread where they are neighbours in the workspace and in C, and both are 16-byte aligned
        const bool vec = !a.mode_b && a.R % 4u == 0 && (reinterpret_cast<uintptr_t>(a.ws) & 15u) == 0 &&
                         (reinterpret_cast<uintptr_t>(a.C) & 15u) == 0;
        if (vec) sp_skinny_reduce<F16T, true><<<(uint32_t)((total / 4u + 255) / 256), 256, 0, g_stream>>>(a, p.splits);
        else sp_skinny_reduce<F16T, false><<<(uint32_t)((total + 255) / 256), 256, 0, g_stream>>>(a, p.splits);
    }
}

// Layers that run in one launch of sp_gemm16_small: more than 64 outputs (fewer stream the activations), at most 512
// tiles of 32 x 32, K up to 2048 (its eight waves are all the K split there is), and tiles x K up to 512 K: every tile
// reads 64 rows of K elements from L2.  Measured, whole nets, against the streaming / tiled kernels with their K split
// over the grid, second launch and separate conversion of the input: 784-512-1000-10 INT8 at 16 / 256 / 512 samples
// 16.5 / 18.9 / 22.3 against 24.8 / 29.8 / 28.0 us, FP16 at 5 samples 16 against 23 us; eight 256 x 256 layers at 5 / 64 /
// 1024 samples 25 / 31 / 35 against 42 / 51 / 49 us, three 1024 x 1024 layers at 256 samples 24 against 38 us, at 512
// samples (512 tiles x 1024) 40 against 41 us; beyond the bound it loses: two 2048 x 2048 layers at 256 samples (512
// tiles x 2048) 46 against 35 us.
bool gemm16_small_layer(uint32_t M, uint32_t N, uint32_t K, uint32_t halves)
{
    if (K % 8u != 0 || K > 2048u || N <= 64u) return false;
    const uint64_t tiles = (uint64_t)((M + 31u) / 32u) * ((N + 31u) / 32u);
    // (split activations: two activation matrices against one of weights, a tile reads 96 rows instead of 64)
    return tiles <= 512u && tiles * K * (1u + halves) <= (1024u << 10);
}

template <int FMT, bool F16T>
void launch_gemm16_fmt(const LayerArgs &L, const uint16_t *A, void *C, uint32_t M, int out_f32, const ThinCtx &ctx)
{
    const uint32_t halves = tl_route.halves;
    // (a small layer behind a padded input stays on the single-stage kernel: its conversion is a launch of its own anyway)
    const bool single = ctx.padded_in && gemm16_small_layer(M, L.N, L.K, halves);
    if (!single && gemm16_small_layer(M, L.N, L.K, halves) && (reinterpret_cast<uintptr_t>(A) & 15u) == 0) {
        GemmArgs g{L, A, C, M, out_f32, nullptr, 0, 1, 1};
        tl_route.name = "sp_gemm16_small";
        if (tl_route.dry) return;
        const uint32_t grid = ((M + 31u) / 32u) * ((L.N + 31u) / 32u);
        if constexpr (F16T) {
            if (halves == 2) {
                if (ctx.x_f32) sp_gemm16_small<FMT, F16T, true, 2><<<grid, 512, 0, g_stream>>>(g);
                else sp_gemm16_small<FMT, F16T, false, 2><<<grid, 512, 0, g_stream>>>(g);
                return;
            }
        }
        if (ctx.x_f32) sp_gemm16_small<FMT, F16T, true><<<grid, 512, 0, g_stream>>>(g);
        else sp_gemm16_small<FMT, F16T, false><<<grid, 512, 0, g_stream>>>(g);
        return;
    }
    const ThinPlan tp = plan_thin(FMT, M, L.N, L.K, ctx.ws_floats / halves, halves);
    if (tp.use && !single && (!tp.mode_b || ctx.w16) &&
        ((tp.splits == 1 && (halves == 1 || tp.head)) || (uint64_t)tp.splits * halves * tp.NC * tp.R <= ctx.ws_floats)) {
        SkinnyArgs a{};
        a.halves = halves; a.half_elems = (uint64_t)M * L.K;
        a.L = L; a.C = C; a.ws = ctx.ws; a.R = tp.R; a.NC = tp.NC; a.row_blocks = tp.row_blocks; a.cblocks = tp.cblocks; a.kper = tp.kper; a.out_f32 = out_f32; a.mode_b = tp.mode_b ? 1 : 0;
        tl_route.name = tp.head ? "sp_skinny16_kw_head" : tp.kw ? "sp_skinny16_kw" : tp.regs ? "sp_skinny16_regs" : "sp_skinny16";
        if (tp.mode_b) {
            if (ctx.soft_out && tp.head && tp.splits == 1 && ctx.soft_kind != 3) {
                a.soft_out = ctx.soft_out;
                a.soft_kind = ctx.soft_kind;
                *ctx.soft_done = true;
            }
            a.stream = reinterpret_cast<const uint8_t *>(A);
            a.thin = ctx.w16;
            launch_thin<F16T ? F16 : BF16, F16T>(a, tp);
        } else {
            if (ctx.soft_out && (tp.splits > 1 || halves == 2) && soft_sums_pay(M, L.N)) {
                a.soft_out = ctx.soft_out;
                a.soft_kind = ctx.soft_kind;
                *ctx.soft_done = true;
            }
            a.stream = L.w;
            a.thin = A;
            launch_thin<FMT, F16T>(a, tp);
        }
        return;
    }
    GemmArgs g{L, A, C, M, out_f32, nullptr, 0, 1, halves};
    const bool soft_sums = ctx.soft_out && soft_sums_pay(M, L.N);          // if there are partial sums
    const bool aligned = rows_aligned(FMT, L.K) && (L.K % 8u == 0);
    const bool fits32 = (uint64_t)M * L.K * 2u < (1ull << 32) && (uint64_t)L.N * L.K * 2u < (1ull << 32);   // 32-bit DMA offsets
    // the 256 x 256 tiles need about a tile per compute unit; smaller problems fill the chip better with 128 x 128
    const uint32_t bm = gemm16_tile_rows(FMT, M, L.N);
    const uint32_t big_tiles = ((M + bm - 1) / bm) * ((L.N + 255u) / 256u);
    const uint32_t splits = gemm16_splits(FMT, M, L.N, L.K, &g.kper);
    const bool split_ok = splits > 1 && (uint64_t)splits * halves * M * L.N <= ctx.ws_floats;
    const bool halves_ok = halves == 1 || (uint64_t)halves * M * L.N <= ctx.ws_floats;     // (checked by the caller's reserve)
    // (too few tiles and no K split, gemm16_splits: the single-stage kernel below)
    const bool shared_cu = halves == 1 && bm == 256u && L.K <= gemm16_shared_limit(FMT, L.act, big_tiles, (uint64_t)M * L.N);
    const bool wasted = ctx.padded_in && fmt_bits(FMT) < 16 && splits > 1u && gemm16_split_wasted(M, L.N, L.K, big_tiles * splits);
    if (aligned && !shared_cu && !wasted && L.K >= 128u && M > 64 && L.N >= 256 && fits32 && (big_tiles >= 192u || split_ok) && halves_ok) {
        if (big_tiles >= 192u) g.kper = 0;
        else g.ksplits = splits;
        if (g.kper || halves == 2) g.ws = ctx.ws;
        const dim3 grid(big_tiles, g.ksplits * halves);
        tl_route.name = "sp_gemm16_big";
        if (tl_route.dry) return;
        if (bm == 128u) {
            // 128-row tiles (gemm16_tile_rows)
            constexpr size_t lds = BigTile<FMT, 4>::LDS;
            auto kern = sp_gemm16_big<FMT, F16T, 4>;
            static bool once = ((void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), true);
            (void)once;
            kern<<<grid, 256, lds, g_stream>>>(g);
        } else {
            constexpr size_t lds = BigTile<FMT, 8>::LDS;
            auto kern = sp_gemm16_big<FMT, F16T, 8>;
            static bool once = ((void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), true);
            (void)once;
            kern<<<grid, 256, lds, g_stream>>>(g);
        }
        if (g.ws && soft_sums) {
            launch_sum_softmax({g.ws, g.ksplits, g.ksplits * halves, M, L.N, L, ctx.soft_out, ctx.soft_kind, 0});
            *ctx.soft_done = true;
        } else if (g.ws) {
            const uint64_t total = (uint64_t)M * L.N;
            const bool vec = L.N % 4u == 0 && (reinterpret_cast<uintptr_t>(g.ws) & 15u) == 0 && (reinterpret_cast<uintptr_t>(C) & 15u) == 0;
            if (vec) sp_gemm16_reduce<F16T, true><<<(uint32_t)((total / 4u + 255) / 256), 256, 0, g_stream>>>(g, g.ksplits);
            else sp_gemm16_reduce<F16T, false><<<(uint32_t)((total + 255) / 256), 256, 0, g_stream>>>(g, g.ksplits);
        }
        return;
    }
    g.kper = 0;
    g.ksplits = 1;
    if (halves == 2) g.ws = ctx.ws;                  // one partial sum per activation matrix, added by the reduction
    const bool words = !aligned && L.K % 8u == 0 && ((uint64_t)L.K * fmt_bits(FMT)) % 32u == 0 && (FMT == I8 || FMT == I4 || FMT == I2);
    {
        const bool plain = (!aligned && !words) || single;
        uint32_t kper = 0;
        const uint32_t sp = plain ? gemm16_ragged_splits(M, L.N, L.K, &kper) : gemm16_single_splits(M, L.N, L.K, &kper);
        if (sp > 1 && (uint64_t)sp * halves * M * L.N <= ctx.ws_floats) {
            g.kper = kper;
            g.ksplits = sp;
            g.ws = ctx.ws;
        }
    }
    tl_route.name = "sp_gemm16";
    if (tl_route.dry) return;
    // This kernel has one LDS stage, so it lives on the number of resident workgroups: the largest of 128 x 128,
    // 64 x 128 and 64 x 64 tiles that still gives two workgroups per compute unit (measured: 4096 x 512 x 784 INT8
    // 21.7 / 16.2 / 12.9 us, 8192 x 8192 x 1000 BF16 0.27 / 0.37 / 0.42 ms); the element-wise loads of unaligned
    // rows always want the smallest (8192 x 8192 x 1000 INT8: 1.90 / 1.69 / 1.51 ms).
    auto tiles = [&](uint32_t bm, uint32_t bn) { return ((M + bm - 1) / bm) * ((L.N + bn - 1) / bn); };
    // (words: integer codes whose rows are whole 32-bit words, not whole 16-byte units, next to aligned activations)
    const int shape = !(aligned || words) ? 11 : tiles(128, 128) >= 512u ? 22 : tiles(64, 128) >= 512u ? 12 : 11;
    // K of 1024 and more: K tiles of 128 instead of 64, half as many rounds of load, barrier, store, barrier (600 x 1280 x
    // 1536 FP16 18.2 -> 14.1 us, 4096 x 512 x 4096 48.6 -> 37.9 us; below 1024 no gain: 4096 x 512 x 784 INT8 12.5 / 13.0 us)
    const bool deep = (aligned || words) && (single ? g.kper == 0 : g.kper % 128u == 0) && L.K >= 1024u;
    auto go = [&](auto tm_c, auto tn_c) {
        constexpr int TM = decltype(tm_c)::value, TN = decltype(tn_c)::value;
        const dim3 grid(tiles(64 * TM, 64 * TN), g.ksplits * halves);
        if constexpr (TM == 1) {
            if (deep) {
                if constexpr (FMT == I8 || FMT == I4 || FMT == I2) {
                    if (words) {
                        sp_gemm16<FMT, F16T, TM, TN, true, true, 128><<<grid, 256, 0, g_stream>>>(g);
                        return;
                    }
                }
                sp_gemm16<FMT, F16T, TM, TN, true, false, 128><<<grid, 256, 0, g_stream>>>(g);
                return;
            }
        }
        if constexpr (FMT == I8 || FMT == I4 || FMT == I2) {
            if (words) {
                sp_gemm16<FMT, F16T, TM, TN, true, true><<<grid, 256, 0, g_stream>>>(g);
                return;
            }
        }
        if (aligned) sp_gemm16<FMT, F16T, TM, TN, true><<<grid, 256, 0, g_stream>>>(g);
        else sp_gemm16<FMT, F16T, TM, TN, false><<<grid, 256, 0, g_stream>>>(g);
    };
    using I1 = std::integral_constant<int, 1>;
    using I2c = std::integral_constant<int, 2>;
    if (shape == 22) go(I2c{}, I2c{});
    else if (shape == 12) go(I1{}, I2c{});
    else go(I1{}, I1{});
    if (g.ws && soft_sums) {
        launch_sum_softmax({g.ws, g.ksplits, g.ksplits * halves, M, L.N, L, ctx.soft_out, ctx.soft_kind, 0});
        *ctx.soft_done = true;
    } else if (g.ws) {
        const uint64_t total = (uint64_t)M * L.N;
        const bool vec = L.N % 4u == 0 && (reinterpret_cast<uintptr_t>(g.ws) & 15u) == 0 && (reinterpret_cast<uintptr_t>(C) & 15u) == 0;
        if (vec) sp_gemm16_reduce<F16T, true><<<(uint32_t)((total / 4u + 255) / 256), 256, 0, g_stream>>>(g, g.ksplits);
        else sp_gemm16_reduce<F16T, false><<<(uint32_t)((total + 255) / 256), 256, 0, g_stream>>>(g, g.ksplits);
    }
}

void launch_gemm16(int fmt, const LayerArgs &L, const uint16_t *A, void *C, uint32_t M, int out_f32, const ThinCtx &ctx)
{
    switch (fmt) {
    case F16:  launch_gemm16_fmt<F16, true>(L, A, C, M, out_f32, ctx); break;
    case BF16: launch_gemm16_fmt<BF16, false>(L, A, C, M, out_f32, ctx); break;
    // integer codes are exact in either 16-bit type; FP16 keeps 11 bits of the activations instead of 8
    case I8:   launch_gemm16_fmt<I8, true>(L, A, C, M, out_f32, ctx); break;
    case I4:   launch_gemm16_fmt<I4, true>(L, A, C, M, out_f32, ctx); break;
    default:   launch_gemm16_fmt<I2, true>(L, A, C, M, out_f32, ctx); break;     // FP32 weights never come here
    }
}

// K splits of the FP32 GEMM: enough workgroups for four per compute unit, at least two K tiles each (also for tiny
// layers: eight 256 x 256 layers at 5 .. 256 samples 58-62 us with the split and its second launch, 78-90 us without)
uint32_t gemm32_splits(uint32_t M, uint32_t N, uint32_t K, uint32_t *kper)
{
    const uint32_t tiles = ((M + 63) / 64) * ((N + 63) / 64), ktiles = (K + 31) / 32;
    uint32_t splits = (1024u + tiles - 1) / tiles;
    if (splits > 16u) splits = 16u;
    if (splits > ktiles / 2u) splits = ktiles / 2u;
    if (splits < 1u) splits = 1u;
    const uint32_t per = (ktiles + splits - 1) / splits;
    *kper = per * 32u;
    return (ktiles + per - 1) / per;
}

// The forward products' K splits.  From 512 tiles on, and from 256 tiles on when K is below 1024 (a short kernel, on
// which the second launch and the partial sums weigh most), the split costs more than idle compute units do: forward
// of one layer, no split against the rule above, 4096 x 512 x 784 40 against 48 us, 2048 x 1000 x 512 29 against 37 us,
// 1024 x 1000 x 512 19 against 26 us, 4096 x 256 x 256 11 against 21 us, 3000 x 1000 x 2000 135 against 142 us, four 512 x 512
// layers at 2048 / 4096 samples 67 / 106 against 105 / 149 us; but 256 to 511 tiles with a longer K keep it (130 x 8192 x
// 1024 46 against 56 us, 200 x 4096 x 1100 36 against 48 us, 700 x 2048 x 1536 63 against 72 us, 1500 x 1024 x 1024 47 against
// 50 us), and so do rows that are not whole 16-byte units, whose element-wise loads make every tile slow and an uneven
// last round expensive (4096 x 257 x 999).  Fewer than 256 tiles: as above (300 x 2048 x 2048 68 us unsplit, 42 us split
// seven ways).
uint32_t gemm32_fwd_splits(uint32_t M, uint32_t N, uint32_t K, uint32_t *kper)
{
    const uint32_t tiles = ((M + 63) / 64) * ((N + 63) / 64);
    if (K % 4u == 0 && (tiles >= 512u || (tiles >= 256u && K < 1024u))) {
        *kper = (K + 31u) / 32u * 32u;
        return 1;
    }
    return gemm32_splits(M, N, K, kper);
}

// FP32 layers of at most 64 outputs are one row of tiles at most; with up to eight samples, one pass of the vector
// kernel (a workgroup per row), that kernel is quicker than the matrix-core kernel and its reduction launch
// (16384 -> 64 -> 10 at 5 / 8 samples: 24 / 25 against 43 us; 8192 -> 10: 13 against 23 us; at 16 samples, two passes,
// 48 against 43 us.  Up to 64 K splits instead of 16 gave 32 us on the first and cost other thin layers 10 us.)
bool f32_thin_vector(const LayerArgs &L, uint32_t n) { return L.N <= 64u && n <= 8u; }

// Tile of sp_gemm32_small (32) or sp_gemm32_small16 for a layer that would otherwise need a K split and a second launch (or a handful of
// workgroups), 0 where the other kernels are the faster ones: 32 x 32 tiles up to 512 of them and K = 1024 (measured
// against the split path: 256 x 512 x 784 8 against 12 us, 1024 x 512 x 784 17 against 20 us, 1024 x 1024 x 1024 42 against 32 us); 16 x 16 tiles where the 32 x 32
// ones are at most 128 (128 x 1024 x 1024 7.3 against 8.8 us in a net of three, 400 x 300 x 300 even), which pays for longer
// and unaligned rows too (64 x 300 x 2000, 64 x 233 x 1038: 7 against 10 us), as long as their twice as many reads of K do
// not decide (64 x 2048 x 2048: 57 against 50 us for two layers).  *seg: the cut of the kernel that would take the layer
// without the 16 x 16 tiles.
uint32_t gemm32_small_tile(uint32_t M, uint32_t N, uint32_t K, bool vec, KSegments *seg)
{
    const uint64_t tiles = (uint64_t)((M + 31u) / 32u) * ((N + 31u) / 32u);
    uint32_t kper = 0;
    const uint32_t splits = gemm32_fwd_splits(M, N, K, &kper);
    const bool fits32 = splits > 1u && vec && tiles <= 512u && K <= 1024u;
    if (fits32) {
        const uint32_t steps = (K + 7u) / 8u, per = (steps + 7u) / 8u;
        *seg = KSegments{8u * per, (steps + per - 1u) / per, 1};
    } else {
        *seg = KSegments{kper, splits, 0};
    }
    if (tiles <= 128u && K <= 2048u && tiles * K <= (128u << 10)) return 16u;
    return fits32 ? 32u : 0u;
}

void launch_gemm32_small(const Gemm32Args &g, uint32_t tile, const KSegments &seg, float *soft_out, const DeltaTail &tail)
{
    const uint32_t grid = ((g.M + tile - 1u) / tile) * ((g.L.N + tile - 1u) / tile);
    if (tile == 32u) sp_gemm32_small<<<grid, 512, 0, g_stream>>>(g, soft_out);       // (no deltas: the caller's own launch)
    else if (seg.paired) sp_gemm32_small16<true><<<grid, 512, 0, g_stream>>>(g, seg, soft_out, tail);
    else sp_gemm32_small16<false><<<grid, 512, 0, g_stream>>>(g, seg, soft_out, tail);
}

// FP32 layers of up to 16 outputs and many samples: sp_gemm32_head up to K = 512 (16384 samples, softmax included: 128 x 10 16.8 ->
// 7.1 us, 256 x 16 19.3 -> 10.9, 512 x 16 24.2 -> 18.1; 777 x 10 26.9 against 34.9, 1000 x 10 35.8 against 42.8: its loads take 64
// bytes of 16 rows, the tiles' DMA whole lines).  Where it also forms a training step's output deltas, the launch and the passes it
// saves pay up to K = 1024 in one segment, from the second round of tiles on (a step of 32-K-N, tiles / head, us):
//                 K x N   640 x 1      640 x 10     784 x 1      784 x 10     1000 x 1     1000 x 10    1000 x 16
//   16384 samples       135 / 136    145 / 139    152 / 157    161 / 164    168 / 177    178 / 182    183 / 190
//   20000               163 / 163    175 / 165    177 / 178    191 / 182    203 / 206    216 / 210    225 / 222
//   50000                                         392 / 393                 467 / 475
// (a single output has no softmax to save).  Rows that are not whole 16-byte units: its loads lie across lines, while the tiles'
// go through LDS once (a layer alone, tiles / head, us: 10 outputs of 6000 samples K = 129 7.9 / 7.7, 301 10.1 / 11.2, 511 12.5 /
// 16.5; 10000 301 12.8 / 11.4, 402 13.4 / 13.2, 511 15.1 / 20.5; 20000 301 16.4 / 13.6, 482 21.9 / 24.5; 32768 402 24.4 / 22.5, 511
// 27.5 / 27.5; 66000 402 78 / 42).
bool gemm32_head_takes(uint32_t M, uint32_t N, uint32_t K, bool deltas, KSegments *seg)
{
    if (N > 16u || M < 2048u || K > 1024u) return false;
    uint32_t kper = 0;
    const uint32_t splits = gemm32_fwd_splits(M, N, K, &kper);
    *seg = KSegments{kper, splits, 0};
    if (K <= 512u) return K % 4u == 0 || K <= 128u || M >= 32768u || (K <= 320u && M >= 10000u);
    return deltas && splits == 1u && (K <= 640u || (N > 1u && M > 16384u));
}

void launch_gemm32_head(const Gemm32Args &g, const KSegments &seg, float *soft_out, const DeltaTail &tail)
{
    sp_gemm32_head<<<(g.M + 63u) / 64u, 256, 0, g_stream>>>(g, seg, soft_out, tail);
}

// Whether a forward product takes sp_gemm32_bf16_parts: from 2 G multiply-adds on, where its tiles fill the chip with more than
// their own start-up (2048 x 1024 x 1024 42 against 49 us in the FP32 kernels, 4096 x 1000 x 1000 68 against 91, 10000 x 512 x
// 784 71 against 88, 700 x 3000 x 3000 104 against 185; below: 2048 x 512 x 784 30 against 25, 1000 x 1024 x 1024 30 against 32),
// unless more than a fifth of the tiles would be padding (20000 x 130 x 100 25 against 17 us).  Training's products stay in
// the FP32 kernels and their order of sums: a run whose gradients nearly cancel multiplies a last-bit difference.
bool gemm32_parts_pay(uint32_t M, uint32_t N, uint32_t K)
{
    const uint64_t rows = (M + 127ull) / 128u * 128u, cols = (N + 127ull) / 128u * 128u;
    return K >= 64u && 5u * (uint64_t)M * N >= 4u * rows * cols && (double)M * N * K >= 2e9;
}

// K splits of sp_gemm32_bf16_parts: two workgroups per compute unit where there are fewer tiles than compute units, at least
// four K tiles each (512 x 4096 x 4096 106 us, 168 unsplit; three per compute unit 109; 700 x 3000 x 3000 104 / 143 / 109)
uint32_t gemm32_parts_splits(uint32_t M, uint32_t N, uint32_t K, uint32_t *kper)
{
    const uint64_t tiles = (M + 127ull) / 128u * ((N + 127ull) / 128u);
    const uint32_t ktiles = (K + 31u) / 32u;
    uint32_t splits = tiles >= 256u ? 1u : (uint32_t)((512u + tiles - 1u) / tiles);
    if (splits > 32u) splits = 32u;
    if (splits > ktiles / 4u) splits = ktiles / 4u;
    if (splits < 1u) splits = 1u;
    const uint32_t per = (ktiles + splits - 1u) / splits;
    *kper = per * 32u;
    return (ktiles + per - 1u) / per;
}

// Tiles of 64 rows where those of 128 would be one on some compute units and two on others (256 to 383: twice as many are
// still resident at once; 10000 x 512 x 784 82 -> 71 us, 4096 x 1000 x 1000 78 -> 68, but 512 tiles of 2000 x 4096 x 4096 359
// -> 390), and for short sums, which are mostly load, split and store (8192 x 16384 x 64 230 -> 200 us)
void launch_gemm32_parts(const PartsGemm32Args &g, uint32_t splits, bool rows64)
{
    const uint32_t cols = (g.N + 127u) / 128u;
    const uint64_t tiles = (g.M + 127ull) / 128u * cols;
    if (rows64 || (splits == 1u && ((tiles >= 256u && tiles < 384u) || g.K <= 128u)))
        sp_gemm32_bf16_parts<1><<<dim3((g.M + 63u) / 64u * cols, splits), 256, 0, g_stream>>>(g);
    else sp_gemm32_bf16_parts<2><<<dim3((g.M + 127u) / 128u * cols, splits), 256, 0, g_stream>>>(g);
}

// soft_out: the layer is a softmax layer whose normalised outputs belong there; returns true if they were written
// (a split-K layer of at most 64 outputs: the reduction does it), false if C holds the logits.  batch: samples of the caller's
// batch, of which M are multiplied here
bool launch_gemm32(const LayerArgs &L, const float *A, float *C, uint32_t M, float *ws, uint64_t ws_floats, float *soft_out, uint32_t batch,
                   bool training = false)
{
    Gemm32Args g{L, A, C, nullptr, M, 0};
    const bool vec = L.K % 4u == 0 && (reinterpret_cast<uintptr_t>(A) & 15u) == 0 && (reinterpret_cast<uintptr_t>(L.w) & 15u) == 0;
    if (!training && gemm32_parts_pay(batch, L.N, L.K)) {
        PartsGemm32Args b{};
        uint32_t parts = gemm32_parts_splits(M, L.N, L.K, &b.kper);
        // A block of rows of a larger batch, which would be cut into many partial sums: tiles of 64 rows, in as few parts as
        // give every compute unit one (10000 samples of 784-512-1000-10 evaluated in blocks of 2560 rows 976 -> 910 us in
        // 128-row tiles of six and four parts / these; 870 in the FP32 kernels, whose sums are further off).
        const uint64_t tiles64 = (M + 63ull) / 64u * ((L.N + 127u) / 128u);
        const bool rows64 = M < batch && parts > 1;
        if (rows64) {
            const uint32_t ktiles = (L.K + 31u) / 32u, fewer = (uint32_t)((255u + tiles64) / tiles64);
            if (fewer < parts) {
                const uint32_t per = (ktiles + fewer - 1u) / fewer;
                b.kper = per * 32u;
                parts = (ktiles + per - 1u) / per;
            }
        }
        if (parts > 1 && (uint64_t)parts * M * L.N > ws_floats) { parts = 1; b.kper = (L.K + 31u) / 32u * 32u; }
        tl_route.name = "sp_gemm32_bf16_parts";
        if (tl_route.dry) return false;
        b.A = A; b.B = reinterpret_cast<const float *>(L.w); b.C = C; b.ws = parts > 1 ? ws : nullptr;
        b.M = M; b.N = L.N; b.K = L.K;
        b.bias = L.bias; b.bscale = L.bscale; b.bias_fmt = L.bias_fmt; b.act = L.act;
        launch_gemm32_parts(b, parts, rows64);
        if (parts > 1 && soft_out && soft_sums_pay(M, L.N)) {
            launch_sum_softmax({ws, parts, parts, M, L.N, L, soft_out, 0, 0});
            return true;
        }
        if (parts > 1) {
            g.ws = ws;
            sp_gemm32_reduce<<<(uint32_t)(((uint64_t)M * L.N + 255) / 256), 256, 0, g_stream>>>(g, parts);
        }
        return false;
    }
    // weights beyond the L2s (4 MB per XCD) and enough 128 x 128 tiles for two per compute unit: the larger tile
    if (vec && M >= 512u && (uint64_t)L.N * L.K * sizeof(float) > (4ull << 20) &&
        (uint64_t)((M + 127u) / 128u) * ((L.N + 127u) / 128u) >= 512u) {
        tl_route.name = "sp_gemm32_f32_big";
        if (tl_route.dry) return false;
        constexpr size_t lds = 2 * 2 * 128 * 36 * sizeof(float);
        static bool once = ((void)hipFuncSetAttribute((const void *)sp_gemm32_f32_big, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), true);
        (void)once;
        sp_gemm32_f32_big<<<((M + 127u) / 128u) * ((L.N + 127u) / 128u), 256, lds, g_stream>>>(g);
        return false;
    }
    uint32_t splits = gemm32_fwd_splits(M, L.N, L.K, &g.kper);
    KSegments seg;
    const uint32_t small = gemm32_small_tile(M, L.N, L.K, vec, &seg);
    if (small) {
        tl_route.name = small == 16u ? "sp_gemm32_small16" : "sp_gemm32_small";
        if (tl_route.dry) return false;
        const bool soft = soft_out && L.N <= small;
        launch_gemm32_small(g, small, seg, soft ? soft_out : nullptr, DeltaTail{});
        return soft;
    }
    if (gemm32_head_takes(M, L.N, L.K, false, &seg)) {
        tl_route.name = "sp_gemm32_head";
        if (tl_route.dry) return false;
        launch_gemm32_head(g, seg, soft_out, DeltaTail{});
        return soft_out != nullptr;
    }
    if (splits > 1 && (uint64_t)splits * M * L.N > ws_floats) { splits = 1; g.kper = (L.K + 31u) / 32u * 32u; }
    if (splits > 1) g.ws = ws;
    tl_route.name = "sp_gemm32_f32";
    if (tl_route.dry) return false;
    if (gemm32_tile_takes(A, L.w, L.K, L.K)) {
        const Tile32Args t{A, reinterpret_cast<const float *>(L.w), C, g.ws, nullptr, L.bias, L.bias_fmt, L.bscale,
                           M, L.N, L.K, L.K, L.K, g.kper, L.act, 1.0f};
        launch_gemm32_tile<T32_LAYER, false, false>(t, splits);
    } else {
        sp_gemm32_f32_any<<<dim3(((M + 63) / 64) * ((L.N + 63) / 64), splits), 256, 0, g_stream>>>(g);
    }
    if (splits > 1 && soft_out && L.N <= 64u) {
        sp_gemm32_reduce_softmax<<<(M + 15u) / 16u, 256, 0, g_stream>>>(g, splits, soft_out);
        return true;
    }
    if (splits > 1 && soft_out && !training && soft_sums_pay(M, L.N)) {     // (training keeps the order of its sums)
        launch_sum_softmax({ws, splits, splits, M, L.N, L, soft_out, 0, 0});
        return true;
    }
    if (splits > 1) sp_gemm32_reduce<<<(uint32_t)(((uint64_t)M * L.N + 255) / 256), 256, 0, g_stream>>>(g, splits);
    return false;
}

// What a forward of n samples needs of a Workspace (the same routing decisions as the launch_* functions)
struct WorkspaceNeed {
    uint64_t act_floats;       // each of the two ping-pong buffers
    uint64_t soft_floats;
    uint64_t plane_bytes;      // digit planes: 4 bytes per element (+ padding of the last chunk) ...
    uint64_t plane_recs;       // ... and one scale (+ four digit sums) per 64 elements
    uint64_t split_floats;
    uint64_t split_least;      // what of it no layer can do without (sp_skinny16, sp_skinny16_kw_head and sp_gemm16 split K as far as there is room)
    uint64_t parts_floats;     // the partial sums that sp_gemm32_bf16_parts would like room for (it runs without them too)
    uint64_t cat_elems;        // split mode of an FP32 net: FP16 elements of the widest three-part layer input
};

// an integer layer with at most 64 outputs streams the activations against an FP16 copy of its codes
bool layer_wants_codes16(const sphip_net *net, const std::vector<uint32_t> &width, uint32_t l /*1-based*/, uint32_t n)
{
    if (net->prec < I8) return false;
    const ThinPlan tp = plan_thin(net->prec, n, width[l], width[l - 1]);
    return tp.use && tp.mode_b;
}

uint32_t cat3_kp(uint32_t K) { return (K + 7u) & ~7u; }

// Split mode of an FP32 net: which layers run as three FP16 products.  Measured against sp_gemm32_f32 on layers of
// 512 to 4096 inputs and outputs, conversion of the input included: even at 1-2 GFLOP per layer, 1.4x at 4 GFLOP,
// 2.6x at 70 GFLOP; layers of a hundred outputs and fewer lose at every batch tried (streaming kernels over a row
// three times as long).  The other layers keep the FP32 kernel; FP32 activations between the layers either way.
bool cat3_layer(uint32_t n, uint32_t N, uint32_t K) { return N >= 128u && 2.0 * (double)n * N * K >= 3e9; }

// In a split-activation forward of a 16-bit or integer net every matrix-core layer writes one set of partial sums per
// activation matrix (halves = 2).  width: the net's padded widths, which it runs with, or those it was made with.
// batch: samples of the caller's batch, by which the arithmetic of FP32 nets is chosen, when n is a part of them (0: n is all).
WorkspaceNeed workspace_need(const sphip_net *net, const std::vector<uint32_t> &width, uint32_t n, uint32_t flags, uint32_t batch = 0)
{
    if (!batch) batch = n;
    WorkspaceNeed w{};
    uint32_t widest = 0;
    for (uint32_t l = 0; l < net->layers; ++l)
        if (width[l] > widest) widest = width[l];
    const Regime reg = pick_regime(net, n, flags);
    const uint32_t halves = (flags & SPHIP_SPLIT_ACTIVATIONS) && reg == R_GEMM16 ? 2u : 1u;
    w.act_floats = (uint64_t)n * widest;
    for (uint32_t l = 1; l < net->layers; ++l)
        if (net->act[l - 1] == A_SOFTMAX && (uint64_t)n * width[l] > w.soft_floats) w.soft_floats = (uint64_t)n * width[l];
    if (n <= 64 && net->prec >= I8) {
        const uint64_t padded = (uint64_t)n * ((uint64_t)widest + 4096u);
        w.plane_bytes = padded * 4u;
        w.plane_recs = padded / 64u + 64u;
    }
    for (uint32_t l = 1; l < net->layers; ++l) {
        const uint32_t N = width[l], K = width[l - 1];
        uint32_t kper = 0;
        uint64_t ws = 0, spare = 0;
        if (reg == R_CAT3 && cat3_layer(batch, N, K)) {
            const uint32_t K3 = 3u * cat3_kp(K);
            if ((uint64_t)n * K3 > w.cat_elems) w.cat_elems = (uint64_t)n * K3;
            const ThinPlan tp = plan_thin(F16, n, N, K3);
            if (tp.use) {
                if (tp.splits > 1) ws = (uint64_t)tp.splits * tp.NC * tp.R;
                if (!tp.kw && !tp.regs) spare = ws;
            } else {
                const uint32_t sp = gemm16_splits(F16, n, N, K3, &kper);
                if (sp > 1) ws = (uint64_t)sp * n * N;
                const uint64_t single = gemm16_single_splits(n, N, K3, &kper);
                if (single > 1 && single * n * N > ws) {
                    spare = single * n * N - ws;
                    ws += spare;
                }
            }
        } else if (net->prec == F32) {
            if (reg == R_GEMV) continue;
            const uint32_t sp = gemm32_fwd_splits(n, N, K, &kper);
            if (sp > 1) ws = (uint64_t)sp * n * N;
            const uint64_t parts = gemm32_parts_pay(batch, N, K) ? gemm32_parts_splits(n, N, K, &kper) : 1u;
            if (parts > 1 && parts * n * N > w.parts_floats) w.parts_floats = parts * n * N;
        } else {
            const ThinPlan tp = plan_thin(net->prec, n, N, K, ~0ull, halves);
            if (tp.use) {
                if (tp.splits > 1 || halves > 1) ws = (uint64_t)tp.splits * halves * tp.NC * tp.R;
                if (!tp.kw && !tp.regs) spare = ws - (halves > 1 ? (uint64_t)halves * tp.NC * tp.R : 0u);
            } else {
                const uint32_t sp = gemm16_splits(net->prec, n, N, K, &kper);
                if (sp > 1 || halves > 1) ws = (uint64_t)sp * halves * n * N;
                const bool aligned = rows_aligned(net->prec, K) && K % 8u == 0;
                const bool words = !aligned && K % 8u == 0 && ((uint64_t)K * fmt_bits(net->prec)) % 32u == 0 && net->prec >= I8;
                if (!aligned && !words) {
                    const uint32_t rs = gemm16_ragged_splits(n, N, K, &kper);
                    if (rs > 1) ws = (uint64_t)rs * halves * n * N;
                } else {
                    const uint64_t single = (uint64_t)gemm16_single_splits(n, N, K, &kper) * halves;
                    if (single > halves && single * n * N > ws) {
                        spare = single * n * N - ws;
                        ws += spare;
                    }
                }
            }
        }
        if (reg == R_GEMM16 && l == 1 && K != net->topo[0] && gemm16_small_layer(n, N, K, halves)) {
            const uint32_t rs = gemm16_ragged_splits(n, N, K, &kper);
            if ((uint64_t)rs * halves * n * N > ws) { ws = (uint64_t)rs * halves * n * N; spare = 0; }
        }
        if (ws > w.split_floats) w.split_floats = ws;
        if (ws - spare > w.split_least) w.split_least = ws - spare;
    }
    return w;
}

void launch_codes16(int prec, const uint8_t *codes, uint16_t *out, uint64_t count)
{
    const uint32_t grid = (uint32_t)((count + 255) / 256);
    if (prec == I8) sp_codes16<I8><<<grid, 256, 0, g_stream>>>(codes, out, count);
    else if (prec == I4) sp_codes16<I4><<<grid, 256, 0, g_stream>>>(codes, out, count);
    else sp_codes16<I2><<<grid, 256, 0, g_stream>>>(codes, out, count);
}

// The three-part FP16 form of an FP32 weight array [N][K] (sp_cat3_w): one small reduction for the shift, one wait,
// one conversion.  The word the reduction leaves its result in sits behind the copy, in the same allocation.
int make_cat3(DevArray &wa, uint32_t N, uint32_t K)
{
    const uint32_t Kp = cat3_kp(K);
    const size_t copy_bytes = (size_t)N * 3u * Kp * sizeof(uint16_t);          // a multiple of 16
    if (!wa.cat3) HCHECK(hipMalloc((void **)&wa.cat3, copy_bytes + 16u));
    uint32_t *word = reinterpret_cast<uint32_t *>(reinterpret_cast<uint8_t *>(wa.cat3) + copy_bytes);
    const float *src = reinterpret_cast<const float *>(wa.base);
    uint32_t top = 0;
    HCHECK(hipMemsetAsync(word, 0, sizeof(uint32_t), g_stream));
    uint64_t blocks = (wa.count + 255) / 256;
    if (blocks > 512) blocks = 512;                       // (every wave ends in one atomic on the same word)
    sp_absmax_f32<<<(uint32_t)blocks, 256, 0, g_stream>>>(src, wa.count, word);
    HCHECK(hipMemcpyAsync(&top, word, sizeof(uint32_t), hipMemcpyDeviceToHost, g_stream));
    HCHECK(hipStreamSynchronize(g_stream));
    wa.cat3_shift = top ? 14 - ((int)(top >> 23) - 127) : 0;       // largest magnitude = 1.m x 2^(e - 127)
    sp_cat3_w<<<(uint32_t)(((uint64_t)N * Kp + 255) / 256), 256, 0, g_stream>>>(src, wa.cat3, N, K, Kp, wa.cat3_shift);
    HCHECK(hipGetLastError());
    wa.cat3_valid = true;
    return 0;
}

// Rows r0 .. r0 + rows of a layer's weights, as uploaded, into its padded array, and zero rows behind the last one
// (sp_pad_rows).  Enqueues only.
int pad_rows(sphip_net *net, uint32_t l, const uint8_t *src, uint32_t r0, uint32_t rows)
{
    const uint32_t N = net->topo[l + 1], K = net->topo[l], Np = net->ptopo[l + 1], Kp = net->ptopo[l];
    const uint64_t row_bytes = fmt_bytes(net->prec, Kp);                        // (a multiple of 16)
    const uint64_t words = row_bytes / 4u * (r0 + rows == N ? Np - r0 : rows);
    const uint32_t grid = (uint32_t)((words + 255u) / 256u);
    uint32_t *out = reinterpret_cast<uint32_t *>(net->PW[l].base + row_bytes * r0);
    switch (fmt_bits(net->prec)) {
    case 16: sp_pad_rows<16><<<grid, 256, 0, g_stream>>>(src, out, rows, K, Kp, words); break;
    case 8:  sp_pad_rows<8><<<grid, 256, 0, g_stream>>>(src, out, rows, K, Kp, words); break;
    case 4:  sp_pad_rows<4><<<grid, 256, 0, g_stream>>>(src, out, rows, K, Kp, words); break;
    default: sp_pad_rows<2><<<grid, 256, 0, g_stream>>>(src, out, rows, K, Kp, words); break;
    }
    HCHECK(hipGetLastError());
    return 0;
}

// A layer's weights to where they lie.  Layers behind a padded one go row by row through pad_stage, four rows at a time or
// a multiple of that: the codes of four rows are whole bytes.
int upload_weights(sphip_net *net, uint32_t l, const uint8_t *codes)
{
    const DevArray &a = net->W[l];
    if (a.base) {
        HCHECK(hipMemcpyAsync(a.base, codes, a.bytes, hipMemcpyHostToDevice, g_stream));
        return net->PW[l].base ? pad_rows(net, l, a.base, 0, net->topo[l + 1]) : 0;
    }
    const uint32_t N = net->topo[l + 1], K = net->topo[l];
    const uint64_t four = fmt_bytes(net->prec, 4ull * K);
    const uint64_t step64 = net->pad_stage_bytes / four * 4u;
    const uint32_t step = step64 < N ? (uint32_t)step64 : N;
    for (uint32_t r0 = 0; r0 < N; r0 += step) {
        const uint32_t rows = N - r0 < step ? N - r0 : step;
        HCHECK(hipMemcpyAsync(net->pad_stage, codes + four * (r0 / 4u), fmt_bytes(net->prec, (uint64_t)rows * K), hipMemcpyHostToDevice, g_stream));
        if (pad_rows(net, l, net->pad_stage, r0, rows)) return 1;
    }
    return 0;
}

// grows the net's own workspace to what n samples, of a batch of `batch` (0: all of it), need
int reserve(sphip_net *net, uint32_t n, bool keep_layers, uint32_t flags = 0, uint32_t batch = 0)
{
    if (!batch) batch = n;
    const WorkspaceNeed need = workspace_need(net, net->ptopo, n, flags, batch);
    if (need.cat_elems > net->cat_cap) {
        if (net->cat_buf) { HCHECK(hipFree(net->cat_buf)); net->cat_buf = nullptr; }
        net->cat_cap = 0;
        HCHECK(hipMalloc((void **)&net->cat_buf, need.cat_elems * sizeof(uint16_t)));
        net->cat_cap = need.cat_elems;
    }
    if (need.cat_elems)
        for (uint32_t l = 1; l < net->layers; ++l)
            if (cat3_layer(batch, net->ptopo[l], net->ptopo[l - 1]) && !net->w(l - 1).cat3_valid && net->W[l - 1].uploaded &&
                make_cat3(net->w(l - 1), net->ptopo[l], net->ptopo[l - 1])) return 1;
    if (need.act_floats > net->cap_elems) {
        for (int i = 0; i < 2; ++i) {
            if (net->buf[i]) { HCHECK(hipFree(net->buf[i])); net->buf[i] = nullptr; }
        }
        net->cap_elems = 0;
        for (int i = 0; i < 2; ++i) HCHECK(hipMalloc(&net->buf[i], need.act_floats * sizeof(float)));
        net->cap_elems = need.act_floats;
    }
    if (need.soft_floats > net->soft_cap) {
        if (net->soft_tmp) { HCHECK(hipFree(net->soft_tmp)); net->soft_tmp = nullptr; }
        net->soft_cap = 0;
        HCHECK(hipMalloc((void **)&net->soft_tmp, need.soft_floats * sizeof(float)));
        net->soft_cap = need.soft_floats;
    }
    if (need.plane_bytes && n > net->aq_cap_n) {
        if (net->aq) { HCHECK(hipFree(net->aq)); HCHECK(hipFree(net->aq_inv)); HCHECK(hipFree(net->aq_dsum)); net->aq = nullptr; }
        net->aq_cap_n = 0;
        HCHECK(hipMalloc((void **)&net->aq, need.plane_bytes));
        HCHECK(hipMalloc((void **)&net->aq_inv, need.plane_recs * sizeof(float)));
        HCHECK(hipMalloc((void **)&net->aq_dsum, need.plane_recs * 4u * sizeof(int)));
        net->aq_cap_n = n;
        net->aq_valid_layer = 0;
    }
    if (keep_layers && !net->layers_buf)
        HCHECK(hipMalloc((void **)&net->layers_buf, net->slots_total * sizeof(float)));
    const uint64_t split_floats = need.parts_floats > need.split_floats ? need.parts_floats : need.split_floats;
    if (split_floats > net->split_cap) {
        if (net->split_ws) { HCHECK(hipFree(net->split_ws)); net->split_ws = nullptr; }
        net->split_cap = 0;
        HCHECK(hipMalloc((void **)&net->split_ws, split_floats * sizeof(float)));
        net->split_cap = split_floats;
    }
    for (uint32_t l = 1; l < net->layers; ++l) {
        DevArray &wa = net->w(l - 1);
        if (layer_wants_codes16(net, net->ptopo, l, n) && !wa.codes16_valid && net->W[l - 1].uploaded) {
            if (!wa.codes16) HCHECK(hipMalloc((void **)&wa.codes16, wa.laid * sizeof(uint16_t)));
            launch_codes16(net->prec, wa.base, wa.codes16, wa.laid);
            HCHECK(hipGetLastError());
            wa.codes16_valid = true;
        }
        net->codes16_ptrs[l - 1] = wa.codes16_valid ? wa.codes16 : nullptr;
    }
    return 0;
}

int grow(float **p, uint64_t *cap, uint64_t need)
{
    if (need <= *cap) return 0;
    if (*p) { HCHECK(hipFree(*p)); *p = nullptr; }
    *cap = 0;
    HCHECK(hipMalloc((void **)p, need * sizeof(float)));
    *cap = need;
    return 0;
}

int check_uploaded(const sphip_net *net)
{
    for (uint32_t l = 0; l + 1 < net->layers; ++l)
        if (!net->W[l].uploaded || !net->B[l].uploaded) return fail_msg("sphip: an array of this net was never uploaded");
    return 0;
}

// Enqueues every kernel of one forward.  d_x, d_y are device pointers.
// only_layer != 0 restricts the launch to the main kernel of that layer.
// keep (n == 1): every layer's output goes to its slot of layers_buf, d_x must be slot 0 and d_y the last slot.
// batch: samples of the caller's batch, of which these are n (0: all of it).
int enqueue_forward(sphip_net *net, const Workspace &wk, const float *d_x, uint32_t n, float *d_y, uint32_t flags,
                    uint32_t only_layer, bool keep = false, const float **logits = nullptr, uint32_t batch = 0)
{
    if (!batch) batch = n;
    // logits: the caller applies the softmax of the last layer; set to where its logits are, nullptr if there is none to apply
    if (logits) *logits = nullptr;
    const Regime reg = pick_regime(net, n, flags);
    // split activations: two FP16 matrices between the layers, whatever else the flags say
    const bool split = (flags & SPHIP_SPLIT_ACTIVATIONS) && reg == R_GEMM16;
    tl_route.halves = split ? 2u : 1u;
    // BF16 weights: FP16 activations against the FP16 copy of the weights unless BF16 activations are asked for
    const bool wide = (split || !(flags & SPHIP_BF16_ACTIVATIONS)) && net->prec == BF16 && reg == R_GEMM16;
    const bool f16t = net->prec != BF16 || wide;  // 16-bit activation type of the matrix-core path
    const uint32_t last = net->layers - 1;

    const void *in = d_x;
    const uint32_t in_w = net->topo[0], in_pw = net->ptopo[0];
    const bool x_fused = reg == R_GEMM16 && in_pw == in_w && gemm16_small_layer(n, net->ptopo[1], in_w, tl_route.halves) &&
                         (reinterpret_cast<uintptr_t>(d_x) & 15u) == 0;
    const bool raw = raw_rows(net->prec, in_w, net->ptopo[1], n);
    if (reg == R_GEMV && in_pw != in_w && !raw && only_layer <= 1u) {
        const uint64_t quads = (uint64_t)n * (in_pw / 4u);
        sp_pad_input<0><<<(uint32_t)((quads + 255u) / 256u), 256, 0, g_stream>>>(d_x, wk.buf[1], n, in_w, in_pw);
        in = wk.buf[1];
    } else if (x_fused) {
        // (the first layer's kernel rounds, or splits, the FP32 input itself)
    } else if (in_pw != in_w && reg == R_GEMM16 && !only_layer) {
        // rows of a padded input, converted on the way
        const uint64_t quads = (uint64_t)n * ((in_pw + 3u) / 4u);
        const uint32_t grid = (uint32_t)((quads + 255u) / 256u);
        if (split) sp_pad_input<3><<<grid, 256, 0, g_stream>>>(d_x, wk.buf[1], n, in_w, in_pw);
        else if (f16t) sp_pad_input<2><<<grid, 256, 0, g_stream>>>(d_x, wk.buf[1], n, in_w, in_pw);
        else sp_pad_input<1><<<grid, 256, 0, g_stream>>>(d_x, wk.buf[1], n, in_w, in_pw);
        in = wk.buf[1];
    } else if (split && !only_layer) {
        const uint64_t cnt = (uint64_t)n * net->topo[0];
        sp_cvt16_split<<<(uint32_t)((cnt / 4 + 255) / 256 + 1), 256, 0, g_stream>>>(d_x, (uint16_t *)wk.buf[1], cnt);
        in = wk.buf[1];
    } else if (reg == R_GEMM16 && !only_layer) {
        const uint64_t cnt = (uint64_t)n * net->topo[0];
        const uint32_t grid = (uint32_t)((cnt / 4 + 255) / 256 + 1);
        if (f16t) sp_cvt16<true><<<grid, 256, 0, g_stream>>>(d_x, (uint16_t *)wk.buf[1], cnt);
        else sp_cvt16<false><<<grid, 256, 0, g_stream>>>(d_x, (uint16_t *)wk.buf[1], cnt);
        in = wk.buf[1];
    } else if (reg == R_GEMM16) {
        in = wk.buf[1];
    }

    for (uint32_t l = 1; l <= last; ++l) {
        const DevArray &wa = net->w(l - 1);
        LayerArgs L = make_layer_args(net, l, l == 1 && reg == R_GEMV && raw);
        if (wide) {
            L.w = reinterpret_cast<const uint8_t *>(wa.wide16);
            L.wscale = ldexpf(L.wscale, -wa.wide_shift);
        }
        const bool cat3 = reg == R_CAT3 && cat3_layer(batch, L.N, L.K);
        if (cat3) {
            if (!wa.cat3_valid) return fail_msg("sphip: the FP16 parts of this net's FP32 weights were not made (split mode)");
            L.w = reinterpret_cast<const uint8_t *>(wa.cat3);
            L.wscale = ldexpf(L.wscale, -wa.cat3_shift);
            L.K = 3u * cat3_kp(net->ptopo[l - 1]);
        }
        const bool softmax = net->act[l - 1] == A_SOFTMAX;
        const bool is_last = l == last;
        void *dst = is_last ? (void *)d_y : keep ? (void *)(net->layers_buf + net->slot_off[l]) : wk.buf[(l + 1) & 1];
        // logits of a softmax layer go to FP32 scratch first
        void *main_out = softmax ? (void *)wk.soft_tmp : dst;
        const int out_f32 = (reg != R_GEMM16) || is_last || softmax;
        const bool run = !only_layer || only_layer == l;
        bool soft_done = false;                 // the layer's own kernel wrote the softmax
        if (run) {
            if (reg == R_GEMV) launch_gemv(net->prec, wk, L, (const float *)in, (float *)main_out, n,
                                          only_layer != 0 && net->aq_valid_layer == l && net->aq_valid_n == n, net->ptopo[l - 1] != net->topo[l - 1]);
            if (reg == R_GEMV) { net->aq_valid_layer = l; net->aq_valid_n = n; }
            else if ((reg == R_GEMM32 || (reg == R_CAT3 && !cat3)) && f32_thin_vector(L, n))
                launch_gemv(net->prec, wk, L, (const float *)in, (float *)main_out, n, false);
            else if (reg == R_GEMM32 || (reg == R_CAT3 && !cat3))
                soft_done = launch_gemm32(L, (const float *)in, (float *)main_out, n, wk.split_ws, wk.split_cap,
                                          softmax && !only_layer ? (float *)dst : nullptr, batch);
            else if (cat3) {
                // (timing one layer includes the conversion of its input)
                const uint32_t K = net->ptopo[l - 1], Kp = cat3_kp(K);
                const int vec = K % 4u == 0 && (reinterpret_cast<uintptr_t>(in) & 15u) == 0;
                sp_cat3_x<<<(uint32_t)(((uint64_t)n * (Kp / 8u) + 255) / 256), 256, 0, g_stream>>>((const float *)in, wk.cat, n, K, Kp, vec);
                ThinCtx ctx{};
                ctx.w16 = wa.cat3;
                ctx.ws = wk.split_ws;
                ctx.ws_floats = wk.split_cap;
                if (softmax && !only_layer) {
                    ctx.soft_out = dst;
                    ctx.soft_kind = 0;
                    ctx.soft_done = &soft_done;
                }
                launch_gemm16((int)F16, L, wk.cat, main_out, n, 1, ctx);
            } else {
                ThinCtx ctx{};
                if (wide) ctx.w16 = wa.wide16;
                else if (net->prec == F16 || net->prec == BF16) ctx.w16 = reinterpret_cast<const uint16_t *>(wa.base);
                else ctx.w16 = wk.codes16[l - 1];
                ctx.ws = wk.split_ws;
                ctx.ws_floats = wk.split_cap;
                ctx.x_f32 = x_fused && l == 1;
                ctx.padded_in = l == 1 && in_pw != in_w;
                if (softmax && !only_layer) {
                    ctx.soft_out = dst;
                    ctx.soft_kind = !is_last ? (split ? 3 : f16t ? 2 : 1) : 0;
                    ctx.soft_done = &soft_done;
                }
                launch_gemm16(wide ? (int)F16 : net->prec, L, (const uint16_t *)in, main_out, n, out_f32, ctx);
            }
        }
        if (softmax && !only_layer && !soft_done && is_last && logits) {
            *logits = wk.soft_tmp;
        } else if (softmax && !only_layer && !soft_done) {
            const int kind = (reg == R_GEMM16 && !is_last) ? (split ? 3 : f16t ? 2 : 1) : 0;
            launch_softmax(wk.soft_tmp, dst, kind, n, net->topo[l]);
        }
        in = dst;
    }
    tl_route.halves = 1;
    HCHECK(hipGetLastError());
    return 0;
}

// Rows per pass over a large batch.  The activations between two layers are written once and read once; when the
// two buffers of a whole batch exceed the memory-side cache (256 MB), every layer boundary goes through HBM.  Running
// all layers over one block of rows after the other keeps the boundaries in that cache (the weights are re-read per
// block, from HBM or from the same cache).  Rows are independent (Training.c:313-345 computes them by one sgemm, but
// no row's result depends on another's), so the outputs are those of the whole batch up to the choice of K splits.
// Blocks are equal, a multiple of 256 rows, and as large as fits 64 MiB per 16-bit activation buffer.  Batches of up
// to 128 MiB per buffer stay whole: measured on one box, 8192 samples of the 8192-wide BF16 net 7.72 ms whole against
// 7.82 ms in two blocks (the weights, 128 MiB per layer, are then read twice) and of the 8192-wide INT2 net 2.75
// against 2.74 ms; 16384 samples of the latter 5.83 against 5.45 ms, 65536 samples 24.0 against 21.6 ms.
uint32_t batch_block_rows(const sphip_net *net, uint32_t n, uint32_t flags)
{
    if ((flags & SPHIP_WHOLE_BATCH) || pick_regime(net, n, flags) != R_GEMM16) return n;
    const uint64_t per_row = (uint64_t)net->max_width * 2u;
    if ((uint64_t)n * per_row <= (128ull << 20)) return n;
    uint64_t rows = (64ull << 20) / per_row / 256u * 256u;
    if (rows < 1024u) rows = 1024u;
    if (rows >= n) return n;
    const uint64_t blocks = (n + rows - 1) / rows;
    rows = ((n + blocks - 1) / blocks + 255u) / 256u * 256u;
    return (uint32_t)rows;
}

// reserve() for a batch that may run in blocks of rows: the workspace of a full block and of the last, smaller one
int reserve_batch(sphip_net *net, uint32_t n, uint32_t flags)
{
    const uint32_t rows = batch_block_rows(net, n, flags);
    if (reserve(net, rows, false, flags)) return 1;
    if (rows < n && n % rows != 0 && reserve(net, n % rows, false, flags)) return 1;
    return 0;
}

// enqueue_forward over the blocks of rows of batch_block_rows(); the caller has called reserve_batch()
int enqueue_forward_batch(sphip_net *net, const float *d_x, uint32_t n, float *d_y, uint32_t flags, uint32_t only_layer)
{
    const uint32_t rows = batch_block_rows(net, n, flags);
    const uint32_t in_w = net->topo[0], out_w = net->topo[net->layers - 1];
    for (uint32_t r0 = 0; r0 < n; r0 += rows) {
        const uint32_t m = n - r0 < rows ? n - r0 : rows;
        if (enqueue_forward(net, net->workspace(), d_x + (size_t)r0 * in_w, m, d_y + (size_t)r0 * out_w, flags, only_layer)) return 1;
    }
    return 0;
}

}  // namespace

extern "C" {

int sphip_device_count(void)
{
    int cnt = 0;
    if (hipGetDeviceCount(&cnt) != hipSuccess) return 0;
    return cnt;
}

const char *sphip_last_error_string(void) { return g_err; }

int sphip_create(const sphip_desc *desc, sphip_net **out)
{
    if (!desc || !out || desc->layers < 2 || !desc->topology || !desc->act) return fail_msg("sphip_create: invalid descriptor");
    if (desc->precision >= NFMT) return fail_msg("sphip_create: invalid precision");
    for (uint32_t l = 0; l < desc->layers; ++l)
        if (desc->topology[l] == 0) return fail_msg("sphip_create: empty layer");
    for (uint32_t l = 0; l + 1 < desc->layers; ++l)
        if (desc->act[l] >= A_COUNT) return fail_msg("sphip_create: invalid activation");
    if (ensure_stream()) return 1;
    sphip_net *net = new (std::nothrow) sphip_net;
    if (!net) return fail_msg("sphip_create: out of host memory");
    net->layers = desc->layers;
    net->topo.assign(desc->topology, desc->topology + desc->layers);
    net->act.assign(desc->act, desc->act + desc->layers - 1);
    net->prec = desc->precision;
    net->W.resize(desc->layers - 1);
    net->B.resize(desc->layers - 1);
    net->PW.resize(desc->layers - 1);
    net->codes16_ptrs.assign(desc->layers - 1, nullptr);
    for (uint32_t l = 0; l < desc->layers; ++l) {
        const bool hidden_softmax = l && net->act[l - 1] == A_SOFTMAX;
        net->ptopo.push_back(l + 1 == desc->layers || hidden_softmax ? net->topo[l] : padded_width(net->prec, net->topo[l], net->topo[l + 1], l > 0));
        if (net->ptopo[l] > net->max_width) net->max_width = net->ptopo[l];
        net->total_neurons += net->topo[l];
        net->slot_off.push_back((uint32_t)net->slots_total);
        net->slots_total += ((uint64_t)net->ptopo[l] + 3u) & ~3ull;
    }
    // All arrays in one allocation, each at a multiple of 256 bytes with 16 bytes of slack: vector loads of the last chunk
    // never leave it.  (A hipMalloc takes 10 to 100 us.)
    size_t at = 0;
    std::vector<DevArray *> placed;
    auto place = [&](DevArray &a, uint64_t laid) {
        a.laid = laid;
        a.base = reinterpret_cast<uint8_t *>(at);
        at += (fmt_bytes(net->prec, laid) + 16u + 255u) & ~(size_t)255u;
        placed.push_back(&a);
    };
    bool padded = false;
    for (uint32_t l = 0; l + 1 < desc->layers; ++l) {
        const uint64_t K = net->topo[l], N = net->topo[l + 1], Kp = net->ptopo[l], Np = net->ptopo[l + 1];
        DevArray &w = net->W[l], &b = net->B[l];
        w.count = K * N;
        w.bytes = fmt_bytes(net->prec, w.count);
        b.count = N;
        b.bytes = fmt_bytes(net->prec, b.count);
        if (Kp == K || l == 0) place(w, K * Np);
        if (Kp != K) place(net->PW[l], Kp * Np);
        place(b, Np);
        padded |= Np != N || Kp != K;
        if (!w.base && l) {
            // at most 4 MiB, at least four rows
            const size_t four = fmt_bytes(net->prec, 4ull * K);
            size_t stage = w.bytes + four < (4u << 20) ? w.bytes + four : (4u << 20);
            if (stage < four) stage = four;
            if (stage > net->pad_stage_bytes) net->pad_stage_bytes = stage;
        }
    }
    if (hipMalloc((void **)&net->arrays, at + net->pad_stage_bytes) != hipSuccess) {
        for (DevArray *a : placed) a->base = nullptr;
        net->arrays = nullptr;
        sphip_destroy(net);
        return fail_msg("sphip_create: device allocation failed");
    }
    for (DevArray *a : placed) a->base = net->arrays + reinterpret_cast<size_t>(a->base);
    net->pad_stage = net->arrays + at;
    if (padded)                                             // the zeros around the arrays that are uploaded
        sp_fill0<<<(uint32_t)((at / 4u + 255u) / 256u), 256, 0, g_stream>>>(reinterpret_cast<float *>(net->arrays), at / 4u);
    *out = net;
    return 0;
}

void sphip_destroy(sphip_net *net)
{
    if (!net) return;
    if (g_stream) (void)hipStreamSynchronize(g_stream);
    train_free(net);
    for (auto *arrays : {&net->W, &net->PW, &net->B})
        for (auto &a : *arrays) {
            if (a.codes16) (void)hipFree(a.codes16);
            if (a.wide16) (void)hipFree(a.wide16);
            if (a.cat3) (void)hipFree(a.cat3);
        }
    if (net->arrays) (void)hipFree(net->arrays);
    if (net->split_ws) (void)hipFree(net->split_ws);
    if (net->cat_buf) (void)hipFree(net->cat_buf);
    if (net->eval_buf) (void)hipFree(net->eval_buf);
    for (int i = 0; i < 2; ++i) if (net->buf[i]) (void)hipFree(net->buf[i]);
    if (net->soft_tmp) (void)hipFree(net->soft_tmp);
    if (net->aq) (void)hipFree(net->aq);
    if (net->aq_inv) (void)hipFree(net->aq_inv);
    if (net->aq_dsum) (void)hipFree(net->aq_dsum);
    if (net->layers_buf) (void)hipFree(net->layers_buf);
    if (net->pin_in) (void)hipHostFree(net->pin_in);
    if (net->pin_out) (void)hipHostFree(net->pin_out);
    if (net->pin_flag) (void)hipHostFree(net->pin_flag);
    if (net->stage_x) (void)hipFree(net->stage_x);
    if (net->stage_y) (void)hipFree(net->stage_y);
    delete net;
}

// A BF16 weight array's FP16 copy for the matrix-core path with FP16 activations: the weights times the power of
// two that brings the array's largest magnitude into [2^14, 2^15).  One small reduction, one wait, one conversion.
// The word the reduction leaves its result in sits behind the copy, in the same allocation.
int make_wide(DevArray &wa)
{
    const size_t copy_bytes = (wa.laid * sizeof(uint16_t) + 15u) & ~(size_t)15u;
    if (!wa.wide16) HCHECK(hipMalloc((void **)&wa.wide16, copy_bytes + 16u));
    uint32_t *word = reinterpret_cast<uint32_t *>(reinterpret_cast<uint8_t *>(wa.wide16) + copy_bytes);
    const uint16_t *src = reinterpret_cast<const uint16_t *>(wa.base);
    uint32_t top = 0;
    HCHECK(hipMemsetAsync(word, 0, sizeof(uint32_t), g_stream));
    uint64_t blocks = (wa.laid + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    sp_absmax_bf16<<<(uint32_t)blocks, 256, 0, g_stream>>>(src, wa.laid, word);
    HCHECK(hipMemcpyAsync(&top, word, sizeof(uint32_t), hipMemcpyDeviceToHost, g_stream));
    HCHECK(hipStreamSynchronize(g_stream));
    wa.wide_shift = top ? 14 - ((int)(top >> 7) - 127) : 0;       // largest magnitude = 1.m x 2^(e - 127)
    sp_bf16_to_f16<<<(uint32_t)((wa.laid + 255) / 256), 256, 0, g_stream>>>(src, wa.wide16, wa.laid, wa.wide_shift);
    HCHECK(hipGetLastError());
    HCHECK(hipStreamSynchronize(g_stream));
    wa.wide16_valid = true;
    return 0;
}

int sphip_upload_array(sphip_net *net, uint32_t l, int which, const void *codes, size_t bytes, float max_val)
{
    if (!net || l + 1 >= net->layers || (which != 0 && which != 1) || !codes) return fail_msg("sphip_upload_array: invalid argument");
    DevArray &a = which == 0 ? net->W[l] : net->B[l];
    if (bytes != a.bytes) return fail_msg("sphip_upload_array: byte count does not match the array's serialized size");
    if (which == 1) HCHECK(hipMemcpyAsync(a.base, codes, bytes, hipMemcpyHostToDevice, g_stream));
    else if (upload_weights(net, l, static_cast<const uint8_t *>(codes))) return 1;
    HCHECK(hipStreamSynchronize(g_stream));
    a.max_val = max_val;
    a.uploaded = true;
    for (DevArray *copies : {&a, which == 0 ? &net->PW[l] : &a}) copies->codes16_valid = copies->wide16_valid = copies->cat3_valid = false;
    if (which == 0 && net->prec == BF16 && make_wide(net->w(l))) return 1;
    return 0;
}

int sphip_clone(const sphip_net *src, sphip_net **out)
{
    if (!src || !out) return fail_msg("sphip_clone: invalid argument");
    sphip_desc d{src->layers, src->topo.data(), src->act.data(), (uint8_t)src->prec};
    sphip_net *net = nullptr;
    if (sphip_create(&d, &net)) return 1;
    hipError_t e = hipSuccess;
    for (uint32_t l = 0; l + 1 < src->layers && e == hipSuccess; ++l) {
        // (array by array: a profile's copy of known size is the largest one's)
        for (int which = 0; which < 3; ++which) {
            const DevArray &s = which == 0 ? src->W[l] : which == 1 ? src->B[l] : src->PW[l];
            DevArray &t = which == 0 ? net->W[l] : which == 1 ? net->B[l] : net->PW[l];
            if (s.base && e == hipSuccess) e = hipMemcpyAsync(t.base, s.base, fmt_bytes(src->prec, s.laid), hipMemcpyDeviceToDevice, g_stream);
            t.max_val = s.max_val;
            t.uploaded = s.uploaded;
        }
        const DevArray &s = src->w(l);
        DevArray &t = net->w(l);
        if (!s.wide16_valid) continue;
        e = hipMalloc((void **)&t.wide16, ((s.laid * sizeof(uint16_t) + 15u) & ~(size_t)15u) + 16u);
        if (e == hipSuccess) e = hipMemcpyAsync(t.wide16, s.wide16, s.laid * sizeof(uint16_t), hipMemcpyDeviceToDevice, g_stream);
        t.wide_shift = s.wide_shift;
        t.wide16_valid = e == hipSuccess;
    }
    if (e != hipSuccess) { sphip_destroy(net); return fail_hip("sphip_clone copy", e); }
    HCHECK(hipStreamSynchronize(g_stream));
    *out = net;
    return 0;
}

// Waits until everything enqueued so far has finished, for calls whose results are a few values in pinned host
// memory: a last one-wave launch stores the call's sequence number into a pinned word and the host polls it (the
// runtime's own wait costs several microseconds after the last kernel has ended).  Bounded: after about 50 ms
// without the number the stream is waited for in the ordinary way, which also reports a failed kernel.
static int next_signal(sphip_net *net, uint32_t *seq)
{
    if (!net->pin_flag) {
        HCHECK(hipHostMalloc((void **)&net->pin_flag, 64, hipHostMallocDefault));
        *net->pin_flag = 0;
    }
    *seq = ++net->flag_seq ? net->flag_seq : ++net->flag_seq;     // never 0
    return 0;
}

static int wait_for_signal(sphip_net *net, uint32_t seq)
{
    HCHECK(hipGetLastError());
    const volatile uint32_t *flag = net->pin_flag;
    const auto t0 = std::chrono::steady_clock::now();
    for (uint32_t spin = 1;; ++spin) {
        if (__atomic_load_n(flag, __ATOMIC_ACQUIRE) == seq) return 0;
        __builtin_ia32_pause();
        if ((spin & 0xFFFu) == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(50)) break;
    }
    HCHECK(hipStreamSynchronize(g_stream));
    return 0;
}

static int wait_for_small_results(sphip_net *net)
{
    uint32_t seq = 0;
    if (next_signal(net, &seq)) return 1;
    sp_signal_host<<<1, 64, 0, g_stream>>>(net->pin_flag, seq);
    return wait_for_signal(net, seq);
}

// Small host inputs travel through a pinned staging buffer and a copy kernel; small outputs are
// written by the last layer's kernel straight into pinned memory (scattered stores over PCIe do
// not pay beyond a few thousand values), and the call ends with one stream synchronisation.
static const uint64_t kSmallIn = 256u * 1024u, kSmallOut = 4096u;

static int grow_pinned(float **p, uint64_t *cap, uint64_t need)
{
    if (need <= *cap) return 0;
    if (*p) { HCHECK(hipHostFree(*p)); *p = nullptr; }
    *cap = 0;
    HCHECK(hipHostMalloc((void **)p, need * sizeof(float), hipHostMallocDefault));
    *cap = need;
    return 0;
}

}  // extern "C"
#include "hip_transfer.inl"
extern "C" {

// Rows per block when a batch comes from the host and its layers run over the rows that have landed while the others are
// under way, 0 if they wait for all of them.  Only where the layers are the shorter part by far, so that running them in
// smaller blocks costs nothing: per value of a sample the bus takes 0.085 ns, a multiply-add of FP32 layers at 100 TFLOP/s
// 0.00002 ns; the line lies at half of that.  A block is what 8 MB hold, in whole tiles of 256 rows, and 2048 at
// least (10000 samples of 784-512-1000-10 FP32 from the host 955 -> 865 us, 20000 1780 -> 1575; 20000 of 784-128-10 1570
// -> 1455); a rest of fewer than kLastRows joins the block before it, so that no few rows take a path for few rows.
static const uint32_t kLastRows = 512;
static const size_t kLandedBytes = 8u << 20;
static uint32_t landing_rows(const sphip_net *net, const float *x, uint32_t n, uint32_t flags)
{
    const uint32_t in_w = net->topo[0];
    if ((flags & SPHIP_WHOLE_BATCH) || (uint64_t)n * in_w * sizeof(float) < 2u * kLandedBytes || host_registered(x)) return 0;
    if (pick_regime(net, n, flags) == R_GEMV || batch_block_rows(net, n, flags) < n) return 0;
    uint64_t macs = 0;
    for (uint32_t l = 1; l < net->layers; ++l) macs += (uint64_t)net->topo[l - 1] * net->topo[l];
    if (macs > 2000ull * in_w) return 0;
    uint32_t rows = (uint32_t)(kLandedBytes / sizeof(float) / in_w / 256u * 256u);
    if (rows < 2048u) rows = 2048u;
    return rows + kLastRows <= n ? rows : 0;
}

// x from the host to net->stage_x and through all layers into d_y
static int enqueue_forward_from_host(sphip_net *net, const float *x, uint32_t n, float *d_y, uint32_t flags)
{
    const uint32_t rows = landing_rows(net, x, n, flags), in_w = net->topo[0], out_w = net->topo[net->layers - 1];
    const size_t row_bytes = (size_t)in_w * sizeof(float);
    if (!rows) {
        if (upload_from_host(net->stage_x, x, n * row_bytes)) return 1;
        return enqueue_forward_batch(net, net->stage_x, n, d_y, flags, 0);
    }
    const uint32_t last = (n - kLastRows) % rows + kLastRows;
    if (reserve(net, rows, false, flags, n) || reserve(net, last, false, flags, n)) return 1;
    uint32_t r0 = 0;
    return upload_from_host(net->stage_x, x, n * row_bytes, [&](size_t upto) {
        while (r0 < n) {
            const uint32_t m = n - r0 < rows + kLastRows ? n - r0 : rows;
            if ((r0 + m) * row_bytes > upto) break;
            if (enqueue_forward(net, net->workspace(), net->stage_x + (size_t)r0 * in_w, m, d_y + (size_t)r0 * out_w, flags, 0, false, nullptr, n))
                return 1;
            r0 += m;
        }
        return 0;
    });
}

int sphip_forward(sphip_net *net, const float *x, uint32_t n, float *y, uint32_t flags)
{
    if (!net || !x || !y || n == 0) return fail_msg("sphip_forward: invalid argument");
    if (check_uploaded(net)) return 1;
    const uint32_t fwd_flags = flags & (SPHIP_FORCE_GEMM | SPHIP_FORCE_GEMV | SPHIP_BF16_ACTIVATIONS | SPHIP_WHOLE_BATCH | SPHIP_SPLIT_ACTIVATIONS);
    if (reserve_batch(net, n, fwd_flags)) return 1;
    const uint64_t in_cnt = (uint64_t)n * net->topo[0], out_cnt = (uint64_t)n * net->topo[net->layers - 1];
    const float *d_x = x;
    float *d_y = y;
    bool y_pinned = false, x_large = false;
    if (!(flags & SPHIP_X_ON_DEVICE)) {
        if (grow(&net->stage_x, &net->stage_x_cap, in_cnt)) return 1;
        if (in_cnt <= kSmallIn) {
            if (grow_pinned(&net->pin_in, &net->pin_in_cap, in_cnt)) return 1;
            memcpy(net->pin_in, x, in_cnt * sizeof(float));
            sp_copy32<<<(uint32_t)((in_cnt + 255) / 256), 256, 0, g_stream>>>(net->pin_in, net->stage_x, in_cnt);
        } else {
            x_large = true;
        }
        d_x = net->stage_x;
    }
    if (!(flags & SPHIP_Y_ON_DEVICE)) {
        if (out_cnt <= kSmallOut) {
            if (grow_pinned(&net->pin_out, &net->pin_out_cap, out_cnt)) return 1;
            d_y = net->pin_out;
            y_pinned = true;
        } else {
            if (grow(&net->stage_y, &net->stage_y_cap, out_cnt)) return 1;
            d_y = net->stage_y;
        }
    }
    if (x_large ? enqueue_forward_from_host(net, x, n, d_y, fwd_flags) : enqueue_forward_batch(net, d_x, n, d_y, fwd_flags, 0)) return 1;
    if (!(flags & SPHIP_Y_ON_DEVICE)) {
        if (y_pinned) {
            if (wait_for_small_results(net)) return 1;
            memcpy(y, net->pin_out, out_cnt * sizeof(float));
        } else {
            if (download_to_host(y, d_y, out_cnt * sizeof(float))) return 1;
        }
    }
    return 0;
}

int sphip_forward_noalloc(sphip_net *net, const float *d_x, uint32_t n, float *d_y, uint32_t flags)
{
    if (!net || !d_x || !d_y || n == 0) return fail_msg("sphip_forward_noalloc: invalid argument");
    if (check_uploaded(net)) return 1;
    if (!g_stream) return fail_msg("sphip_forward_noalloc: library not initialised");    // sphip_create did it
    constexpr uint32_t kMaxLayers = 64;
    if (net->layers > kMaxLayers) return fail_msg("sphip_forward_noalloc: more than 64 layers");
    unsigned char *base = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_init_mutex);
        if (scratch_lookup(&base)) return 1;
    }
    // an integer layer with few outputs reads an FP16 copy of its codes: the net's own if an earlier call made one,
    // else one made here, in the scratch array, on every call
    // (only the matrix-core regime reads them: a forced vector forward or one of up to four samples never does)
    const uint32_t fwd_flags = flags & (SPHIP_FORCE_GEMM | SPHIP_FORCE_GEMV | SPHIP_BF16_ACTIVATIONS | SPHIP_SPLIT_ACTIVATIONS);
    const bool reads_codes = pick_regime(net, n, fwd_flags) == R_GEMM16;
    // every piece of the workspace lies at a multiple of 256 bytes
    auto room = [](uint64_t bytes) { return (size_t)((bytes + 255u) & ~(uint64_t)255u); };
    auto pieces = [&](const WorkspaceNeed &w) {
        return 2u * room(w.act_floats * sizeof(float)) + room(w.soft_floats * sizeof(float)) + room(w.plane_bytes) +
               (w.plane_bytes ? room(w.plane_recs * sizeof(float)) + room(w.plane_recs * 4u * sizeof(int)) : 0u) +
               room(w.split_floats * sizeof(float)) + room(w.cat_elems * sizeof(uint16_t));
    };
    auto least = [](WorkspaceNeed w) { w.split_floats = w.split_least; return w; };
    auto all = [&](const std::vector<uint32_t> &width, const WorkspaceNeed &w) {
        size_t bytes = pieces(w);
        for (uint32_t l = 1; l < net->layers && reads_codes; ++l)
            if (layer_wants_codes16(net, width, l, n) && !net->w(l - 1).codes16_valid)
                bytes += room((uint64_t)width[l - 1] * width[l] * sizeof(uint16_t));
        return bytes;
    };
    // A batch that fits at the widths of the caller's net is accepted, whatever the padding needs.
    const WorkspaceNeed plain = workspace_need(net, net->topo, n, flags);
    if (plain.cat_elems)
        for (uint32_t l = 1; l < net->layers; ++l)
            if (cat3_layer(n, net->ptopo[l], net->ptopo[l - 1]) && !net->w(l - 1).cat3_valid)
                return fail_msg("sphip_forward_noalloc: the split mode of an FP32 net needs FP16 parts of its weights, which the first sphip_forward in that mode makes");
    uint32_t rows = n;
    WorkspaceNeed need = workspace_need(net, net->ptopo, rows, flags);
    const size_t known = all(net->topo, least(plain));
    if (known > kScratchBytes && all(net->ptopo, least(need)) > kScratchBytes) {
        snprintf(g_err, sizeof g_err, "sphip_forward_noalloc: %u samples of this net need %zu bytes of workspace, the fixed scratch array holds %zu",
                 n, known, kScratchBytes);
        return 1;
    }
    // Where the padded widths do need more, the batch runs in the fewest equal blocks of rows that fit, and without the
    // copies of codes that do not (the tile kernels read the codes themselves).
    for (uint32_t blocks = 2; pieces(least(need)) > kScratchRoom && rows > 1u; ++blocks) {
        rows = (n + blocks - 1u) / blocks;
        if (rows > 4u) rows = (rows + 3u) & ~3u;             // the next block's rows start as aligned as the first one's
        need = workspace_need(net, net->ptopo, rows, flags);
    }
    // Partial sums of sp_skinny16, sp_skinny16_kw_head and sp_gemm16 take what the rest leaves.
    const size_t total = all(net->ptopo, need);
    if (total > kScratchRoom) {
        const uint64_t over = (total - kScratchRoom + 255u) / 256u * (256u / sizeof(float));
        need.split_floats = need.split_floats > need.split_least + over ? need.split_floats - over : need.split_least;
    }
    if (pieces(need) > kScratchRoom) return fail_msg("sphip_forward_noalloc: one row of this net does not fit the fixed scratch array");
    size_t used = 0;
    auto take = [&](uint64_t bytes) -> unsigned char * {
        unsigned char *p = base + used;
        used += room(bytes);
        return p;
    };
    uint16_t *codes[kMaxLayers] = {};
    Workspace wk{};
    wk.buf[0] = take(need.act_floats * sizeof(float));
    wk.buf[1] = take(need.act_floats * sizeof(float));
    wk.soft_tmp = reinterpret_cast<float *>(take(need.soft_floats * sizeof(float)));
    if (need.plane_bytes) {
        wk.aq = take(need.plane_bytes);
        wk.aq_inv = reinterpret_cast<float *>(take(need.plane_recs * sizeof(float)));
        wk.aq_dsum = reinterpret_cast<int *>(take(need.plane_recs * 4u * sizeof(int)));
    }
    wk.split_ws = reinterpret_cast<float *>(take(need.split_floats * sizeof(float)));
    wk.split_cap = need.split_floats;
    if (need.cat_elems) wk.cat = reinterpret_cast<uint16_t *>(take(need.cat_elems * sizeof(uint16_t)));
    for (uint32_t l = 1; l < net->layers; ++l) {
        if (!reads_codes || !layer_wants_codes16(net, net->ptopo, l, rows)) continue;
        const DevArray &wa = net->w(l - 1);
        if (wa.codes16_valid) { codes[l - 1] = wa.codes16; continue; }
        if (used + room(wa.laid * sizeof(uint16_t)) > kScratchRoom) continue;
        codes[l - 1] = reinterpret_cast<uint16_t *>(take(wa.laid * sizeof(uint16_t)));
        launch_codes16(net->prec, wa.base, codes[l - 1], wa.laid);
    }
    wk.codes16 = codes;
    if (need.parts_floats > need.split_floats && used + need.parts_floats * sizeof(float) <= kScratchBytes) {
        wk.split_ws = reinterpret_cast<float *>(take(need.parts_floats * sizeof(float)));
        wk.split_cap = need.parts_floats;
    }
    // the integer GEMV's quantise launch is never skipped here (that shortcut belongs to the layer timer)
    net->aq_valid_layer = 0;
    const uint32_t in_w = net->topo[0], out_w = net->topo[net->layers - 1];
    for (uint32_t r0 = 0; r0 < n; r0 += rows)
        if (enqueue_forward(net, wk, d_x + (size_t)r0 * in_w, n - r0 < rows ? n - r0 : rows, d_y + (size_t)r0 * out_w, fwd_flags, 0)) return 1;
    return 0;
}

int sphip_forward_layers(sphip_net *net, const float *x, float *host_neurons)
{
    if (!net || !x || !host_neurons) return fail_msg("sphip_forward_layers: invalid argument");
    if (check_uploaded(net)) return 1;
    if (reserve(net, 1, true)) return 1;
    const uint32_t last = net->layers - 1;
    if (grow_pinned(&net->pin_in, &net->pin_in_cap, net->topo[0])) return 1;
    if (grow_pinned(&net->pin_out, &net->pin_out_cap, net->total_neurons)) return 1;
    memcpy(net->pin_in, x, (size_t)net->topo[0] * sizeof(float));
    sp_copy32<<<(net->topo[0] + 255) / 256, 256, 0, g_stream>>>(net->pin_in, net->layers_buf, net->topo[0]);
    const bool one_launch = net->layers <= 16u && net->total_neurons <= kGatherMost;
    // (a softmax of more than 1024 outputs wants more than the gathering launch's last wave)
    const float *logits = nullptr;
    if (enqueue_forward(net, net->workspace(), net->layers_buf, 1, net->layers_buf + net->slot_off[last], 0, 0, true,
                        one_launch && net->topo[last] <= 1024u ? &logits : nullptr)) return 1;
    // all slots, densely packed, straight into pinned memory
    uint32_t dense = 0;
    for (uint32_t l0 = 0; l0 < net->layers; l0 += 16) {
        PackArgs pa{};
        pa.src = net->layers_buf;
        pa.dst = net->pin_out;
        pa.count = net->layers - l0 < 16 ? net->layers - l0 : 16;
        uint32_t widest = 1;
        for (uint32_t i = 0; i < pa.count; ++i) {
            pa.src_off[i] = net->slot_off[l0 + i];
            pa.dst_off[i] = dense;
            pa.len[i] = net->topo[l0 + i];
            dense += net->topo[l0 + i];
            if (pa.len[i] > widest) widest = pa.len[i];
        }
        if (one_launch) {
            uint32_t seq = 0;
            if (next_signal(net, &seq)) return 1;
            sp_gather_host<<<1, 1024, 0, g_stream>>>(GatherArgs{pa, dense, logits, net->pin_flag, seq});
            if (wait_for_signal(net, seq)) return 1;
            break;
        }
        uint32_t gx = (widest + 255) / 256;
        if (gx > 64) gx = 64;
        sp_pack_layers<<<dim3(gx, pa.count), 256, 0, g_stream>>>(pa);
    }
    if (!one_launch && wait_for_small_results(net)) return 1;
    memcpy(host_neurons, net->pin_out, net->total_neurons * sizeof(float));
    return 0;
}

int sphip_evaluate(sphip_net *net, const float *x, const float *targets, uint32_t n, int loss_func, uint32_t flags,
                   float *total_loss, uint32_t *predictions, uint32_t *correct)
{
    if (!net || !x || !targets || n == 0 || (loss_func != 0 && loss_func != 1))
        return fail_msg("sphip_evaluate: invalid argument");
    if (check_uploaded(net)) return 1;
    const uint32_t fwd_flags = flags & (SPHIP_FORCE_GEMM | SPHIP_FORCE_GEMV | SPHIP_BF16_ACTIVATIONS | SPHIP_WHOLE_BATCH | SPHIP_SPLIT_ACTIVATIONS);
    if (reserve_batch(net, n, fwd_flags)) return 1;
    const uint32_t width = net->topo[net->layers - 1];
    const uint64_t in_cnt = (uint64_t)n * net->topo[0], out_cnt = (uint64_t)n * width;
    const bool on_dev = (flags & SPHIP_X_ON_DEVICE) != 0;
    // layout of the evaluation buffer (4-byte units): outputs | staged targets | loss | pred | hit | totals (16 bytes)
    const uint64_t need = out_cnt * (on_dev ? 1u : 2u) + 3ull * n + 8u;
    if (grow(&net->eval_buf, &net->eval_cap, need)) return 1;
    float *d_y = net->eval_buf;
    float *d_t = on_dev ? nullptr : net->eval_buf + out_cnt;
    float *d_loss = net->eval_buf + out_cnt * (on_dev ? 1u : 2u);
    uint32_t *d_pred = reinterpret_cast<uint32_t *>(d_loss + n);
    uint32_t *d_hit = d_pred + n;
    double *d_tot = reinterpret_cast<double *>((reinterpret_cast<uintptr_t>(d_hit + n) + 7u) & ~(uintptr_t)7u);
    uint32_t *d_hits = reinterpret_cast<uint32_t *>(d_tot + 1);
    if (on_dev) {
        if (enqueue_forward_batch(net, x, n, d_y, fwd_flags, 0)) return 1;
    } else {
        if (grow(&net->stage_x, &net->stage_x_cap, in_cnt)) return 1;
        if (upload_from_host(d_t, targets, out_cnt * sizeof(float))) return 1;
        if (enqueue_forward_from_host(net, x, n, d_y, fwd_flags)) return 1;
    }
    EvalArgs a{d_y, on_dev ? targets : d_t, d_loss, d_pred, d_hit, n, width, loss_func,
               net->act[net->layers - 2] == A_SIGMOID ? 1 : 0};
    sp_eval_rows<<<(n + 3) / 4, 256, 0, g_stream>>>(a);
    sp_eval_total<<<1, 1024, 0, g_stream>>>(d_loss, d_hit, n, d_tot, d_hits);
    HCHECK(hipGetLastError());
    struct { double loss; uint32_t hits; uint32_t pad; } tot;
    HCHECK(hipMemcpyAsync(&tot, d_tot, 16, hipMemcpyDeviceToHost, g_stream));
    if (predictions) HCHECK(hipMemcpyAsync(predictions, d_pred, (size_t)n * sizeof(uint32_t), hipMemcpyDeviceToHost, g_stream));
    HCHECK(hipStreamSynchronize(g_stream));
    if (total_loss) *total_loss = (float)tot.loss;
    if (correct) *correct = tot.hits;
    return 0;
}

int sphip_decode(sphip_net *net, uint32_t l, int which, int mode, float *host_out)
{
    if (!net || l + 1 >= net->layers || (which != 0 && which != 1) || !host_out || (mode != 0 && mode != 1))
        return fail_msg("sphip_decode: invalid argument");
    const DevArray &a = which == 0 ? net->W[l] : net->B[l];
    if (!a.uploaded) return fail_msg("sphip_decode: array not uploaded");
    float *d_out = nullptr;
    HCHECK(hipMalloc((void **)&d_out, a.count * sizeof(float)));
    DecodeParams p{};
    p.codes = which == 0 && !a.base ? net->PW[l].base : a.base;
    p.cols = which == 0 ? net->topo[l] : 1u;
    p.pcols = which == 0 && !a.base ? net->ptopo[l] : p.cols;
    p.out = d_out;
    p.n = a.count;
    p.max_val = a.max_val;
    p.mode = mode;
    const float d = fmt_divisor(net->prec);
    {
        volatile float r = 1.0f / d;
        volatile float s = a.max_val * r;
        p.rel_scale = s;
    }
    if (net->prec == I8) for (int q = -128; q < 128; ++q) { volatile float fq = (float)q; volatile float tq = fq / 127.0f; p.lut[q + 128] = tq; }
    if (net->prec == I4) for (int q = -8; q < 8; ++q) { volatile float fq = (float)q; volatile float tq = fq / 7.0f; p.lut[q + 8] = tq; }
    const uint32_t grid = (uint32_t)((a.count + 255) / 256);
    switch (net->prec) {
    case F32:  sp_decode<F32><<<grid, 256, 0, g_stream>>>(p); break;
    case F16:  sp_decode<F16><<<grid, 256, 0, g_stream>>>(p); break;
    case BF16: sp_decode<BF16><<<grid, 256, 0, g_stream>>>(p); break;
    case I8:   sp_decode<I8><<<grid, 256, 0, g_stream>>>(p); break;
    case I4:   sp_decode<I4><<<grid, 256, 0, g_stream>>>(p); break;
    default:   sp_decode<I2><<<grid, 256, 0, g_stream>>>(p); break;
    }
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(host_out, d_out, a.count * sizeof(float), hipMemcpyDeviceToHost, g_stream);
    if (e == hipSuccess) e = hipStreamSynchronize(g_stream);
    (void)hipFree(d_out);
    if (e != hipSuccess) return fail_hip("sphip_decode", e);
    return 0;
}

int sphip_synchronize(void)
{
    if (!g_stream) return 0;
    HCHECK(hipStreamSynchronize(g_stream));
    return 0;
}

int sphip_malloc(void **dptr, size_t bytes)
{
    if (!dptr) return fail_msg("sphip_malloc: null");
    if (ensure_stream()) return 1;
    HCHECK(hipMalloc(dptr, bytes ? bytes : 1));
    return 0;
}

int sphip_device_memory(size_t *free_bytes, size_t *total_bytes)
{
    if (!free_bytes || !total_bytes) return fail_msg("sphip_device_memory: null");
    if (ensure_stream()) return 1;
    HCHECK(hipMemGetInfo(free_bytes, total_bytes));
    return 0;
}

int sphip_free(void *dptr)
{
    if (dptr) HCHECK(hipFree(dptr));
    return 0;
}

int sphip_memcpy_h2d(void *dst, const void *src, size_t bytes)
{
    if (ensure_stream()) return 1;
    if (upload_from_host(dst, src, bytes)) return 1;
    HCHECK(hipStreamSynchronize(g_stream));
    return 0;
}

int sphip_memcpy_d2h(void *dst, const void *src, size_t bytes)
{
    if (ensure_stream()) return 1;
    HCHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, g_stream));
    HCHECK(hipStreamSynchronize(g_stream));
    return 0;
}

static int time_common(sphip_net *const *nets, int count, const float *d_x, uint32_t n, float *d_y,
                       uint32_t flags, int iters, float *ms, uint32_t only_layer)
{
    if (!nets || count <= 0 || iters <= 0 || !ms) return fail_msg("sphip_time: invalid argument");
    for (int i = 0; i < count; ++i) {
        if (!nets[i]) return fail_msg("sphip_time: null net");
        if (check_uploaded(nets[i])) return 1;
        if (reserve_batch(nets[i], n, flags)) return 1;
    }
    TimingEvents ev;
    if (ev.create()) return 1;
    hipEvent_t e0 = ev.e0, e1 = ev.e1;
    int rc = 0;
    HCHECK(hipEventRecord(e0, g_stream));
    for (int it = 0; it < iters && !rc; ++it) rc = enqueue_forward_batch(nets[it % count], d_x, n, d_y, flags, only_layer);
    hipError_t e = hipEventRecord(e1, g_stream);
    if (e == hipSuccess) e = hipEventSynchronize(e1);
    if (e == hipSuccess) e = hipEventElapsedTime(ms, e0, e1);
    if (rc) return rc;
    if (e != hipSuccess) return fail_hip("sphip_time", e);
    return 0;
}

int sphip_time_forward(sphip_net *const *nets, int count, const float *d_x, uint32_t n, float *d_y,
                       uint32_t flags, int iters, float *ms)
{
    if (!d_x || !d_y || n == 0) return fail_msg("sphip_time_forward: invalid argument");
    return time_common(nets, count, d_x, n, d_y, flags, iters, ms, 0);
}

int sphip_time_layer(sphip_net *const *nets, int count, uint32_t layer, uint32_t n, uint32_t flags,
                     int iters, float *ms)
{
    if (!nets || count <= 0 || !nets[0] || layer == 0 || layer >= nets[0]->layers || n == 0)
        return fail_msg("sphip_time_layer: invalid argument");
    // inputs and outputs are the nets' own scratch buffers (contents irrelevant for timing)
    for (int i = 0; i < count; ++i) {
        if (reserve_batch(nets[i], n, flags)) return 1;
        if (grow(&nets[i]->stage_y, &nets[i]->stage_y_cap, (uint64_t)n * nets[i]->topo[nets[i]->layers - 1])) return 1;
        if (grow(&nets[i]->stage_x, &nets[i]->stage_x_cap, (uint64_t)n * nets[i]->topo[0])) return 1;
    }
    return time_common(nets, count, nets[0]->stage_x, n, nets[0]->stage_y, flags, iters, ms, layer);
}

uint32_t sphip_batch_block_rows(sphip_net *net, uint32_t n, uint32_t flags)
{
    if (!net || n == 0) return 0;
    return batch_block_rows(net, n, flags);
}

const char *sphip_layer_kernel_name(sphip_net *net, uint32_t layer, uint32_t n, uint32_t flags)
{
    if (!net || layer == 0 || layer >= net->layers || n == 0) return "";
    // the routing code itself, run without launching: workspaces are taken as reserve() would have sized them and
    // pointers as aligned, which is how sphip_forward calls it
    tl_route.dry = true;
    tl_route.name = "";
    const LayerArgs L = make_layer_args(net, layer, layer == 1 && pick_regime(net, n, flags) == R_GEMV && raw_rows(net->prec, net->topo[0], net->ptopo[1], n));
    const float *aligned_ptr = reinterpret_cast<const float *>(uintptr_t{256});     // never dereferenced
    switch (pick_regime(net, n, flags)) {
    case R_GEMV:
        launch_gemv(net->prec, net->workspace(), L, aligned_ptr, nullptr, n, false, net->ptopo[layer - 1] != net->topo[layer - 1]);
        break;
    case R_GEMM32:
        if (f32_thin_vector(L, n)) launch_gemv(net->prec, net->workspace(), L, aligned_ptr, nullptr, n, false);
        else (void)launch_gemm32(L, aligned_ptr, nullptr, n, nullptr, ~0ull, nullptr, n);
        break;
    case R_CAT3: {
        if (!cat3_layer(n, L.N, L.K)) {
            if (f32_thin_vector(L, n)) launch_gemv(net->prec, net->workspace(), L, aligned_ptr, nullptr, n, false);
            else (void)launch_gemm32(L, aligned_ptr, nullptr, n, nullptr, ~0ull, nullptr, n);
            break;
        }
        LayerArgs L3 = L;
        L3.K = 3u * cat3_kp(L.K);
        ThinCtx ctx{};
        ctx.w16 = reinterpret_cast<const uint16_t *>(aligned_ptr);
        ctx.ws_floats = ~0ull;
        launch_gemm16((int)F16, L3, reinterpret_cast<const uint16_t *>(aligned_ptr), nullptr, n, 1, ctx);
        break;
    }
    default: {
        ThinCtx ctx{};
        ctx.w16 = reinterpret_cast<const uint16_t *>(aligned_ptr);
        ctx.ws_floats = ~0ull;
        ctx.padded_in = layer == 1 && net->ptopo[0] != net->topo[0];
        tl_route.halves = (flags & SPHIP_SPLIT_ACTIVATIONS) ? 2u : 1u;
        launch_gemm16(net->prec, L, reinterpret_cast<const uint16_t *>(aligned_ptr), nullptr, n, 1, ctx);
        break;
    }
    }
    tl_route.dry = false;
    tl_route.halves = 1;
    return tl_route.name;
}

}  // extern "C"

// the batched training step (its own kernels and entry points)
#include "hip_train.inl"
#include "hip_train_tiny.inl"
