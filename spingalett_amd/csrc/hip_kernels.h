// hip_kernels.h — element formats, device helpers and the template kernels that several translation units share: the
// one that launches them (hip_forward.hip) and those that compile them (hip_part.hip).
#ifndef SPINGALETT_HIP_KERNELS_H
#define SPINGALETT_HIP_KERNELS_H

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <type_traits>

namespace sphip_kernels {

// ---------------------------------------------------------------------------
// formats and small helpers
// ---------------------------------------------------------------------------
enum : int { F32 = 0, F16 = 1, BF16 = 2, I8 = 3, I4 = 4, I2 = 5, NFMT = 6 };
enum : int { A_SIGMOID = 0, A_RELU, A_TANH, A_LEAKY, A_FOO52, A_SOFTMAX, A_NONE, A_COUNT };

constexpr int kWave = 64;

__host__ __device__ constexpr int fmt_bits(int f)
{
    return f == F32 ? 32 : (f == F16 || f == BF16) ? 16 : f == I8 ? 8 : f == I4 ? 4 : 2;
}

// ---------------------------------------------------------------------------
// device-side element access
// ---------------------------------------------------------------------------
__device__ __forceinline__ float bits_to_float(uint32_t u) { return __uint_as_float(u); }

// binary16 -> binary32, integer arithmetic only; any NaN becomes the quiet NaN
// of the same sign (Serialize.c:45-72).
__device__ __forceinline__ float half_bits_to_float_exact(uint32_t h)
{
    uint32_t s = (h & 0x8000u) << 16;
    uint32_t e = (h >> 10) & 31u;
    uint32_t m = h & 1023u;
    uint32_t f;
    if (e == 31u) {
        f = s | (m ? 0x7FC00000u : 0x7F800000u);
    } else if (e != 0u) {
        f = s | ((e + 112u) << 23) | (m << 13);
    } else if (m == 0u) {
        f = s;
    } else {
        int lz = __clz((int)m) - 21;               // shifts until bit 10 is set
        m = (m << lz) & 1023u;
        f = s | ((uint32_t)(113 - lz) << 23) | (m << 13);
    }
    return bits_to_float(f);
}

// integer code of element i of a packed INT array
template <int FMT>
__device__ __forceinline__ int int_code(const uint8_t *codes, uint64_t i)
{
    if constexpr (FMT == I8) {
        return (int)(int8_t)codes[i];
    } else if constexpr (FMT == I4) {
        uint32_t byte = codes[i >> 1];
        uint32_t nib = (i & 1u) ? (byte >> 4) : (byte & 15u);
        return (int)nib - (int)((nib & 8u) << 1);
    } else {
        uint32_t c = (codes[i >> 2] >> ((i & 3u) * 2u)) & 3u;
        return (int)c - (int)((c & 2u) << 1);
    }
}

// unscaled value of element i: the float itself for FP formats, (float)q for INT
template <int FMT>
__device__ __forceinline__ float elem_value(const uint8_t *codes, uint64_t i)
{
    if constexpr (FMT == F32) {
        return reinterpret_cast<const float *>(codes)[i];
    } else if constexpr (FMT == F16) {
        return half_bits_to_float_exact(reinterpret_cast<const uint16_t *>(codes)[i]);
    } else if constexpr (FMT == BF16) {
        return bits_to_float((uint32_t)reinterpret_cast<const uint16_t *>(codes)[i] << 16);
    } else {
        return (float)int_code<FMT>(codes, i);
    }
}

__device__ __forceinline__ float elem_value_rt(int fmt, const uint8_t *codes, uint64_t i)
{
    switch (fmt) {
    case F32:  return elem_value<F32>(codes, i);
    case F16:  return elem_value<F16>(codes, i);
    case BF16: return elem_value<BF16>(codes, i);
    case I8:   return elem_value<I8>(codes, i);
    case I4:   return elem_value<I4>(codes, i);
    default:   return elem_value<I2>(codes, i);
    }
}

// Activation.c:23-38 (leak factor fixed at 0.01f).  Softmax is a row operation
// and handled by sp_softmax_rows.
__device__ __forceinline__ float apply_act(float x, int act)
{
    switch (act) {
    case A_SIGMOID: return 1.0f / (1.0f + expf(-x));
    case A_RELU:    return x > 0.0f ? x : 0.0f;
    case A_TANH:    return tanhf(x);
    case A_LEAKY:   return x > 0.0f ? x : 0.01f * x;
    case A_FOO52:   return x > 1.0f ? 1.0f + 0.01f * (x - 1.0f) : (x < 0.0f ? 0.01f * x : x);
    default:        return x;
    }
}

// tanhf's result without its branch, for code in which one wave has to hide the latency of its values behind each other: the
// library's function takes arguments below and above 0.625 apart by execution masks, one value after the other.  The first call
// is known to be a near one, which leaves so little on either side that the compiler does both and chooses.
__device__ __forceinline__ float tanh_straight(float x)
{
    const bool near = __builtin_fabsf(x) < 0.625f;
    const float a = near ? x : 0.0f;
    __builtin_assume(__builtin_fabsf(a) < 0.625f);
    const float p = tanhf(a);
    if (near) return p;
    return tanhf(x);
}

// derivative of an activation as a function of its output (Activation.c:40-56, SIMD.c:90-188)
__device__ __forceinline__ float act_derivative(float a, int act)
{
    switch (act) {
    case A_RELU:    return a > 0.0f ? 1.0f : 0.0f;
    case A_LEAKY:   return a > 0.0f ? 1.0f : 0.01f;
    case A_SIGMOID:
    case A_SOFTMAX: return a * (1.0f - a);
    case A_TANH:    return 1.0f - a * a;
    case A_FOO52:   return (a > 1.0f || a < 0.0f) ? 0.01f : 1.0f;
    default:        return 1.0f;
    }
}

// f(integral_constant<int, ACT>): a copy of an epilogue for each activation.  Behind every output of a lane, in an unrolled
// loop, a switch over the activations is a chain of branches and code fetched for nothing (FP32 layers 4096 x 512 x 784 with
// tanh 36.9 -> 35.5 us, 2048 x 1000 x 512 with a leaky ReLU 25.8 -> 24.3).
template <class F>
__device__ __forceinline__ void with_act(int act, F &&f)
{
    switch (act) {
    case A_SIGMOID: f(std::integral_constant<int, A_SIGMOID>{}); break;
    case A_RELU:    f(std::integral_constant<int, A_RELU>{}); break;
    case A_TANH:    f(std::integral_constant<int, A_TANH>{}); break;
    case A_LEAKY:   f(std::integral_constant<int, A_LEAKY>{}); break;
    case A_FOO52:   f(std::integral_constant<int, A_FOO52>{}); break;
    default:        f(std::integral_constant<int, A_NONE>{}); break;
    }
}

// FP32 -> BF16, round to nearest even, NaNs stay NaNs: the part's own conversion instruction
__device__ __forceinline__ uint16_t f32_to_bf16_rne(float x)
{
    const __bf16 h = (__bf16)x;
    uint16_t r;
    __builtin_memcpy(&r, &h, 2);
    return r;
}

// FP32 -> FP16: finite values beyond the FP16 range become +-65504 (an activation that large stays finite in the
// reference's FP32 arithmetic; an infinity here would turn into NaNs in the next layer), infinities and NaNs stay
// what they are.
__device__ __forceinline__ uint16_t f32_to_f16_sat(float x)
{
    // without a branch, which every output of an unrolled epilogue would take (8192 samples of the 8192-wide BF16 net
    // 7.28 -> 7.13 ms, 256 of 784-512-1000-10 INT8 19.7 -> 19.1 us)
    constexpr int kInfNan = 0x207;
    const float c = __builtin_amdgcn_classf(x, kInfNan) ? x : __builtin_amdgcn_fmed3f(x, -65504.0f, 65504.0f);
    const _Float16 h = (_Float16)c;
    uint16_t r;
    __builtin_memcpy(&r, &h, 2);
    return x != x ? (uint16_t)0x7E00u : r;
}

template <bool F16T>
__device__ __forceinline__ uint16_t f32_to_t16(float x)
{
    if constexpr (F16T) return f32_to_f16_sat(x);
    else return f32_to_bf16_rne(x);
}

// A value loaded at the start of a kernel for its end is here from now on: said in front of the last barrier, it keeps the
// compiler from asking for it behind that, where nothing hides the latency
__device__ __forceinline__ void here(float &v) { asm volatile("" : "+v"(v)); }

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>)
template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(F &&f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}

__device__ __forceinline__ float wave_sum(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}

__device__ __forceinline__ int wave_sum_i(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}

__device__ __forceinline__ uint32_t wave_max_u(uint32_t v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, o, kWave));
    return v;
}

__device__ __forceinline__ float wave_max(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, kWave));
    return v;
}

#include "hip_gemv.inl"

#include "hip_gemm16.inl"

#include "hip_skinny.inl"

}  // namespace sphip_kernels

#endif
