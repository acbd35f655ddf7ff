// FP32 values as two scaled fp16 terms, for the 16-bit matrix cores:
// v 2^s = hi + 2^-11 lo with hi = rn(v 2^s), lo = rn(2^11 (v 2^s - hi)), s a
// power of two for a group of values that puts the largest in [2^13, 2^14).
// |error| <= max(2^-23 |v 2^s|, 2^-36).  Used by fir_f16x2.hip and fir_vjp.hip.
#pragma once

#include "common.hpp"

namespace scir {
namespace {

typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// f over the wave (idempotent f: min or max): DPP row shifts, then row
// broadcasts; all VALU.
template <class F>
__device__ __forceinline__ int wave_reduce(int v, F f)
{
    v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x111, 0xF, 0xF, false));  // row_shr:1
    v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x112, 0xF, 0xF, false));  // row_shr:2
    v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x114, 0xF, 0xF, false));  // row_shr:4
    v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x118, 0xF, 0xF, false));  // row_shr:8
    v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xA, 0xF, false));  // row_bcast:15
    v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xC, 0xF, false));  // row_bcast:31
    return __builtin_amdgcn_readlane(v, 63);
}

// max(a, |b|, |c|), NaN if any is: one v_maximum3_f32.
__device__ __forceinline__ float maximum3(float a, float b, float c)
{
    return __builtin_elementwise_maximum(
        __builtin_elementwise_maximum(__builtin_fabsf(b), __builtin_fabsf(c)), a);
}

// min(a, |b|, |c|), NaN if any is: one v_minimum3_f32.
__device__ __forceinline__ float minimum3(float a, float b, float c)
{
    return __builtin_elementwise_minimum(
        __builtin_elementwise_minimum(__builtin_fabsf(b), __builtin_fabsf(c)), a);
}

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
constexpr float kLoUnscale = 1.0f / 2048.0f;  // 2^-11: the low term's scale is 2^11

// The powers of two of an F16x2 split, of samples or taps.
struct SplitScale {
    float to;       // 2^s
    float from;     // 2^-s
    float to_lo;    // 2^(s + 11)
};

// The two fp16 terms, as packed words, of four values: three mixed-precision
// multiply-adds a value (hi = rn(2^s v); v - 2^-s hi, exact; lo), where the
// compiler's choice takes four and a half.  Each write of half a register is
// one instruction away from the next use of that register, as the hardware
// requires.
__device__ __forceinline__ void split2_quad(const f32x4 &v, const SplitScale &c,
                                            unsigned int (&h)[2], unsigned int (&l)[2])
{
    float r1, r3;
    asm("v_fma_mixlo_f16 %0, %6, %10, 0\n\t"
        "v_fma_mixlo_f16 %1, %8, %10, 0\n\t"
        "v_fma_mixhi_f16 %0, %7, %10, 0\n\t"
        "v_fma_mixhi_f16 %1, %9, %10, 0\n\t"
        "v_fma_mix_f32 %2, %0, -%11, %6 op_sel_hi:[1,0,0]\n\t"
        "v_fma_mix_f32 %4, %0, -%11, %7 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
        "v_fma_mix_f32 %3, %1, -%11, %8 op_sel_hi:[1,0,0]\n\t"
        "v_fma_mix_f32 %5, %1, -%11, %9 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
        "v_fma_mixlo_f16 %2, %2, %12, 0\n\t"
        "v_fma_mixlo_f16 %3, %3, %12, 0\n\t"
        "v_fma_mixhi_f16 %2, %4, %12, 0\n\t"
        "v_fma_mixhi_f16 %3, %5, %12, 0\n\t"
        "s_nop 0"
        : "=&v"(h[0]), "=&v"(h[1]), "=&v"(l[0]), "=&v"(l[1]), "=&v"(r1), "=&v"(r3)
        : "v"(v.x), "v"(v.y), "v"(v.z), "v"(v.w), "s"(c.to), "s"(c.from), "s"(c.to_lo));
}

__device__ __forceinline__ unsigned int abs_bits(float v)
{
    return __builtin_bit_cast(unsigned int, v) & 0x7fffffffu;
}
__device__ __forceinline__ float pow2(int e)  // |e| <= 126
{
    return __builtin_bit_cast(float, (unsigned int)(e + 127) << 23);
}
__device__ __forceinline__ SplitScale split_scale(int s)  // |s| <= 100
{
    return {pow2(s), pow2(-s), pow2(s + 11)};
}
__device__ __forceinline__ int wave_umax(unsigned int v)
{
    return wave_reduce((int)v, [](int a, int b) { return (int)max((unsigned)a, (unsigned)b); });
}
__device__ __forceinline__ int wave_umin(unsigned int v)
{
    return wave_reduce((int)v, [](int a, int b) { return (int)min((unsigned)a, (unsigned)b); });
}
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float uniform(float v)
{
    return __builtin_bit_cast(float, uniform(__builtin_bit_cast(int, v)));
}

// Scale exponent that puts a largest magnitude (bits mx) in [2^13, 2^14).
__device__ __forceinline__ int scale_exponent(unsigned int mx)
{
    return mx ? 14 - __builtin_amdgcn_frexp_expf(__builtin_bit_cast(float, mx)) : 0;
}

}  // namespace
}  // namespace scir
