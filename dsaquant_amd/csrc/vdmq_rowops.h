// Device code that turns one token row, held in the registers of a wave, into what the quantizers need: reductions over the
// wave, the row's scale, the fused activation, the fused LayerNorm.  Shared by the quantizers (vdmq_quant.hip) and the linear
// that quantizes the rows it works on itself (vdmq_resident.hip): both have to give the same bits.
#pragma once

#include "vdmq_internal.h"

namespace vdmq {
namespace {

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pk_max_u16(uint32_t a, uint32_t b) {
    u16x2 r = __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b));
    return __builtin_bit_cast(uint32_t, r);
}

__device__ __forceinline__ float half_bits_to_float(uint32_t bits16) {
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<unsigned short>(bits16)));
}

// Reductions over the wave's 64 lanes on the VALU (DPP): four steps leave a row of 16 lanes with its own result, two
// broadcasts carry it on to the last lane, and the result comes back as a scalar.  (Six ds_bpermute steps with their
// address arithmetic cost five times the instructions and an LDS round trip each: 240 of the 560 vector instructions
// that a 1536-wide row takes through the fused LayerNorm quantizer.)
template <int CTRL, int ROWS, bool BOUND>
__device__ __forceinline__ uint32_t dpp(uint32_t old, uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(old), static_cast<int>(v), CTRL, ROWS, 0xF, BOUND));
}
constexpr int kDppSwap1 = 0xB1, kDppSwap2 = 0x4E, kDppHalfMirror = 0x141, kDppMirror = 0x140, kDppBcast15 = 0x142, kDppBcast31 = 0x143;

__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
    auto step = [&](uint32_t o) { v = o > v ? o : v; };
    step(dpp<kDppSwap1, 0xF, false>(v, v));
    step(dpp<kDppSwap2, 0xF, false>(v, v));
    step(dpp<kDppHalfMirror, 0xF, false>(v, v));
    step(dpp<kDppMirror, 0xF, false>(v, v));
    step(dpp<kDppBcast15, 0xA, false>(v, v));
    step(dpp<kDppBcast31, 0xC, false>(v, v));
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 63));
}

__device__ __forceinline__ float wave_max(float v) { /* v >= 0 in every lane: the bits order as the values do */
    return __uint_as_float(wave_max(__float_as_uint(v)));
}

// Sum in the order of a butterfly over lane distances 32, 16, 8, 4, 2, 1, the order that the LayerNorm's values rest on: an
// fp32 sum in another order moves single fp16 results, and with them int4 codes.  (From the fourth step on lanes 8 apart hold
// equal values, so a rotation by 4 within the row of 16 meets the same number as an exchange at distance 4.)
constexpr int kDppRotate8 = 0x128, kDppRotate4 = 0x124;
__device__ __forceinline__ float wave_sum(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
    u32x2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r.x) + __uint_as_float(r.y);
    r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r.x) + __uint_as_float(r.y);
#endif
    v += __uint_as_float(dpp<kDppRotate8, 0xF, false>(0u, __float_as_uint(v)));
    v += __uint_as_float(dpp<kDppRotate4, 0xF, false>(0u, __float_as_uint(v)));
    v += __uint_as_float(dpp<kDppSwap2, 0xF, false>(0u, __float_as_uint(v)));
    v += __uint_as_float(dpp<kDppSwap1, 0xF, false>(0u, __float_as_uint(v)));
    return __uint_as_float(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(__float_as_uint(v)))));
}

// fmaxf semantics of the reference's reduction: a NaN operand is ignored.
__device__ __forceinline__ float max_ignoring_nan(float acc, float a) { return (a == a && a > acc) ? a : acc; }

__device__ __forceinline__ uint32_t absmax_bits(u32x4 v, uint32_t m) {
    m = pk_max_u16(m, v.x & 0x7FFF7FFFu);
    m = pk_max_u16(m, v.y & 0x7FFF7FFFu);
    m = pk_max_u16(m, v.z & 0x7FFF7FFFu);
    m = pk_max_u16(m, v.w & 0x7FFF7FFFu);
    return m;
}

__device__ __forceinline__ float absmax_exact(u32x4 v, float mx) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        mx = max_ignoring_nan(mx, fabsf(half_bits_to_float(w[i] & 0xFFFFu)));
        mx = max_ignoring_nan(mx, fabsf(half_bits_to_float(w[i] >> 16)));
    }
    return mx;
}

// An fp32 result about to be rounded to fp16: the compiler may not fold the operation that made it into the conversion
// (v_fma_mixlo_f16 rounds once, the contract's fp32 operation followed by a conversion twice).
__device__ __forceinline__ float rounded_f32(float v) {
    asm("" : "+v"(v));
    return v;
}

// scale = max > 0 ? (max / 7) * clip : 1, rounded to fp16 (token_scale_kernel).
__device__ __forceinline__ __half scale_from_absmax(float amax, float clip) {
    // amax / 7, correctly rounded: amax is an fp16 value, and for every one of those one correction step gives the
    // rounded quotient (three operations; the division takes ten)
    constexpr float kInv7 = 1.0f / 7.0f;
    const float q = amax * kInv7;
    const float seventh = amax < __builtin_inff() ? __builtin_fmaf(__builtin_fmaf(-7.0f, q, amax), kInv7, q) : amax;
    const float s = amax > 0.0f ? seventh * clip : 1.0f;
    return __float2half_rn(rounded_f32(s));
}

// 1 / s, correctly rounded, for an ordinary fp16 scale (checked for every one of them by the tests)
__device__ __forceinline__ float reciprocal_of_scale(float s) {
    const float r = __builtin_amdgcn_rcpf(s);
    return __builtin_fmaf(__builtin_fmaf(-s, r, 1.0f), r, r);
}

__device__ __forceinline__ bool scale_is_ordinary(__half s) {
    uint32_t b = __half_as_ushort(s) & 0x7FFFu;
    return b != 0u && b < 0x7C00u;
}

// GELU, tanh approximation, on an fp16 value: the fp32 evaluation a framework
// applies to an fp16 tensor (the reference's FeedForward uses
// activation_fn="gelu-approximate", dit_block.py:56), rounded once to fp16:
//   u = sqrt(2/pi) * (x + 0.044715 * x^3),  gelu = 0.5 * x * (1 + tanh(u)).
// 0.5 * (1 + tanh(u)) is evaluated as 1 / (1 + exp(-2u)): no cancellation in the
// negative tail, so the fp32 result is a few ulp(fp32) from the exact value and
// the fp16 result is the correctly rounded one except next to a rounding boundary.
// +inf -> +inf, -inf -> NaN (= -inf * 0, as the formula gives), NaN -> NaN.
__device__ __forceinline__ float gelu_tanh_f32(float x) {
    // -2 * log2(e) * u = x * (c1 + c2 * x^2): the exponent of 2 in exp(-2u)
    constexpr float kC1 = -2.8853900817779268f * 0.7978845608028654f;
    constexpr float kC2 = kC1 * 0.044715f;
    const float a = x * __builtin_fmaf(kC2, x * x, kC1);
    const float e = __builtin_amdgcn_exp2f(a);
    return x * __builtin_amdgcn_rcpf(1.0f + e);
}

__device__ __forceinline__ uint32_t gelu_tanh_pair(uint32_t w) {
    const f16x2 h = __builtin_bit_cast(f16x2, w);
    f16x2 r;
    r[0] = static_cast<_Float16>(rounded_f32(gelu_tanh_f32(static_cast<float>(h[0]))));
    r[1] = static_cast<_Float16>(rounded_f32(gelu_tanh_f32(static_cast<float>(h[1]))));
    return __builtin_bit_cast(uint32_t, r);
}

template <int ACT>
__device__ __forceinline__ u32x4 apply_act(u32x4 v) {
    if (ACT == VDMQ_ACT_GELU_TANH) {
        v.x = gelu_tanh_pair(v.x);
        v.y = gelu_tanh_pair(v.y);
        v.z = gelu_tanh_pair(v.z);
        v.w = gelu_tanh_pair(v.w);
    }
    return v;
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x6 __attribute__((ext_vector_type(6)));

// 32 values t, the even ones and the odd ones, as E3M2 floats t / 16: 192 bits.  The instruction writes result registers while it still
// reads operands: with a result that began at an operand's third register, codes came out wrong.  The builtin leaves the compiler free to
// choose such registers, so this is the instruction itself, with a result that is written before the operands are read for the last time
// and hence shares no register with them.  (One instruction and no load: nothing in flight, and its operands are results of
// ordinary fp32 operations, so that no wait is due in front of it or behind.)
__device__ __forceinline__ u32x6 to_bf6(const f32x16 &even, const f32x16 &odds) {
    u32x6 r = {};
#if defined(__HIP_DEVICE_COMPILE__)
    asm("v_cvt_scalef32_2xpk16_bf6_f32 %0, %1, %2, %3" : "=&v"(r) : "v"(even), "v"(odds), "s"(16.0f));
#endif
    return r;
}

// LayerNorm (fp32 statistics over K elements) and modulation or affine of the row in `v` (v[c] = elements 512c + 8*lane ...
// +7, zero beyond K), in place; `pa` and `pb` are the row's two vectors (see ln_quantize_rows_kernel).  The chunks below FULL
// are complete in every lane and need no bounds test.
template <int NCH, int LNMODE, int FULL>
__device__ __forceinline__ void ln_row(u32x4 (&v)[NCH], int lane, int K, float eps, const u32x4 *__restrict__ pa, const u32x4 *__restrict__ pb) {
    float sum = 0.0f;
    float one = 1.0f; /* a multiplier the compiler cannot see through: fma(x, one, y) stays a fused multiply-add */
    asm volatile("" : "+s"(one));
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const uint32_t w[4] = {v[c].x, v[c].y, v[c].z, v[c].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const f16x2 h = __builtin_bit_cast(f16x2, w[i]);
            // fma(x, 1, s) = fl(x + s) as one v_fma_mix_f32, which reads the fp16 value directly (padding adds zeros)
            sum = __builtin_fmaf(static_cast<float>(h[0]), one, sum);
            sum = __builtin_fmaf(static_cast<float>(h[1]), one, sum);
        }
    }
    const float mean = wave_sum(sum) / static_cast<float>(K);
    // Each pass converts the fp16 row again: the compiler would otherwise keep the 8 * NCH converted floats of one
    // pass for the next (80 registers for a 5120-wide row, a workgroup per CU less); the empty asm makes the row
    // a new value for it.
#pragma unroll
    for (int c = 0; c < NCH; ++c) asm volatile("" : "+v"(v[c]));
    float sq = 0.0f;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int k0 = c * 512 + lane * 8;
        if (c < FULL || k0 < K) {
            const uint32_t w[4] = {v[c].x, v[c].y, v[c].z, v[c].w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f16x2 h = __builtin_bit_cast(f16x2, w[i]);
                const float d0 = __builtin_fmaf(static_cast<float>(h[0]), one, -mean), d1 = __builtin_fmaf(static_cast<float>(h[1]), one, -mean);
                sq = __builtin_fmaf(d0, d0, sq);
                sq = __builtin_fmaf(d1, d1, sq);
            }
        }
    }
    const float rstd = 1.0f / __builtin_sqrtf(wave_sum(sq) / static_cast<float>(K) + eps);
#pragma unroll
    for (int c = 0; c < NCH; ++c) asm volatile("" : "+v"(v[c]));

#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int k0 = c * 512 + lane * 8;
        if (c < FULL || k0 < K) {
            const u32x4 a4 = pa[c * 64 + lane], b4 = pb[c * 64 + lane];
            const uint32_t w[4] = {v[c].x, v[c].y, v[c].z, v[c].w};
            const uint32_t aw[4] = {a4.x, a4.y, a4.z, a4.w}, bw[4] = {b4.x, b4.y, b4.z, b4.w};
            uint32_t o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f16x2 h = __builtin_bit_cast(f16x2, w[i]);
                const f16x2 a = __builtin_bit_cast(f16x2, aw[i]), b = __builtin_bit_cast(f16x2, bw[i]);
                const float n0 = __builtin_fmaf(static_cast<float>(h[0]), one, -mean) * rstd;
                const float n1 = __builtin_fmaf(static_cast<float>(h[1]), one, -mean) * rstd;
                f16x2 r;
                if (LNMODE == VDMQ_LN_MODULATE) {
                    const f16x2 ln = {static_cast<_Float16>(n0), static_cast<_Float16>(n1)};
                    const f16x2 one = {static_cast<_Float16>(1.0f), static_cast<_Float16>(1.0f)};
                    r = ln * (one + a) + b; /* three packed fp16 operations, each rounded (no contraction) */
                } else {
                    r[0] = static_cast<_Float16>(n0 * static_cast<float>(a[0]) + static_cast<float>(b[0]));
                    r[1] = static_cast<_Float16>(n1 * static_cast<float>(a[1]) + static_cast<float>(b[1]));
                }
                o[i] = __builtin_bit_cast(uint32_t, r);
            }
            v[c] = u32x4{o[0], o[1], o[2], o[3]};
        }
    }
}

}  // namespace
}  // namespace vdmq
