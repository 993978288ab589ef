// What runs between the W4A4 linears of an attention module, for gfx950: the mask-free attention, and q/k RMS-norm with
// the rotary embedding and its table of rotations.
#include "vdmq_internal.h"

namespace vdmq {
namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

#define VDMQ_LDS_PTR(p) ((__attribute__((address_space(3))) void *)(p))

// ---------------------------------------------------------------- attention
//
// Mask-free attention with a head dimension of 128 (models/base/vdm_attn.py:241-259 of the reference), one pass over the
// keys with a running maximum.  A wave owns 32 queries, held as matrix operands; a workgroup of WAVES waves shares 64 keys
// per step, whose K and V rows (16 KiB each) go from memory straight to LDS, two steps' worth in turn.
//
// Both products run transposed: S^T = K Q^T leaves a query's scores of 16 of 32 keys in one lane (the other 16 in the lane
// 32 further), so the softmax is lane-local but for one exchange of the maximum, and the probabilities, rounded to fp16,
// are the second product's operand as they lie: O^T = V^T P^T, whose k slots are put in the order in which the first
// product's rows came out.  V^T comes from the row-major V rows by transposing LDS reads.  The 16-byte pieces of a row are
// permuted in LDS (K: piece ^ row % 16, V: piece ^ 4 * (row % 4)), by the source address of the loads, so that neither
// read meets a bank twice.
//
// What bounds it: per step and wave 32 matrix instructions (1024 cycles) and 32 exponentials and about 100 other vector
// instructions per lane (900 cycles), which the SIMD's two waves overlap in part, and long launches run at the clock the
// power budget leaves.  TFLOP/s (4 * Lq * Lk * 128 per head) / us, before (the framework's attention) and now:
//   4680 x 4680, 12 heads: 201 / 668 -> 790 / 170     4680 x 512, 12 heads: 373 / 39.5 -> 560 / 26
//   1560 x 1560, 12 heads: 109 / 137 -> 390 / 38      32760 x 32760, 12 heads: 450 / 14640 -> 1060 / 6210
// Error against 64 bits (2-norm, N(0, 1) operands): 2.73e-4 before, 2.73e-4 now.  The maximum is the exact running one:
// rescaling only when it has grown by 2^8 is 3...9 % faster, but then the largest probabilities no longer lie just below
// a power of two, where fp16 is finest, and the error grows by 6 %.  The probabilities are held times 2^15: unscaled, those
// below 2^-14 of the largest are denormal fp16 and below 2^-25 nothing, and tens of thousands of keys there do count; so
// they are rounded at 2^-11 down to 2^-29 of the largest and gone below 2^-40.  (The power of two goes into the maximum that is
// subtracted; not for scores beyond 2^20, whose own rounding could then carry a probability past fp16.)  Within 2 %: raised wave priority around the matrix
// instructions, the two key blocks' instructions interleaved, the next step's loads behind the first product.

constexpr int kHeadDim = 128;
constexpr float kProbLog2 = 15.0f, kExactShift = 1048576.0f;
constexpr int kKeys = 64;                       /* keys per step */
constexpr int kTileBytes = kKeys * kHeadDim * 2; /* one step's K (or V) rows in LDS, 256 bytes each */

struct AttnArgs {
    const __half *q, *k, *v;
    __half *out;
    int64_t q_row, q_head, q_batch, k_row, k_head, k_batch, v_row, v_head, v_batch, o_row, o_head, o_batch; /* elements */
    int heads, lq, lk, q_tiles;
    int64_t tiles; /* batch * heads * q_tiles */
    float scale_log2; /* softmax scale * log2(e) */
};

#if defined(__HIP_DEVICE_COMPILE__)
// Eight bytes per lane; among 16 lanes, which point at four rows of 16 fp16 (lane i at columns 4 * (i % 4) of row i / 4),
// lane i receives column i of the four rows.
__device__ __forceinline__ f16x4 read_transposed(const uint8_t *p) {
    typedef short i16x4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4 *)(p)));
}
// max over the two halves of the wave, in both
__device__ __forceinline__ float max_halves(float x) {
    const u32x2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __builtin_fmaxf(__uint_as_float(r.x), __uint_as_float(r.y));
}
__device__ __forceinline__ float sum_halves(float x) {
    const u32x2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r.x) + __uint_as_float(r.y);
}
#endif

template <int WAVES>
__global__ __launch_bounds__(WAVES * 64, 2) void attention_kernel(AttnArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    __shared__ __attribute__((aligned(1024))) uint8_t lds[2][2][kTileBytes]; /* [buffer][K, V] */
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, lh = lane >> 5;
    // workgroup b runs on XCD b % 8: every XCD takes one run of the tiles, a head's tiles one after the other, whose K and
    // V it then finds in its L2
    const int64_t per_xcd = (a.tiles + 7) / 8, tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (static_cast<int64_t>(blockIdx.x >> 3) >= per_xcd || tile >= a.tiles) return;
    const int qt = static_cast<int>(tile % a.q_tiles), bh = static_cast<int>(tile / a.q_tiles), head = bh % a.heads, batch = bh / a.heads;
    const int q0 = qt * WAVES * 32 + wave * 32;

    f16x8 qf[8]; /* queries past the last: copies of it, never stored */
    {
        const __half *src = a.q + batch * a.q_batch + head * a.q_head + min(q0 + l32, a.lq - 1) * a.q_row + lh * 8;
#pragma unroll
        for (int m = 0; m < 8; ++m) qf[m] = *reinterpret_cast<const f16x8 *>(src + 16 * m);
    }
    const uint8_t *k_base = reinterpret_cast<const uint8_t *>(a.k + batch * a.k_batch + head * a.k_head);
    const uint8_t *v_base = reinterpret_cast<const uint8_t *>(a.v + batch * a.v_batch + head * a.v_head);
    const int k_row = static_cast<int>(a.k_row) * 2, v_row = static_cast<int>(a.v_row) * 2; /* bytes */
    const int r4 = lane >> 4, slot = lane & 15;
    // an instruction moves four rows of 256 bytes; rows past the last key read as zero or not at all (range check): their
    // scores are masked below and their V rows cleared
    const int k_off = r4 * k_row + ((slot ^ (4 * (wave & 3) + r4)) * 16), v_off = r4 * v_row + ((slot ^ (r4 << 2)) * 16);
    auto stage = [&](int kt, int buf) __attribute__((always_inline)) {
        const int64_t left = a.lk - static_cast<int64_t>(kt) * kKeys - 1;
        const int64_t rows = left < kKeys - 1 ? left : kKeys - 1;
        const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(k_base + static_cast<int64_t>(kt) * kKeys * k_row), 0,
                                                                            static_cast<int>(rows * k_row) + kHeadDim * 2, 0x00020000);
        const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(v_base + static_cast<int64_t>(kt) * kKeys * v_row), 0,
                                                                            static_cast<int>(rows * v_row) + kHeadDim * 2, 0x00020000);
#pragma unroll
        for (int j = 0; j < 16 / WAVES; ++j) {
            const int i = j * WAVES + wave;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(kr, VDMQ_LDS_PTR(lds[buf][0] + i * 1024), 16, k_off + 4 * i * k_row, 0, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(vr, VDMQ_LDS_PTR(lds[buf][1] + i * 1024), 16, v_off + 4 * i * v_row, 0, 0, 0);
        }
    };
    const int xk = lh ^ (l32 & 15);
    const int rr = (lane >> 2) & 3;
    const int v_read = (4 * lh + rr) * 256 + (2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) * 16 + (lane & 1) * 8;

    v16f o[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] = 0.0f;
    float m_ref = -__builtin_inff(), shift = 0.0f, l = 0.0f; /* of the scores times scale_log2 */
    const int steps = (a.lk + kKeys - 1) / kKeys;
    const float c = a.scale_log2;
    stage(0, 0);
    __builtin_amdgcn_s_waitcnt(0x0F70); /* vmcnt(0) */
    __syncthreads();
    for (int kt = 0; kt < steps; ++kt) {
        const int buf = kt & 1;
        if (kt + 1 < steps) stage(kt + 1, buf ^ 1);
        const int valid = a.lk - kt * kKeys;
        if (valid < kKeys) { /* (0 * whatever the unused rows hold must not be NaN) */
            for (int i = threadIdx.x; i < (kKeys - valid) * 16; i += WAVES * 64)
                *reinterpret_cast<u32x4 *>(lds[buf][1] + valid * 256 + i * 16) = u32x4{0u, 0u, 0u, 0u};
            __syncthreads();
        }
        v16f s[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const f16x8 kf = *reinterpret_cast<const f16x8 *>(lds[buf][0] + (kb * 32 + l32) * 256 + ((2 * m) ^ xk) * 16);
                s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[m], m == 0 ? zero : s[kb], 0, 0, 0);
            }
        }
        if (valid < kKeys) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (kb * 32 + 8 * (r / 4) + 4 * lh + r % 4 >= valid) s[kb][r] = -__builtin_inff();
        }
        float mx = s[0][0];
#pragma unroll
        for (int i = 1; i < 32; ++i) mx = __builtin_fmaxf(mx, s[i / 16][i % 16]);
        mx = max_halves(mx) * c;
        if (__builtin_amdgcn_ballot_w64(mx > m_ref) != 0) {
            const float m_new = __builtin_fmaxf(m_ref, mx);
            const float shift_new = m_new == -__builtin_inff() ? 0.0f : (__builtin_fabsf(m_new) < kExactShift ? kProbLog2 : 0.0f) - m_new;
            const float alpha = m_new == m_ref ? 1.0f : m_ref == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(shift_new - shift);
            m_ref = m_new;
            shift = shift_new;
            l *= alpha;
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[t][r] *= alpha;
        }
        f16x8 pf[4];
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                f16x2 p;
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    p[i] = static_cast<_Float16>(__builtin_amdgcn_exp2f(__builtin_fmaf(s[g / 2][(g % 2) * 8 + e + i], c, shift)));
                l = __builtin_amdgcn_fdot2(p, f16x2{static_cast<_Float16>(1.0f), static_cast<_Float16>(1.0f)}, l, false);
                pf[g][e] = p[0];
                pf[g][e + 1] = p[1];
            }
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const uint8_t *p = lds[buf][1] + v_read + 64 * (t ^ rr) + 16 * g * 256;
                const f16x4 lo = read_transposed(p), hi = read_transposed(p + 8 * 256);
                const f16x8 vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pf[g], o[t], 0, 0, 0);
            }
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
    }
    const float inv = 1.0f / sum_halves(l);
    if (q0 + l32 < a.lq) {
        __half *dst = a.out + batch * a.o_batch + head * a.o_head + static_cast<int64_t>(q0 + l32) * a.o_row + 4 * lh;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                f16x4 h;
#pragma unroll
                for (int e = 0; e < 4; ++e) h[e] = static_cast<_Float16>(o[t][4 * j + e] * inv);
                *reinterpret_cast<f16x4 *>(dst + 32 * t + 8 * j) = h;
            }
    }
#endif
}

// ---------------------------------------------------------------- q/k norm and rotary embedding

// RMS-norm over the whole row (fp32 statistics, rounded to fp16, times the fp16 weight, rounded again) and, with ROPE,
// the rotation of consecutive element pairs by the token's complex table row (fp32, rounded to fp16): modules/
// attention.py:149-205 of the reference.  One wave per row, the row in registers; blockIdx.y picks one of two matrices
// (q and k of a self-attention), which share a launch.
struct NormRopeArgs {
    const __half *x[2];
    const __half *w[2];
    __half *out[2];
    int64_t ldx[2];
    const f32x4 *table; /* (cos, sin) pairs, head_dim / 2 per position */
    int rows, k, head_dim, positions; /* row r is at position r % positions */
    float eps;
};

constexpr int kNormRows = 4;

template <int NCH, bool ROPE>
__global__ __launch_bounds__(kNormRows * 64) void norm_rope_kernel(NormRopeArgs a) {
    const int lane = threadIdx.x & 63, which = blockIdx.y;
    const int row = blockIdx.x * kNormRows + (threadIdx.x >> 6);
    if (row >= a.rows) return;
    const u32x4 *src = reinterpret_cast<const u32x4 *>(a.x[which] + row * a.ldx[which]), *wp = reinterpret_cast<const u32x4 *>(a.w[which]);
    u32x4 *dst = reinterpret_cast<u32x4 *>(a.out[which] + static_cast<int64_t>(row) * a.k);
    u32x4 v[NCH];
    float sum = 0.0f;
#pragma unroll
    for (int c = 0; c < NCH; ++c) v[c] = c * 512 + lane * 8 < a.k ? src[c * 64 + lane] : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const uint32_t words[4] = {v[c].x, v[c].y, v[c].z, v[c].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const f16x2 h = __builtin_bit_cast(f16x2, words[i]);
            const float lo = static_cast<float>(h[0]), hi = static_cast<float>(h[1]);
            sum = __builtin_fmaf(lo, lo, sum);
            sum = __builtin_fmaf(hi, hi, sum);
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    const float r = 1.0f / sqrtf(sum / static_cast<float>(a.k) + a.eps);
    const f32x4 *table = a.table + static_cast<int64_t>(ROPE ? row % a.positions : 0) * (a.head_dim / 4);
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int k0 = c * 512 + lane * 8;
        if (k0 >= a.k) continue;
        const u32x4 w4 = wp[c * 64 + lane];
        const uint32_t words[4] = {v[c].x, v[c].y, v[c].z, v[c].w}, w[4] = {w4.x, w4.y, w4.z, w4.w};
        uint32_t y[4];
        f32x4 cs[2];
        if (ROPE) {
            const int p = (k0 % a.head_dim) / 4;
            cs[0] = table[p];
            cs[1] = table[p + 1];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const f16x2 h = __builtin_bit_cast(f16x2, words[i]), wh = __builtin_bit_cast(f16x2, w[i]);
            f16x2 n = {static_cast<_Float16>(static_cast<float>(h[0]) * r), static_cast<_Float16>(static_cast<float>(h[1]) * r)};
            n = n * wh;
            if (ROPE) {
                const float re = static_cast<float>(n[0]), im = static_cast<float>(n[1]), co = cs[i / 2][2 * (i % 2)], si = cs[i / 2][2 * (i % 2) + 1];
                n[0] = static_cast<_Float16>(re * co - im * si);
                n[1] = static_cast<_Float16>(re * si + im * co);
            }
            y[i] = __builtin_bit_cast(uint32_t, n);
        }
        dst[c * 64 + lane] = u32x4{y[0], y[1], y[2], y[3]};
    }
}

// The parts of an RMS-norm around its row means, whose sum keeps the order of the framework that takes it, so that the result is the tensor
// operations' bit for bit; their other passes over the rows -- conversion, square, two products, two roundings -- become two.  A thread takes
// eight elements.  Bound by memory (4.6 ... 5.4 TB/s): 4680 x 1536, two matrices, squares 16 us and products as floats 17, one matrix's
// products as fp16 6; the tensor operations take 36, 75 and 30.
struct RowScaleArgs {
    const __half *x[2];
    const float *r[2];  /* null: squares */
    const __half *w[2];
    void *out[2];
    int64_t ldx[2];
    int64_t pieces; /* of eight elements, of a matrix */
    int row_pieces;
};

template <bool SQUARES, bool OUT_F32>
__global__ __launch_bounds__(256) void row_scale_product_kernel(RowScaleArgs a) {
    const int which = blockIdx.y;
    const int64_t at = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (at >= a.pieces) return;
    const int64_t row = a.pieces <= INT32_MAX ? static_cast<int>(at) / a.row_pieces : at / a.row_pieces;
    const int piece = static_cast<int>(at - row * a.row_pieces);
    const f16x8 v = *reinterpret_cast<const f16x8 *>(a.x[which] + row * a.ldx[which] + piece * 8);
    float y[8];
    if (SQUARES) {
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = static_cast<float>(v[e]) * static_cast<float>(v[e]);
    } else {
        const float r = a.r[which][row];
        const f16x8 w = *reinterpret_cast<const f16x8 *>(a.w[which] + piece * 8);
        f16x8 n;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float p = static_cast<float>(v[e]) * r;
            asm("" : "+v"(p)); /* (rounded to fp32 first: no product that is rounded to fp16 at once) */
            n[e] = static_cast<_Float16>(p);
        }
        n *= w;
        if (!OUT_F32) {
            *reinterpret_cast<f16x8 *>(static_cast<__half *>(a.out[which]) + at * 8) = n;
            return;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = static_cast<float>(n[e]);
    }
    f32x4 *out = reinterpret_cast<f32x4 *>(static_cast<float *>(a.out[which]) + at * 8);
    out[0] = f32x4{y[0], y[1], y[2], y[3]};
    out[1] = f32x4{y[4], y[5], y[6], y[7]};
}

// A modulation behind an fp32 LayerNorm: conversion, product and sum of the tensor operations in one pass (4680 x 1536: 26 -> 8 us).
__global__ __launch_bounds__(256) void modulate_rows_kernel(const f32x4 *__restrict__ y, const f16x8 *__restrict__ a, const f16x8 *__restrict__ b,
                                                            f16x8 *__restrict__ out, int64_t pieces, int row_pieces) {
    const int64_t at = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (at >= pieces) return;
    const int piece = pieces <= INT32_MAX ? static_cast<int>(at) % row_pieces : static_cast<int>(at % row_pieces);
    const f32x4 lo = y[2 * at], hi = y[2 * at + 1];
    f16x8 h, one;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        h[e] = static_cast<_Float16>(e < 4 ? lo[e] : hi[e - 4]);
        one[e] = static_cast<_Float16>(1.0f);
    }
    out[at] = h * (one + a[piece]) + b[piece]; /* packed fp16 operations, each rounded (no contraction) */
}

// The table of rotations: position (f, h, w), pair i -> cos and sin of coordinate * 10000^(-2j / dim) for the axis and
// the place j within it that pair i belongs to (frames take head_dim - 2 * (head_dim / 3) channels, rows and columns
// head_dim / 3 each; modules/embedding.py:114-157), in double, rounded to float.  One thread per entry.
__global__ __launch_bounds__(256) void rope_table_kernel(float2 *__restrict__ table, int head_dim, int f, int h, int w) {
    const int third = head_dim / 3, pairs_hw = third / 2, pairs_f = (head_dim - 2 * third) / 2, pairs = pairs_f + 2 * pairs_hw;
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= static_cast<int64_t>(f) * h * w * pairs) return;
    const int pair = static_cast<int>(idx % pairs);
    const int64_t pos = idx / pairs;
    int j = pair, dim = head_dim - 2 * third, coord = static_cast<int>(pos / (static_cast<int64_t>(h) * w));
    if (pair >= pairs_f) {
        j = pair - pairs_f;
        dim = third;
        coord = static_cast<int>(pos / w % h);
        if (j >= pairs_hw) {
            j -= pairs_hw;
            coord = static_cast<int>(pos % w);
        }
    }
    const double angle = coord * (1.0 / pow(10000.0, 2.0 * j / dim));
    double s, c;
    sincos(angle, &s, &c);
    table[idx] = make_float2(static_cast<float>(c), static_cast<float>(s));
}

// The timestep embedding (modules/embedding.py:7-10): cos, then sin, of the `half` angles t * 10000^(-i / half), in double,
// rounded through float to fp16 as the tensor conversion does.  One thread per angle: a single launch bounds it (as tensor
// operations twelve of them, 25 us of GPU time and the host's time for each).
__global__ __launch_bounds__(256) void timestep_embedding_kernel(const double *__restrict__ t, __half *__restrict__ out, int64_t batch, int half) {
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= batch * half) return;
    const int i = static_cast<int>(idx % half);
    const int64_t b = idx / half;
    double s, c;
    sincos(t[b] * pow(10000.0, -static_cast<double>(i) / half), &s, &c);
    out[b * 2 * half + i] = __float2half_rn(static_cast<float>(c));
    out[b * 2 * half + half + i] = __float2half_rn(static_cast<float>(s));
}

template <int NCH>
void launch_norm_rope_nch(const NormRopeArgs &a, int matrices, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>(ceil_div(a.rows, kNormRows)), static_cast<unsigned>(matrices)), block(kNormRows * 64);
    if (a.table != nullptr)
        hipLaunchKernelGGL((norm_rope_kernel<NCH, true>), grid, block, 0, s, a);
    else
        hipLaunchKernelGGL((norm_rope_kernel<NCH, false>), grid, block, 0, s, a);
}

}  // namespace

int launch_norm_rope(const __half *const *x, const int64_t *ldx, const __half *const *w, __half *const *out, int matrices, int64_t rows, int64_t K,
                     float eps, const float *table, int64_t head_dim, int64_t positions, hipStream_t s) {
    NormRopeArgs a = {};
    for (int i = 0; i < matrices; ++i) a.x[i] = x[i], a.ldx[i] = ldx[i], a.w[i] = w[i], a.out[i] = out[i];
    a.table = reinterpret_cast<const f32x4 *>(table);
    a.rows = static_cast<int>(rows), a.k = static_cast<int>(K), a.head_dim = static_cast<int>(head_dim), a.positions = static_cast<int>(positions);
    a.eps = eps;
    const int64_t nch = ceil_div(K, 512);
    (nch <= 1 ? launch_norm_rope_nch<1> : nch <= 3 ? launch_norm_rope_nch<3> : nch <= 6 ? launch_norm_rope_nch<6> : nch <= 10 ? launch_norm_rope_nch<10> :
     launch_norm_rope_nch<16>)(a, matrices, s);
    return check_launch("norm_rope_kernel");
}

static int launch_row_product(const RowScaleArgs &a, bool squares, bool out_f32, int matrices, hipStream_t s) {
    const int64_t blocks = ceil_div(a.pieces, 256);
    if (blocks > INT32_MAX) return fail(VDMQ_ESHAPE, "%lld elements need more workgroups than one launch can hold", (long long)(a.pieces * 8));
    const dim3 grid(static_cast<unsigned>(blocks), static_cast<unsigned>(matrices));
    if (squares) hipLaunchKernelGGL((row_scale_product_kernel<true, true>), grid, dim3(256), 0, s, a);
    else if (out_f32) hipLaunchKernelGGL((row_scale_product_kernel<false, true>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((row_scale_product_kernel<false, false>), grid, dim3(256), 0, s, a);
    return check_launch("row_scale_product_kernel");
}

int launch_row_squares(const __half *const *x, const int64_t *ldx, float *const *out, int matrices, int64_t rows, int64_t K, hipStream_t s) {
    RowScaleArgs a = {};
    for (int i = 0; i < matrices; ++i) a.x[i] = x[i], a.ldx[i] = ldx[i], a.out[i] = out[i];
    a.row_pieces = static_cast<int>(K / 8), a.pieces = rows * a.row_pieces;
    return launch_row_product(a, true, true, matrices, s);
}

int launch_scale_rows(const __half *const *x, const int64_t *ldx, const float *const *r, const __half *const *w, void *const *out, bool out_f32, int matrices,
                      int64_t rows, int64_t K, hipStream_t s) {
    RowScaleArgs a = {};
    for (int i = 0; i < matrices; ++i) a.x[i] = x[i], a.ldx[i] = ldx[i], a.r[i] = r[i], a.w[i] = w[i], a.out[i] = out[i];
    a.row_pieces = static_cast<int>(K / 8), a.pieces = rows * a.row_pieces;
    return launch_row_product(a, false, out_f32, matrices, s);
}

int launch_modulate_rows(const float *y, const __half *a, const __half *b, __half *out, int64_t rows, int64_t K, hipStream_t s) {
    const int64_t pieces = rows * (K / 8), blocks = ceil_div(pieces, 256);
    if (blocks > INT32_MAX) return fail(VDMQ_ESHAPE, "%lld elements need more workgroups than one launch can hold", (long long)(rows * K));
    hipLaunchKernelGGL(modulate_rows_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, reinterpret_cast<const f32x4 *>(y), reinterpret_cast<const f16x8 *>(a),
                       reinterpret_cast<const f16x8 *>(b), reinterpret_cast<f16x8 *>(out), pieces, static_cast<int>(K / 8));
    return check_launch("modulate_rows_kernel");
}

int launch_rope_table(float *table, int64_t head_dim, int64_t f, int64_t h, int64_t w, hipStream_t s) {
    const int64_t third = head_dim / 3, entries = f * h * w * ((head_dim - 2 * third) / 2 + third / 2 * 2);
    if (entries == 0) return VDMQ_OK;
    hipLaunchKernelGGL(rope_table_kernel, dim3(static_cast<unsigned>(ceil_div(entries, 256))), dim3(256), 0, s, reinterpret_cast<float2 *>(table),
                       static_cast<int>(head_dim), static_cast<int>(f), static_cast<int>(h), static_cast<int>(w));
    return check_launch("rope_table_kernel");
}

int launch_timestep_embedding(const double *t, __half *out, int64_t batch, int64_t half, hipStream_t s) {
    hipLaunchKernelGGL(timestep_embedding_kernel, dim3(static_cast<unsigned>(ceil_div(batch * half, 256))), dim3(256), 0, s, t, out, batch,
                       static_cast<int>(half));
    return check_launch("timestep_embedding_kernel");
}

int launch_attention(const AttentionArgs &x, hipStream_t s) {
    AttnArgs a;
    a.q = x.q, a.k = x.k, a.v = x.v, a.out = x.out;
    a.q_row = x.q_stride[0], a.q_head = x.q_stride[1], a.q_batch = x.q_stride[2];
    a.k_row = x.k_stride[0], a.k_head = x.k_stride[1], a.k_batch = x.k_stride[2];
    a.v_row = x.v_stride[0], a.v_head = x.v_stride[1], a.v_batch = x.v_stride[2];
    a.o_row = x.o_stride[0], a.o_head = x.o_stride[1], a.o_batch = x.o_stride[2];
    a.heads = static_cast<int>(x.heads), a.lq = static_cast<int>(x.lq), a.lk = static_cast<int>(x.lk);
    a.scale_log2 = x.scale * 1.4426950408889634f;
    // Four waves per workgroup, two workgroups per CU, unless a head's K and V (512 bytes per key) exceed an XCD's 4 MiB of
    // L2: then eight waves, one workgroup per CU, which read them half as often.  Measured, four / eight: 32760 x 32760
    // (12 heads) 6510 / 6210 us; 3613 x 3613 (40) 321 / 346, 1560 x 1560 (12) 38 / 50, 32760 x 512 (12) 140 / 145.
    const bool wide = x.lk > 8192;
    const int waves = wide ? 8 : 4;
    a.q_tiles = static_cast<int>(ceil_div(x.lq, waves * 32));
    a.tiles = x.batch * x.heads * a.q_tiles;
    const int64_t grid = ceil_div(a.tiles, 8) * 8;
    if (grid > INT32_MAX) return fail(VDMQ_ESHAPE, "attention over %lld tiles of queries needs more workgroups than one launch can hold", (long long)a.tiles);
    if (wide)
        hipLaunchKernelGGL(attention_kernel<8>, dim3(static_cast<unsigned>(grid)), dim3(512), 0, s, a);
    else
        hipLaunchKernelGGL(attention_kernel<4>, dim3(static_cast<unsigned>(grid)), dim3(256), 0, s, a);
    return check_launch("attention_kernel");
}

}  // namespace vdmq
