// Dynamic per-token A4 quantizer for gfx950: one pass over X.
//
// One 64-lane wave owns one token row.  The row is read once with 128-bit
// loads and kept in registers; the absmax is reduced on the packed fp16 bit
// patterns (exact, order-free); the scale is rounded to fp16; every element is
// multiplied by the fp32 reciprocal of that fp16 scale, rounded half-to-even
// and saturated to [-8, 7]; eight results are packed into one 32-bit word and
// stored row-major (element e of a word in nibble e).
//
// Arithmetic contract (IEEE reading of vdm_w4a4_kernel.cu:459-481, 95-102,
// 319-329 of the reference): see quantize_word below, whose literal form serves
// rows that contain NaN/Inf or whose fp16 scale is zero/non-finite; all other
// rows take a shorter, bit-identical sequence.
#include "vdmq_rowops.h"

namespace vdmq {
namespace {

// q = sat_s4(rni(float(x) * rscale)) for the eight elements of `v`, element e in nibble e.  LITERAL: also for rows with
// NaN or Inf and for a scale whose reciprocal is not finite (cvt.rni.s32.f32 + cvt.pack.sat.s4: NaN -> 0, saturate); the
// other form is for finite inputs and a finite non-zero scale.  t = clamp(v) is rounded to an integer by adding 1.5*2^23 + 8 (the fp32 adder rounds half to
// even on the unit grid there), which leaves u = rni(t) + 8 in [0, 15] in the
// low bits of the sum: bits = 0x4B400000 + u.  Eight sums are combined with
// shift-adds; the constant parts add up to 0x4B400000 * 0x11111111 (mod 2^32)
// and are removed at the end; u ^ 8 is the two's complement nibble.
constexpr float kMagic = 12582920.0f; /* 1.5 * 2^23 + 8 */
constexpr uint32_t kMagicSum = static_cast<uint32_t>(0x4B400000ull * 0x11111111ull);

template <bool LITERAL>
__device__ __forceinline__ uint32_t quantize_word(u32x4 v, float rscale) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    uint32_t acc = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const f16x2 h = __builtin_bit_cast(f16x2, w[i]);
        // fma(x, r, +0) = fl(x * r) (a product of -0 becomes +0, which rounds to the same integer): one
        // v_fma_mix_f32 reading the fp16 value, instead of a conversion and a multiplication
        float t0 = __builtin_fmaf(static_cast<float>(h[0]), rscale, 0.0f), t1 = __builtin_fmaf(static_cast<float>(h[1]), rscale, 0.0f);
        if (LITERAL) {
            t0 = t0 == t0 ? t0 : 0.0f;
            t1 = t1 == t1 ? t1 : 0.0f;
        }
        t0 = __builtin_amdgcn_fmed3f(t0, -8.0f, 7.0f);
        t1 = __builtin_amdgcn_fmed3f(t1, -8.0f, 7.0f);
        acc += __float_as_uint(t0 + kMagic) << (8 * i);
        acc += __float_as_uint(t1 + kMagic) << (8 * i + 4);
    }
    return (acc - kMagicSum) ^ 0x88888888u;
}

// The absmax of gelu_tanh over a row from the row's own extremes, without evaluating it on every element: on fp16
// values x >= 0 gelu_tanh_pair does not decrease with x, and on negative ones its magnitude stays below kGeluNegative
// (0.17, near x = -0.75).  So for a finite row whose largest element maps to at least that, the image of the largest
// element is the answer (fp16 bits in m16, the same in every lane); false for any other row.  Both properties of the
// fp16 function are checked over its whole table by the tests.  What it buys: the scale is known before the first
// evaluation, so the evaluation moves behind the loads of the next row that are issued during the conversion.
constexpr uint32_t kGeluNegative = 0x3180u; /* 0.1719 */

__device__ __forceinline__ uint32_t pk_max_i16(uint32_t a, uint32_t b) {
    typedef short i16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(i16x2, a), __builtin_bit_cast(i16x2, b)));
}

template <int NCH>
__device__ __forceinline__ bool gelu_row_absmax(const u32x4 (&v)[NCH], uint32_t &m16) {
    uint32_t up = 0, neg = 0; /* as signed numbers fp16 bits order the values >= 0, as unsigned ones the magnitudes of the negative */
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const uint32_t w[4] = {v[c].x, v[c].y, v[c].z, v[c].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            up = pk_max_i16(up, w[i]);
            neg = pk_max_u16(neg, w[i]);
        }
    }
    const uint32_t largest = wave_max((up & 0xFFFFu) > (up >> 16) ? (up & 0xFFFFu) : (up >> 16));
    const bool neg_inf_nan = __builtin_amdgcn_ballot_w64((neg & 0xFFFFu) >= 0xFC00u || neg >= 0xFC000000u) != 0;
    m16 = gelu_tanh_pair(largest) & 0xFFFFu;
    return __builtin_amdgcn_readfirstlane(largest < 0x7C00u && !neg_inf_nan && m16 >= kGeluNegative ? 1 : 0) != 0;
}

constexpr int kRowsPerBlock = 4; /* one wave per row */

template <bool STREAM>
__device__ __forceinline__ void store_word(uint32_t *p, uint32_t w) {
    if (STREAM)
        __builtin_nontemporal_store(w, p);
    else
        *p = w;
}

// Quantize a row held in registers (v[c] = elements 512c + 8*lane ... +7, zero
// beyond K): absmax, fp16 scale, nibbles, stores.
template <int NCH, bool STREAM_OUT>
__device__ __forceinline__ void quantize_held_row(const u32x4 (&v)[NCH], int lane, int64_t row, int Kp, float clip,
                                                  uint8_t *__restrict__ qact, __half *__restrict__ scale_h) {
    uint32_t m2 = 0;
#pragma unroll
    for (int c = 0; c < NCH; ++c) m2 = absmax_bits(v[c], m2);
    uint32_t m16 = (m2 & 0xFFFFu) > (m2 >> 16) ? (m2 & 0xFFFFu) : (m2 >> 16);
    m16 = wave_max(m16);

    uint32_t *dst = reinterpret_cast<uint32_t *>(qact + row * (Kp / 2));
    __half sh;
    bool fast = m16 < 0x7C00u; /* every element finite */
    if (fast) {
        sh = scale_from_absmax(half_bits_to_float(m16), clip);
        fast = scale_is_ordinary(sh);
    }
    if (fast) {
        const float rscale = reciprocal_of_scale(__half2float(sh));
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int k0 = c * 512 + lane * 8;
            if (k0 < Kp) store_word<STREAM_OUT>(dst + c * 64 + lane, quantize_word<false>(v[c], rscale));
        }
    } else {
        float mx = 0.0f;
#pragma unroll
        for (int c = 0; c < NCH; ++c) mx = absmax_exact(v[c], mx);
        // fmaxf-style wave reduction (no NaN can be held in mx)
        mx = wave_max(mx);
        sh = scale_from_absmax(mx, clip);
        const float rscale = 1.0f / __half2float(sh);
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int k0 = c * 512 + lane * 8;
            if (k0 < Kp) store_word<STREAM_OUT>(dst + c * 64 + lane, quantize_word<true>(v[c], rscale));
        }
    }
    if (lane == 0) scale_h[row] = sh;
}

// The same, written as bf6 blocks (the operand form of the bf6 GEMM, see vdmq_bf6.hip): per row and 32
// consecutive k = 64 * kb + 32 * h + e one 192-bit string of six-bit E3M2 codes, stored by panels of 8 rows
// (bf6_piece in vdmq_internal.h).  A lane holds 8 consecutive k per chunk, a quarter of a string.  Four chunks at a time
// are scaled and go through the conversion instruction as they lie (v_cvt_scalef32_2xpk16_bf6_f32 with a scale of 16: the
// block holds q / 16, an E3M2 value for every q of [-8, 8]); its 192 bits are then four 48-bit quarters of four different
// strings, which are put together in LDS.  (Bringing 32 consecutive k into one lane first, as fp16 through LDS, takes
// 2.7 times the LDS traffic, an LDS round trip in front of every conversion and 34 KiB of LDS more per workgroup, with
// which two fit a CU.  Measured, that way / this way, with the reductions below on the VALU: 32760 x 1536 plain 24.2 /
// 22.8 us, GELU 36 / 30, LayerNorm 41 / 29; 27280 x 3072 LayerNorm 64 / 50; 75637 x 5120 GELU 205 / 169, LayerNorm
// 239 / 222; the streaming floor at 6.3 TB/s is 22, 37 and 169 us.)
// The instruction also rounds: E3M2's grid is 1/16 up to 8/16, so round-to-nearest-even of t / 16 onto it is the
// round-half-even of t the quantizer asks for, ties included (a code's last bit is the integer's).  Only |t| has to
// stay below 8.5, above -8.5 and t below 7.5; rows whose largest |t| is below 7.5 (a clip ratio above 0.934)
// skip the clamp, all others (NaN, Inf, a scale of zero, a small clip ratio) take it.  Rows of the last row-block beyond
// M stay unwritten (the GEMM never stores them); K is padded to 128 with zeros.
constexpr int kPanelRows = 8;        /* rows of a panel of the bf6 blocks */
constexpr int kStringsPerGroup = 64; /* 2048 k = 64 strings of 32 k per row and group */
constexpr int kStringBytes = 24;
// 16 bytes of padding per row: sixteen lanes that read 8 bytes each of eight rows and two strings meet 32 banks
constexpr int kStringRowBytes = kStringsPerGroup * kStringBytes + 16;

// A workgroup owns ROWS rows: a panel or half of one, a wave per row (bf6_split says which), or a quarter, four waves per row (rows_in_parts).
// The parts of a panel go to one XCD, one after the other, whose L2 joins their runs (blocks are dealt to the XCDs in turn): the b-th of `groups`
// groups of rows.
template <int ROWS>
__device__ __forceinline__ int bf6_group(int b, int groups) {
    constexpr int P = kPanelRows / ROWS;
    return P == 1 || (b | (8 * P - 1)) >= groups ? b : (b & ~(8 * P - 1)) | (b & 7) * P | (b >> 3 & (P - 1));
}
template <int ROWS>
struct Bf6Scratch { /* LDS of one workgroup: the strings of one group; two copies in turn: one barrier per group is enough */
    uint8_t strings[2][ROWS][kStringRowBytes];
};

// `valid`: the wave's row exists (a workgroup's waves all run this function -- it synchronises them --
// the ones past M on a copy of the last row, storing nothing).  PARTS > 1: the row is shared by PARTS waves, `part` is this one's (its chunks and its
// staging copies are its own) and `part_max` takes their maxima.  `refill(c)` runs once chunk c of the
// row has been converted and its registers are free: a workgroup that walks several
// row groups loads the next row's chunk there, so those loads overlap the rest of this row's
// conversion.  `phase` counts the groups this workgroup has staged (it picks the staging copy).
// Which row lengths take the walking form (a resident grid whose workgroups take row groups in turn, the next group's
// loads in flight under this group's conversion): rows longer than 9216, of which the registers hold one workgroup per
// CU only (27280 x 12288: 155 us walking, 171 not; 27280 x 14336: 184 / 199), and rows of at most 2048, whose groups are
// too little work for a workgroup of their own (K = 512...1536: +8...17 % at 32760 and 75600 rows).  In between several
// workgroups share a CU and overlap by themselves (32760 x 8960: 133 walking, 130 not).
constexpr bool bf6_walks(int nch) { return nch >= 19 || nch <= 4; }
// Dynamic LDS a launch asks for beside the strings, to keep a third workgroup off the CU: eight-wave workgroups of
// 10 KiB rows stream best with two of them in flight per CU once the rows are many (plain, with two / with three, us:
// 75637 x 5120 162 / 171, x 4096 135 / 141, x 3584 114.5 / 117.4; 32760 x 5120 71 / 73; the streaming floor of the first is 169
// at 6.3 TB/s).  Not so below: 8192 x 4608 18.6 / 17.9, 8192 x 3136 13.7 / 12.1, 75637 x 3136 106 / 101.  The shorter rows and
// the fused producers want every wave they can get (27280 x 3072: 37.1 us with three or more, 39.3 with two; 75637 x 5120
// with the GELU 171 / 175).
constexpr int bf6_spare_lds(int nch, int act) { return nch > 6 && nch <= 10 && act == VDMQ_ACT_NONE ? 30000 : 0; }
// Whether a fused activation is evaluated behind the row's absmax (gelu_row_absmax), chunk by chunk during the
// conversion: with long rows few waves share a SIMD and what they compute between the arrival of a row and its
// conversion runs with no load in flight.  Measured, in front / behind: 27280 x 14336 268 / 214 us, 75600 x 13824 636 /
// 548, 32760 x 8960 193 / 152; short rows have the waves to overlap and pay for the second maximum: 75637 x 5120 176 /
// 180, 27280 x 3072 43 / 45.5.  (The chunk counts that rows run on go from 14 to 18: this is K > 7168.)
constexpr bool bf6_late_act(int nch) { return nch >= 17; }
struct Bf6PartMax {
    float mx;
    int finite;
};
struct NoRefill {
    __device__ __forceinline__ void operator()(int) const {}
};
template <int NCH, int ACT, int ROWS, int PARTS, class Refill>
__device__ __forceinline__ void quantize_held_row_bf6(u32x4 (&v)[NCH], int lane, int wave, int64_t row0, bool valid, int M, int Kb,
                                                      float clip, uint8_t *__restrict__ blocks, __half *__restrict__ scale_h,
                                                      bool stream_out, Bf6Scratch<ROWS> &lds, int &phase, Refill &&refill, int part = 0,
                                                      Bf6PartMax *part_max = nullptr) {
    // `late`: the activation is evaluated chunk by chunk below, in front of the conversion (see gelu_row_absmax)
    uint32_t m16 = 0;
    const bool late = ACT == VDMQ_ACT_GELU_TANH && gelu_row_absmax<NCH>(v, m16);
    if (!late) {
        uint32_t m2 = 0;
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            if (ACT != VDMQ_ACT_NONE) v[c] = apply_act<ACT>(v[c]);
            m2 = absmax_bits(v[c], m2);
        }
        m16 = (m2 & 0xFFFFu) > (m2 >> 16) ? (m2 & 0xFFFFu) : (m2 >> 16);
        m16 = wave_max(m16);
    }
    bool finite = m16 < 0x7C00u;
    float mx = half_bits_to_float(m16);
    if (!finite) {
        mx = 0.0f;
#pragma unroll
        for (int c = 0; c < NCH; ++c) mx = absmax_exact(v[c], mx);
        mx = wave_max(mx);
    }
    if constexpr (PARTS > 1) { /* the row's other parts */
        if (lane == 0) part_max[part * ROWS + wave] = {mx, finite ? 1 : 0};
        __syncthreads();
#pragma unroll
        for (int p = 0; p < PARTS; ++p) {
            const Bf6PartMax other = part_max[p * ROWS + wave];
            mx = __builtin_fmaxf(mx, other.mx);
            finite = finite && other.finite != 0;
        }
    }
    const __half sh = scale_from_absmax(mx, clip);
    const bool fast = __builtin_amdgcn_readfirstlane(finite && scale_is_ordinary(sh) ? 1 : 0) != 0;
    float rscale = 0.0f;
    if (fast)
        rscale = reciprocal_of_scale(__half2float(sh));
    else
        rscale = 1.0f / __half2float(sh);
    // (of a finite row the largest |x| gives the largest |t|: the products round monotonically.  The same in every lane: a
    // scalar branch)
    const bool clamp_u = __builtin_amdgcn_readfirstlane(fast && mx * rscale < 7.5f ? 0 : 1) != 0;
    if (lane == 0 && valid && (PARTS == 1 || part == 0)) scale_h[row0 + wave] = sh;

    const int kblocks = Kb / 64;
    // the lane's quarter of a string: string lane / 4 of each chunk's sixteen, bytes 6p ... 6p + 5, p = lane % 4.  Those
    // are a word and a half word, the word first for even p and last for odd p (so that it is aligned).
    const bool odd = (lane & 1) != 0;
    const uint32_t string0 = (lane >> 2) * kStringBytes + (lane & 3) * 6, off32 = string0 + (odd ? 2 : 0), off16 = string0 + (odd ? 0 : 4);
    // the thread's share of the cooperative store: string t / ROWS of row t % ROWS -- ROWS consecutive threads write
    // the rows' parts of one string slot, contiguous bytes: 128 (and 64) of a whole panel
    const int t = wave * kWaveSize + lane, srow = t % ROWS, sidx = t / ROWS;
    const int64_t grow = row0 + srow;
    constexpr int NG = (NCH + 3) / 4;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        // the conversion takes the even elements from one operand and the odd ones from the other: the low and high halves
        // of the words as they lie
        f32x16 even, odds;
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {
            const int c = 4 * g + cc;
            u32x4 x4 = c < NCH ? v[c < NCH ? c : 0] : u32x4{0u, 0u, 0u, 0u};
            if (c < NCH && late) x4 = apply_act<ACT>(x4);
            const uint32_t w[4] = {x4.x, x4.y, x4.z, x4.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f16x2 h = __builtin_bit_cast(f16x2, w[i]);
                even[cc * 4 + i] = c < NCH ? __builtin_fmaf(static_cast<float>(h[0]), rscale, 0.0f) : 0.0f;
                odds[cc * 4 + i] = c < NCH ? __builtin_fmaf(static_cast<float>(h[1]), rscale, 0.0f) : 0.0f;
            }
        }
        if (clamp_u) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                // NaN -> 0, saturate (cvt.rni + cvt.pack.sat of the reference); the literal rows come through here
                even[i] = __builtin_amdgcn_fmed3f(even[i] == even[i] ? even[i] : 0.0f, -8.0f, 7.0f);
                odds[i] = __builtin_amdgcn_fmed3f(odds[i] == odds[i] ? odds[i] : 0.0f, -8.0f, 7.0f);
            }
        }
        const u32x6 str = to_bf6(even, odds);
#pragma unroll
        for (int cc = 0; cc < 4; ++cc)
            if (4 * g + cc < NCH) refill(4 * g + cc);
        // per-lane stores would scatter pieces over 64 cache lines per instruction (measured: 2x slower than the
        // HBM-bound int4 quantizer): collect the workgroup's strings in LDS -- its rows are a panel or part of one, whose
        // 128-byte and 64-byte runs of one k-block are adjacent in memory
        const int copy = phase & 1;
        ++phase;
        uint8_t *mine = lds.strings[copy][wave];
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {
            if (4 * g + cc >= NCH) continue; /* (beyond Kb <= 512 * NCH: nobody reads those strings) */
            // chunk cc's 48 bits of str: (word, low half of the next) for even cc, (high half of a word, the next) for odd
            const uint32_t lo = str[cc / 2 * 3 + cc % 2], hi = str[cc / 2 * 3 + cc % 2 + 1];
            const uint32_t joined = __builtin_amdgcn_alignbyte(hi, lo, 2);
            if (cc % 2 == 0) {
                *reinterpret_cast<uint32_t *>(mine + cc * 16 * kStringBytes + off32) = odd ? joined : lo;
                *reinterpret_cast<uint16_t *>(mine + cc * 16 * kStringBytes + off16) = static_cast<uint16_t>(odd ? lo : hi);
            } else {
                *reinterpret_cast<uint32_t *>(mine + cc * 16 * kStringBytes + off32) = odd ? hi : joined;
                *reinterpret_cast<uint16_t *>(mine + cc * 16 * kStringBytes + off16) = static_cast<uint16_t>((odd ? lo : hi) >> 16);
            }
        }
        __syncthreads(); /* also orders this group's writes after every thread's reads of the group before last */
        const int k0 = part * (NCH * 512) + 2048 * g + 32 * sidx;
        if (k0 < Kb && grow < M && (PARTS == 1 || 2048 * g + 32 * sidx < NCH * 512)) {
            const int kb = k0 >> 6, h = (k0 >> 5) & 1;
            const u32x2 *string = reinterpret_cast<const u32x2 *>(lds.strings[copy][srow] + sidx * kStringBytes);
            const u32x2 s0 = string[0], s1 = string[1], part_b = string[2];
            const u32x4 part_a = {s0.x, s0.y, s1.x, s1.y};
            u32x4 *dst_a = reinterpret_cast<u32x4 *>(blocks + bf6_piece(grow, kb, h, false, kblocks));
            u32x2 *dst_b = reinterpret_cast<u32x2 *>(blocks + bf6_piece(grow, kb, h, true, kblocks));
            if (stream_out) { /* the same for every thread of the launch */
                // (the empty statements keep the compiler from merging the two branches into plain stores)
                asm volatile("" ::: "memory");
                __builtin_nontemporal_store(part_a, dst_a);
                __builtin_nontemporal_store(part_b, dst_b);
                asm volatile("" ::: "memory");
            } else {
                *dst_a = part_a;
                *dst_b = part_b;
            }
        }
    }
}

// NCH = number of 512-element chunks (one 128-bit load per lane each) that
// cover the padded row.  STREAM_OUT: write the nibbles with non-temporal
// stores -- measured faster once the output no longer fits the 256 MB
// Infinity Cache (5.35 -> 5.9 TB/s at K = 13824, M = 75600), slower below.
// ACT: an elementwise activation applied to the row (in fp32, rounded to fp16)
// before it is quantized: the activation kernel between two linears, its write
// and the quantizer's re-read of its output are saved.
// FMT: 0 = native row-major int4 (Kp = K padded to the int8 GEMM's K step), 1 = bf6 blocks (Kp = K padded to 128)
// Registers decide how many workgroups share a CU with short rows: in 64 of them (NCH 1 and 2) four do, in 80 three.  A scalar wave
// number keeps the row addresses out of them there (32760 rows of 768 / 1024 / 2048 with the GELU 24.2 -> 22.8, 24.9 -> 24.3, 41.1 -> 38.8 us);
// with longer rows it costs time (3072 with the GELU 49.4 -> 54.1).  (The fused LayerNorm's longest form spills: fewer registers so, 0.95 ...
// 1.00 of the time for rows of 9216 ... 16384.)
template <int NCH, bool STREAM_OUT, int ACT, int FMT, int ROWS>
__global__ __launch_bounds__(ROWS * kWaveSize, FMT == 1 && NCH <= 2 ? 8 : FMT == 1 ? 2 : 1) void quantize_rows_kernel(
    const __half *__restrict__ x, int64_t ldx, int M, int K, int Kp, float clip, uint8_t *__restrict__ qact,
    __half *__restrict__ scale_h, int stream_out_bf6) {
    const int lane = threadIdx.x & (kWaveSize - 1), wave = FMT == 1 && NCH <= 4 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x >> 6;
    if constexpr (FMT == 1) {
        // The workgroup walks row groups blockIdx.x, blockIdx.x + gridDim.x, ...: with the launcher's grid
        // (what the chip holds at once) the loads of the next group's rows are in flight while this
        // group's rows are converted -- a long row leaves room for one workgroup per CU only, whose load and
        // convert phases would otherwise alternate.
        __shared__ __attribute__((aligned(16))) Bf6Scratch<ROWS> scratch;
        const int groups = (M + ROWS - 1) / ROWS;
        auto row_ptr = [&](int group) {
            const int64_t r = static_cast<int64_t>(bf6_group<ROWS>(group, groups)) * ROWS + wave;
            return reinterpret_cast<const u32x4 *>(x + (r < M ? r : M - 1) * ldx); /* waves past M stay, on a copy of the last row */
        };
        auto load = [&](const u32x4 *src, int c) {
            return c * 512 + lane * 8 < K ? __builtin_nontemporal_load(src + c * 64 + lane) : u32x4{0u, 0u, 0u, 0u};
        };
        int group = blockIdx.x, phase = 0;
        u32x4 v[NCH];
        const u32x4 *src = row_ptr(group);
#pragma unroll
        for (int c = 0; c < NCH; ++c) v[c] = load(src, c);
        for (; group < groups; group += gridDim.x) {
            const bool more = bf6_walks(NCH) && group + static_cast<int>(gridDim.x) < groups;
            const u32x4 *next = row_ptr(more ? group + gridDim.x : group);
            const int64_t row0 = static_cast<int64_t>(bf6_group<ROWS>(group, groups)) * ROWS;
            if (ACT != VDMQ_ACT_NONE && !bf6_late_act(NCH)) {
#pragma unroll
                for (int c = 0; c < NCH; ++c)
                    if (c * 512 + lane * 8 < K) v[c] = apply_act<ACT>(v[c]);
            }
            quantize_held_row_bf6<NCH, bf6_late_act(NCH) ? ACT : VDMQ_ACT_NONE, ROWS, 1>(v, lane, wave, row0, row0 + wave < M, M, Kp, clip, qact, scale_h, stream_out_bf6 != 0, scratch, phase,
                                            [&](int c) {
                                                if constexpr (bf6_walks(NCH))
                                                    if (more) v[c] = load(next, c);
                                            });
            if (!bf6_walks(NCH)) break; /* one row group per workgroup: several workgroups share a CU and overlap anyway */
        }
    } else {
        const int64_t row = static_cast<int64_t>(blockIdx.x) * ROWS + wave;
        if (row >= M) return;
        const u32x4 *src = reinterpret_cast<const u32x4 *>(x + row * ldx);
        u32x4 v[NCH];
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int k0 = c * 512 + lane * 8;
            v[c] = k0 < K ? apply_act<ACT>(__builtin_nontemporal_load(src + c * 64 + lane)) : u32x4{0u, 0u, 0u, 0u};
        }
        quantize_held_row<NCH, STREAM_OUT>(v, lane, row, Kp, clip, qact, scale_h);
    }
}

// The same for few rows, which a wave each would leave to a part of the chip, one long chain of loads, maximum and conversions per row: PARTS waves
// share a row, NCH chunks each, and exchange their maxima once.  Bound by that chain (512 x 5120: 4.4 us for 9 MB); no walking, and the
// activation goes in front, its absmax is the part's own.
template <int NCH, int ACT, int ROWS, int PARTS>
__global__ __launch_bounds__(ROWS * PARTS * kWaveSize) void quantize_row_parts_kernel(const __half *__restrict__ x, int64_t ldx, int M, int K, int Kp, float clip,
                                                                                      uint8_t *__restrict__ blocks, __half *__restrict__ scale_h) {
    __shared__ __attribute__((aligned(16))) Bf6Scratch<ROWS> scratch[PARTS];
    __shared__ Bf6PartMax part_max[PARTS * ROWS];
    const int lane = threadIdx.x & (kWaveSize - 1), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave = w % ROWS, part = w / ROWS;
    const int64_t row0 = static_cast<int64_t>(bf6_group<ROWS>(blockIdx.x, (M + ROWS - 1) / ROWS)) * ROWS, row = row0 + wave;
    const u32x4 *src = reinterpret_cast<const u32x4 *>(x + (row < M ? row : M - 1) * ldx) + part * (NCH * 64);
    u32x4 v[NCH];
#pragma unroll
    for (int c = 0; c < NCH; ++c) v[c] = (part * NCH + c) * 512 + lane * 8 < K ? __builtin_nontemporal_load(src + c * 64 + lane) : u32x4{0u, 0u, 0u, 0u};
    if (ACT != VDMQ_ACT_NONE) {
#pragma unroll
        for (int c = 0; c < NCH; ++c) v[c] = apply_act<ACT>(v[c]);
    }
    int phase = 0;
    quantize_held_row_bf6<NCH, VDMQ_ACT_NONE, ROWS, PARTS>(v, lane, wave, row0, row < M, M, Kp, clip, blocks, scale_h, false, scratch[part], phase, NoRefill{},
                                                           part, part_max);
}

// Chunk counts the fused LayerNorm kernel is instantiated for (launch_ln_impl picks the first that covers the row):
// with NCH chunks the row is longer than the next smaller count, so the chunks below that one are complete in every
// lane and need no bounds test.
constexpr int ln_full_chunks(int nch) {
    constexpr int counts[] = {1, 2, 3, 4, 6, 10, 16, 32};
    int prev = 0;
    for (int n : counts)
        if (n < nch) prev = n;
    return prev;
}

// LayerNorm over the row (fp32 statistics, no affine) followed by the block's
// modulation, fused in front of the quantizer -- the producer of the attn1 and
// FFN-up inputs (dit_block.py:100, :110 of the reference):
//   VDMQ_LN_MODULATE  h = (fp16(LN(x)) * (1 + a)) + b   with a = scale, b = shift, every
//                     operation a correctly rounded fp16 operation, as the reference's
//                     fp16 tensor arithmetic after FP32LayerNorm's cast back to fp16
//   VDMQ_LN_AFFINE    h = fp16(LN(x) * a + b)           with a = weight, b = bias, in
//                     fp32 with one rounding (FP32LayerNorm with elementwise_affine, norm2)
// Row m takes vector row m / rows_per_vec of a and b (stride ldv elements): one
// vector per batch element, or one per token.  EMIT_H writes h itself instead of
// quantizing it (the same arithmetic: the tests' view of h).
// Bound by vector instructions and the reductions between them, so the bf6 form has ROWS = 4 per workgroup, half a panel, whose halves L2
// joins (so no streamed stores): one workgroup's reductions run under another's loads and conversions.  us, eight rows (streamed beyond 128 MiB)
// / four: 512 x 5120 8.1 / 6.8, 4680 x 1536 8.5 / 7.9, 27280 x 3072 54 / 48, 32760 x 4096 92 / 77, 60000 x 5120 181 / 165, 20000 x 13824 222 / 207; 6000
// rows of up to 3072 1.00; with the GEMM behind it 60000 x 3072 -> 3072 399 / 372, 75600 x 5120 -> 13824 2433 / 2392.
// Up to 512 rows a workgroup has two, so that they spread over the CUs, us, two / four: 512 x 1536 3.64 / 3.71, 512 x 5120 6.3 / 6.7, 512 x 8960 11.6 /
// 12.5; more rows than that are a second workgroup on some CUs (1000 x 5120 8.4 / 7.6).
template <int NCH, int LNMODE, bool EMIT_H, int FMT, int ROWS>
__global__ __launch_bounds__(ROWS * kWaveSize, FMT == 1 ? 2 : 1) void ln_quantize_rows_kernel(
    const __half *__restrict__ x, int64_t ldx, int M, int K, int Kp, float eps, const __half *__restrict__ va,
    const __half *__restrict__ vb, int64_t ldv, int rows_per_vec, float clip, uint8_t *__restrict__ qact,
    __half *__restrict__ scale_h, __half *__restrict__ h_out, int64_t ldh) {
    const int lane = threadIdx.x & (kWaveSize - 1), wave = FMT == 1 && NCH > 16 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x >> 6;
    const int64_t row0 = static_cast<int64_t>(FMT == 1 ? bf6_group<ROWS>(blockIdx.x, (M + ROWS - 1) / ROWS) : blockIdx.x) * ROWS;
    int64_t row = row0 + wave;
    const bool valid = row < M;
    if (!valid) {
        if (FMT == 0) return;
        row = M - 1; /* the bf6 tail synchronises the workgroup: stay, on a copy of the last row */
    }
    const u32x4 *src = reinterpret_cast<const u32x4 *>(x + row * ldx);
    const int64_t vrow = rows_per_vec >= M ? 0 : (static_cast<int>(row) / rows_per_vec) * ldv; /* (one vector for all: no division) */
    const u32x4 *pa = reinterpret_cast<const u32x4 *>(va + vrow), *pb = reinterpret_cast<const u32x4 *>(vb + vrow);

    u32x4 v[NCH];
#pragma unroll
    for (int c = 0; c < NCH; ++c)
        v[c] = c < ln_full_chunks(NCH) || c * 512 + lane * 8 < K ? __builtin_nontemporal_load(src + c * 64 + lane) : u32x4{0u, 0u, 0u, 0u};
    ln_row<NCH, LNMODE, ln_full_chunks(NCH)>(v, lane, K, eps, pa, pb);
    if (EMIT_H) {
        u32x4 *dst = reinterpret_cast<u32x4 *>(h_out + row * ldh);
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int k0 = c * 512 + lane * 8;
            if (k0 < K) dst[c * 64 + lane] = v[c];
        }
        return;
    }
    if (FMT == 1) {
        __shared__ __attribute__((aligned(16))) Bf6Scratch<ROWS> scratch;
        int phase = 0;
        quantize_held_row_bf6<NCH, VDMQ_ACT_NONE, ROWS, 1>(v, lane, wave, row0, valid, M, Kp, clip, qact, scale_h, false, scratch, phase, NoRefill{});
    } else {
        quantize_held_row<NCH, false>(v, lane, row, Kp, clip, qact, scale_h);
    }
}

// Any K: two passes over the row (the second one is served by the caches).
template <int ACT>
__global__ __launch_bounds__(kRowsPerBlock * kWaveSize) void quantize_rows_anyk_kernel(const __half *__restrict__ x, int64_t ldx,
                                                                                       int M, int K, int Kp, float clip,
                                                                                       uint8_t *__restrict__ qact,
                                                                                       __half *__restrict__ scale_h) {
    const int lane = threadIdx.x & (kWaveSize - 1);
    const int64_t row = static_cast<int64_t>(blockIdx.x) * kRowsPerBlock + (threadIdx.x >> 6);
    if (row >= M) return;
    const u32x4 *src = reinterpret_cast<const u32x4 *>(x + row * ldx);
    float mx = 0.0f;
    for (int k0 = lane * 8; k0 < K; k0 += 512) mx = absmax_exact(apply_act<ACT>(src[k0 / 8]), mx);
    mx = wave_max(mx);
    const __half sh = scale_from_absmax(mx, clip);
    const float rscale = 1.0f / __half2float(sh);
    uint32_t *dst = reinterpret_cast<uint32_t *>(qact + row * (Kp / 2));
    for (int k0 = lane * 8; k0 < Kp; k0 += 512) {
        u32x4 v = k0 < K ? apply_act<ACT>(src[k0 / 8]) : u32x4{0u, 0u, 0u, 0u};
        dst[k0 / 8] = quantize_word<true>(v, rscale);
    }
    if (lane == 0) scale_h[row] = sh;
}

// Per-row scale only (weights: quantize_weight_per_channel's first launch).
__global__ __launch_bounds__(kRowsPerBlock * kWaveSize) void row_scale_kernel(const __half *__restrict__ x, int64_t rows, int K,
                                                                              float clip, __half *__restrict__ scale_h) {
    const int lane = threadIdx.x & (kWaveSize - 1);
    const int64_t row = static_cast<int64_t>(blockIdx.x) * kRowsPerBlock + (threadIdx.x >> 6);
    if (row >= rows) return;
    const u32x4 *src = reinterpret_cast<const u32x4 *>(x + row * static_cast<int64_t>(K));
    float mx = 0.0f;
    for (int k0 = lane * 8; k0 < K; k0 += 512) mx = absmax_exact(src[k0 / 8], mx);
    mx = wave_max(mx);
    if (lane == 0) scale_h[row] = scale_from_absmax(mx, clip);
}

// Quantize rows with caller-provided fp16 scales into the native layout
// (weights: quantize_warp_static_scale, vdm_w4a4_kernel.cu:296-338).
__global__ __launch_bounds__(256) void quantize_given_scale_kernel(const __half *__restrict__ x, const __half *__restrict__ scale_h,
                                                                   int64_t rows, int K, int Kp, uint8_t *__restrict__ q) {
    const int64_t words_per_row = Kp / 8;
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= rows * words_per_row) return;
    const int64_t row = idx / words_per_row;
    const int k0 = static_cast<int>(idx % words_per_row) * 8;
    u32x4 v = k0 < K ? *reinterpret_cast<const u32x4 *>(x + row * K + k0) : u32x4{0u, 0u, 0u, 0u};
    const float rscale = 1.0f / __half2float(scale_h[row]);
    reinterpret_cast<uint32_t *>(q)[idx] = quantize_word<true>(v, rscale);
}

// Weights [N, K] into the checkpoint's v1 buffers (pack_weight_with_scale, quantize_weight_per_channel) in one pass: a
// workgroup owns a quarter of a 16-row tile of the v1 order (vdmq_layout.hip), rows 2p, 2p + 1, 2p + 8 and 2p + 9, whose words
// share the order's 16-byte pieces; a wave per row, the row in registers (NCH chunks of 512; 0: rows too long for that are
// read twice, the second time mostly from the caches).  The scale is the given one or absmax / 7; 2048 k at a time the
// rows' words meet in LDS and leave as 128-byte runs.  `native` (optional) takes the row-major int4 form as well.
// Bound by memory, 2.5 bytes per weight, where loads and conversions overlap: the rows of a workgroup arrive together and are
// then converted together, so the fewer rows it has, the earlier the first is at work while the next load.  us for a whole tile /
// half / a quarter / an eighth of one per workgroup (16, 8, 4, 2 waves; sixteen leave long rows half the registers, too): 13824 x 5120
// 38.0 / 34.1 / 32.6 / 33.7, 5120 x 13824 61.7 / 49.0 / 36.7 / 37.6, 3072 x 14336 51 / 32.4 / 24.1 / 24.5, 13824 x 13824 159 / 119 / 90 / 93,
// 1536 x 1536 5.2 / 4.6 / 4.6 / 4.6 (6.3 TB/s: 28, 28, 18, 76 and 1).
constexpr int kTileRows = 16, kPackRows = 4, kPackParts = kTileRows / kPackRows, kPackWords = 256 /* words of a row per 2048 k */, kPackRowWords = kPackWords + 4 /* bank spread */;
// waves a SIMD holds, which is what bounds the registers: the row's 4 * NCH and some 40 more
constexpr int pack_waves(int nch) { return nch <= 6 ? 8 : nch <= 10 ? 6 : nch <= 18 ? 4 : nch <= 28 ? 3 : 2; }

template <int NCH>
__global__ __launch_bounds__(kPackRows * kWaveSize, pack_waves(NCH)) void pack_weight_kernel(const __half *__restrict__ w, const __half *__restrict__ scale_in,
                                                                            int units, int K, int Kp, u32x4 *__restrict__ q_v1,
                                                                            u32x2 *__restrict__ scales_v1, __half *__restrict__ scale_out,
                                                                            uint32_t *__restrict__ native) {
    __shared__ __attribute__((aligned(16))) uint32_t words[2][kPackRows][kPackRowWords];
    __shared__ unsigned short scales[kPackRows];
    // the 32 quarters of a 128-row block interleave in memory: they go to one XCD, one after the other, whose L2 joins
    // their runs (blocks are dealt to the XCDs in turn)
    int unit = blockIdx.x;
    if ((unit | 255) < units) unit = (unit & ~255) | (unit & 7) << 5 | (unit >> 3 & 31);
    const int tile = unit / kPackParts, part = unit % kPackParts;
    const int lane = threadIdx.x & (kWaveSize - 1), wave = threadIdx.x >> 6;
    const int64_t row = static_cast<int64_t>(tile) * kTileRows + 2 * part + (wave & 1) + 8 * (wave >> 1);
    const u32x4 *src = reinterpret_cast<const u32x4 *>(w + row * K);
    auto load = [&](int c) { return c * 512 + lane * 8 < K ? __builtin_nontemporal_load(src + c * 64 + lane) : u32x4{0u, 0u, 0u, 0u}; };
    u32x4 v[NCH > 0 ? NCH : 1];
    const int chunks = NCH > 0 ? NCH : (K + 511) / 512;
    uint32_t m2 = 0;
    if constexpr (NCH > 0) {
#pragma unroll
        for (int c = 0; c < NCH; ++c) v[c] = load(c);
#pragma unroll
        for (int c = 0; c < NCH; ++c) m2 = absmax_bits(v[c], m2);
    } else {
        for (int c = 0; c < chunks; ++c) m2 = absmax_bits(load(c), m2);
    }
    const uint32_t m16 = wave_max((m2 & 0xFFFFu) > (m2 >> 16) ? (m2 & 0xFFFFu) : (m2 >> 16));
    const bool finite = m16 < 0x7C00u;
    __half sh;
    if (scale_in != nullptr) {
        sh = scale_in[row];
    } else {
        float mx = half_bits_to_float(m16);
        if (!finite) {
            mx = 0.0f;
            if constexpr (NCH > 0) {
#pragma unroll
                for (int c = 0; c < NCH; ++c) mx = absmax_exact(v[c], mx);
            } else {
                for (int c = 0; c < chunks; ++c) mx = absmax_exact(load(c), mx);
            }
            mx = wave_max(mx);
        }
        sh = scale_from_absmax(mx, 1.0f);
        if (lane == 0) scale_out[row] = sh;
    }
    if (lane == 0) scales[wave] = __half_as_ushort(sh);
    const float rscale = 1.0f / __half2float(sh);
    const bool fast = __builtin_amdgcn_readfirstlane(finite && scale_is_ordinary(sh) ? 1 : 0) != 0;

    const int KG = K / 64;
    const int64_t tile_base = static_cast<int64_t>(tile >> 3) * KG * 8 + (tile & 7); /* in 512-byte runs: + 8 per 64 k */
    const int piece = threadIdx.x & 7, row_lo = piece >> 2, t4 = piece & 3, k64 = threadIdx.x >> 3;
    auto group = [&](int g, auto &&chunk) __attribute__((always_inline)) {
        const int copy = g & 1;
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {
            const int c = 4 * g + cc, k0 = c * 512 + lane * 8;
            const u32x4 x = chunk(c);
            const uint32_t word = fast ? quantize_word<false>(x, rscale) : quantize_word<true>(x, rscale);
            words[copy][wave][cc * 64 + lane] = word;
            if (native != nullptr && k0 < Kp) native[row * (Kp / 8) + k0 / 8] = word;
        }
        __syncthreads(); /* one per group: the copy written next was read before the barrier in front of this one */
        const int bk = 32 * g + k64;
        if (bk < KG) {
            const uint32_t *lo = words[copy][row_lo] + k64 * 8 + t4, *hi = lo + 2 * kPackRowWords;
            q_v1[(tile_base + 8ll * bk) * 32 + 8 * part + piece] = u32x4{lo[0], lo[4], hi[0], hi[4]};
        }
    };
    if constexpr (NCH > 0) {
#pragma unroll
        for (int g = 0; g < (NCH + 3) / 4; ++g) group(g, [&](int c) { return c < NCH ? v[c < NCH ? c : 0] : u32x4{0u, 0u, 0u, 0u}; });
    } else {
        for (int g = 0; g < (chunks + 3) / 4; ++g) group(g, load);
    }
    // the tile's sixteen scales per 64 k, 32 bytes in the order of pack_wscales: row r at 4 * (r % 8 / 2) + 2 * (r / 8) + r % 2; this
    // quarter's four are adjacent
    const u32x2 four = {scales[0] | static_cast<uint32_t>(scales[1]) << 16, scales[2] | static_cast<uint32_t>(scales[3]) << 16};
    for (int i = threadIdx.x; i < KG; i += kPackRows * kWaveSize) scales_v1[(static_cast<int64_t>(tile >> 3) * KG + i) * 32 + (tile & 7) * 4 + part] = four;
}

constexpr int64_t kStreamOutBytes = int64_t(224) << 20; /* outputs larger than this bypass the caches */
// The same for the bf6 blocks, judged by the quantizer and the GEMM that reads its output together: streamed stores
// cost the GEMM the part of its operand that plain stores leave in the Infinity Cache (38 MB and 63 MB of blocks:
// the pair 3 % and 2 % slower), and spare it the wait for the dirty lines of a large one (220 MB, 290 MB, 780 MB:
// the pair 3 %, 0.7 % and 0.7 % faster).  For workgroups of a whole panel; halves of one never stream (bf6_split).
constexpr int64_t kStreamOutBytesBf6 = int64_t(128) << 20, kInfinityCacheBytes = int64_t(256) << 20;

// Workgroups of `kernel` the current device runs at once (CUs x workgroups per CU), or -1.  The answer is
// kept per device in `cache` (one array per kernel, zero-initialised): the occupancy query costs tens of
// microseconds, which a launch on an idle stream would show.
constexpr int kMaxDevices = 64;
int64_t resident_workgroups(const void *kernel, int threads, int (&cache)[kMaxDevices]) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return -1;
    if (cache[dev] > 0) return cache[dev];
    int cus = 0, per_cu = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, 0) != hipSuccess || cus <= 0 || per_cu <= 0) {
        (void)hipGetLastError();
        return -1;
    }
    cache[dev] = cus * per_cu; /* racing first calls store the same value */
    return cache[dev];
}

// Rows per workgroup of the bf6 quantizer, and whether it streams its output.  The rows of a workgroup arrive together and are then
// reduced and converted together: with four the next workgroup's loads run under that, few rows spread over twice as many CUs, and many leave a
// smaller last wave of workgroups.  Against that stand half-panel runs of 64 and 32 bytes, which plain stores join in L2 and streamed ones do
// not (75600 x 5120 streamed: 162 / 220 us with eight / four).  What computes more gains more.  us, eight / four:
//   plain            512 x 5120 5.8 / 5.0   1000 x 13824 12.0 / 10.4   2500 x 8960 15.3 / 13.7   12000 x 8960 50.3 / 48.4
//                    12000 x 3072 18.1 / 18.8   32760 x 1536 23.4 / 24.1
//   GELU             512 x 5120 8.3 / 6.3   2500 x 10240 31.9 / 25.1   4680 x 8960 36.0 / 31.0   32760 x 1536 34.4 / 32
//                    streamed / plain stores: 32760 x 8960 151 / 142, with its GEMM 384 / 366; 60000 x 7168 197 / 218, 32760 x 13824 240 / 272
// Rows that are only quantized keep eight where there are many short ones, and where long ones (a CU holds one workgroup of eight or two of
// four, the chip 2048 rows) fill more than half of the last round: then four have only the shorter runs.  After one round, us, eight / four: 3328 x
// 8960 17.1 / 18.3, 4096 x 8960 19.1 / 20.6, 3840 x 7168 15.5 / 16.1, 4096 x 13824 30.6 / 31.4 (2304 x 8960 15.4 / 13.8, 4608 x 13824 37.2 / 33.8); after
// two 5376 x 13824 39.4 / 41.9, 6144 x 8960 29.7 / 31.5, 6144 x 5632 18.9 / 19.5; after three 7168 x 13824 53.3 / 55.8, 7424 x 12288 47.7 / 50.0, 8192 x 16384 77.1 / 79.0, but 7936 x 8960 37.8 / 37.2.
// Beyond 10240 elements and four rounds eight in any case: 11776 x 13824 84.5 / 87.7, 9216 x 16384 87.5 / 90.4.  With the activation evaluated late (bf6_late_act) four and plain stores
// still win while the output stays in the memory-side cache.
struct Bf6Split {
    int rows, stream_out;
};
template <int NCH, int ACT>
Bf6Split bf6_split(int64_t M, int64_t K) {
    const int64_t bytes = bf6_bytes(M, K);
    const bool large = bytes > kStreamOutBytesBf6;
    const bool full_round = M > 2048 && M <= (K > 10240 ? 8192 : 7680) && (M - 1) % 2048 >= (M > 6144 ? 896 : 1024) && K > (M > 5120 && M <= 6144 ? 5120 : 6144);
    const bool many_long = M > 8704 && K > 10240;
    const bool four = ACT == VDMQ_ACT_NONE ? !large && (M <= 5120 || K > 3584) && !full_round && !many_long
                                           : !large || (bf6_late_act(NCH) && K <= 9216 && bytes <= kInfinityCacheBytes);
    return four ? Bf6Split{kPanelRows / 2, 0} : Bf6Split{kPanelRows, large ? 1 : 0};
}

template <int NCH, int ACT, int ROWS>
int launch_reg_bf6(const __half *x, int64_t M, int64_t K, int64_t ldx, float clip, uint8_t *qact, __half *scale_h, int stream_out, hipStream_t s) {
    const int64_t groups = ceil_div(M, ROWS);
    static int cache[kMaxDevices];
    const int64_t resident = !bf6_walks(NCH) ? groups
                                             : resident_workgroups(reinterpret_cast<const void *>(&quantize_rows_kernel<NCH, false, ACT, 1, ROWS>),
                                                                   ROWS * kWaveSize, cache);
    if (resident <= 0) return fail(VDMQ_ELAUNCH, "quantize_rows_kernel: the occupancy query for the current device failed");
    hipLaunchKernelGGL((quantize_rows_kernel<NCH, false, ACT, 1, ROWS>), dim3(static_cast<unsigned>(groups < resident ? groups : resident)),
                       dim3(ROWS * kWaveSize), ROWS == kPanelRows ? bf6_spare_lds(NCH, ACT) : 0, s, x, ldx, static_cast<int>(M),
                       static_cast<int>(K), static_cast<int>(bf6_kblocks(K) * 64), clip, qact, scale_h, stream_out);
    return check_launch("quantize_rows_kernel");
}

template <int NCH, int ACT>
int launch_reg(const __half *x, int64_t M, int64_t K, int64_t ldx, float clip, int fmt, uint8_t *qact, __half *scale_h, hipStream_t s) {
    if (fmt == 1) {
        const Bf6Split split = bf6_split<NCH, ACT>(M, K);
        return split.rows == kPanelRows ? launch_reg_bf6<NCH, ACT, kPanelRows>(x, M, K, ldx, clip, qact, scale_h, split.stream_out, s)
                                        : launch_reg_bf6<NCH, ACT, kPanelRows / 2>(x, M, K, ldx, clip, qact, scale_h, split.stream_out, s);
    }
    const dim3 grid(static_cast<unsigned>(ceil_div(M, kRowsPerBlock))), block(kRowsPerBlock * kWaveSize);
    if (M * (k_padded(K) / 2) > kStreamOutBytes)
        hipLaunchKernelGGL((quantize_rows_kernel<NCH, true, ACT, 0, kRowsPerBlock>), grid, block, 0, s, x, ldx, static_cast<int>(M), static_cast<int>(K),
                           static_cast<int>(k_padded(K)), clip, qact, scale_h, 0);
    else
        hipLaunchKernelGGL((quantize_rows_kernel<NCH, false, ACT, 0, kRowsPerBlock>), grid, block, 0, s, x, ldx, static_cast<int>(M), static_cast<int>(K),
                           static_cast<int>(k_padded(K)), clip, qact, scale_h, 0);
    return check_launch("quantize_rows_kernel");
}

// Whether rows go to four waves each (quantize_row_parts_kernel): while a wave per row leaves CUs idle or with one workgroup.  us, a wave per row /
// four: 64 x 2048 2.7 / 2.6, 512 x 5120 5.0 / 4.4, 512 x 13824 8.0 / 6.5, 1200 x 5120 6.6 / 6.3, 1200 x 13824 13.2 / 11.0; with the GELU 512 x 2048
// 3.8 / 3.5, 512 x 5120 6.3 / 5.3, 512 x 13824 13.2 / 8.5, 1200 x 13824 21.0 / 16.8.  Beyond: 1200 x 2048 3.8 / 4.3, 3000 x 5120
// 9.4 / 11.4, 2000 x 13824 15.8 / 16.5.  One line for both producers, although the GELU's shortest rows are the same either way around 800 (x 5120
// 6.6 / 6.8; a wave per row by eights, as such calls ran before, 8.7).
constexpr int kPartRows = 2, kParts = 4;
bool rows_in_parts(int64_t M, int64_t K) { return K > 1536 && M <= (K > 2560 ? 1536 : 512); }

template <int ACT>
int launch_row_parts(const __half *x, int64_t M, int64_t K, int64_t ldx, float clip, uint8_t *qact, __half *scale_h, hipStream_t s) {
    const int64_t nch = ceil_div(k_padded(K), 512 * kParts);
    using Kernel = void (*)(const __half *, int64_t, int, int, int, float, uint8_t *, __half *);
    const Kernel kernel = nch <= 1 ? quantize_row_parts_kernel<1, ACT, kPartRows, kParts> : nch <= 2 ? quantize_row_parts_kernel<2, ACT, kPartRows, kParts> :
                          nch <= 3 ? quantize_row_parts_kernel<3, ACT, kPartRows, kParts> : nch <= 4 ? quantize_row_parts_kernel<4, ACT, kPartRows, kParts> :
                          nch <= 5 ? quantize_row_parts_kernel<5, ACT, kPartRows, kParts> : nch <= 6 ? quantize_row_parts_kernel<6, ACT, kPartRows, kParts> :
                          nch <= 7 ? quantize_row_parts_kernel<7, ACT, kPartRows, kParts> : quantize_row_parts_kernel<8, ACT, kPartRows, kParts>;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(ceil_div(M, kPartRows))), dim3(kPartRows * kParts * kWaveSize), 0, s, x, ldx,
                       static_cast<int>(M), static_cast<int>(K), static_cast<int>(bf6_kblocks(K) * 64), clip, qact, scale_h);
    return check_launch("quantize_row_parts_kernel");
}

template <int ACT>
int launch_quantize_act_impl(const __half *x, int64_t M, int64_t K, int64_t ldx, float clip, int fmt, uint8_t *qact, __half *scale_h,
                             hipStream_t s) {
    const int64_t nch = ceil_div(k_padded(K), 512);
    if (fmt == 1 && nch <= 8 * kParts && rows_in_parts(M, K)) return launch_row_parts<ACT>(x, M, K, ldx, clip, qact, scale_h, s);
#define VDMQ_CASE(n) \
    if (nch <= n) return launch_reg<n, ACT>(x, M, K, ldx, clip, fmt, qact, scale_h, s)
    // Rows are held in registers, so the chunk count is a template parameter; a row runs on the first count that
    // covers it (loads beyond K are predicated off: the spare chunks cost registers, not bytes).  Instantiated: what
    // the Wan models' linears need -- K = 1536, 3072, 5120 (3, 6, 10), the FFN widths 8960, 13824 and 14336 (18, 28,
    // 28) -- the small counts, and a sparse cover of the rest up to K = 16384.
    VDMQ_CASE(1);
    VDMQ_CASE(2);
    VDMQ_CASE(3);
    VDMQ_CASE(4);
    VDMQ_CASE(6);
    VDMQ_CASE(10);
    VDMQ_CASE(14);
    VDMQ_CASE(18);
    VDMQ_CASE(24);
    VDMQ_CASE(28);
    VDMQ_CASE(32);
#undef VDMQ_CASE
    if (fmt == 1) return fail(VDMQ_ESHAPE, "the bf6 quantizer needs K <= 16384 (got %lld)", (long long)K);
    const unsigned grid = static_cast<unsigned>(ceil_div(M, kRowsPerBlock));
    hipLaunchKernelGGL(quantize_rows_anyk_kernel<ACT>, dim3(grid), dim3(kRowsPerBlock * kWaveSize), 0, s, x, ldx, static_cast<int>(M),
                       static_cast<int>(K), static_cast<int>(k_padded(K)), clip, qact, scale_h);
    return check_launch("quantize_rows_anyk_kernel");
}

constexpr int64_t kLnFewRows = 512; /* two rows per workgroup up to here: a workgroup per CU (see ln_quantize_rows_kernel) */

template <int NCH, int LNMODE>
int launch_ln_reg(const __half *x, int64_t M, int64_t K, int64_t ldx, float eps, const __half *va, const __half *vb, int64_t ldv,
                  int64_t rows_per_vec, float clip, int fmt, uint8_t *qact, __half *scale_h, __half *h_out, int64_t ldh, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>(ceil_div(M, kRowsPerBlock))), block(kRowsPerBlock * kWaveSize);
    if (h_out != nullptr)
        hipLaunchKernelGGL((ln_quantize_rows_kernel<NCH, LNMODE, true, 0, kRowsPerBlock>), grid, block, 0, s, x, ldx, static_cast<int>(M), static_cast<int>(K),
                           static_cast<int>(k_padded(K)), eps, va, vb, ldv, static_cast<int>(rows_per_vec), clip, qact, scale_h, h_out, ldh);
    else if (fmt == 1) { /* (plain stores at any size: see ln_quantize_rows_kernel) */
        auto launch = [&](auto kernel, int rows) {
            hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(ceil_div(M, rows))), dim3(rows * kWaveSize), 0, s, x, ldx, static_cast<int>(M),
                               static_cast<int>(K), static_cast<int>(bf6_kblocks(K) * 64), eps, va, vb, ldv, static_cast<int>(rows_per_vec), clip, qact,
                               scale_h, h_out, ldh);
        };
        if (M <= kLnFewRows)
            launch(ln_quantize_rows_kernel<NCH, LNMODE, false, 1, 2>, 2);
        else
            launch(ln_quantize_rows_kernel<NCH, LNMODE, false, 1, kPanelRows / 2>, kPanelRows / 2);
    }
    else
        hipLaunchKernelGGL((ln_quantize_rows_kernel<NCH, LNMODE, false, 0, kRowsPerBlock>), grid, block, 0, s, x, ldx, static_cast<int>(M), static_cast<int>(K),
                           static_cast<int>(k_padded(K)), eps, va, vb, ldv, static_cast<int>(rows_per_vec), clip, qact, scale_h, h_out, ldh);
    return check_launch("ln_quantize_rows_kernel");
}

template <int LNMODE>
int launch_ln_impl(const __half *x, int64_t M, int64_t K, int64_t ldx, float eps, const __half *va, const __half *vb, int64_t ldv,
                   int64_t rows_per_vec, float clip, int fmt, uint8_t *qact, __half *scale_h, __half *h_out, int64_t ldh, hipStream_t s) {
    const int64_t nch = ceil_div(k_padded(K), 512);
#define VDMQ_CASE(n) \
    if (nch <= n) return launch_ln_reg<n, LNMODE>(x, M, K, ldx, eps, va, vb, ldv, rows_per_vec, clip, fmt, qact, scale_h, h_out, ldh, s)
    // (the counts of ln_full_chunks: the LayerNorm runs over a model's width -- 1536, 3072, 5120: 3, 6, 10)
    VDMQ_CASE(1);
    VDMQ_CASE(2);
    VDMQ_CASE(3);
    VDMQ_CASE(4);
    VDMQ_CASE(6);
    VDMQ_CASE(10);
    VDMQ_CASE(16);
    VDMQ_CASE(32);
#undef VDMQ_CASE
    return fail(VDMQ_ESHAPE, "the fused LayerNorm needs K <= 16384 (got %lld)", (long long)K);
}

__global__ __launch_bounds__(256) void gelu_tanh_kernel(const uint32_t *__restrict__ x, uint32_t *__restrict__ y, int64_t pairs) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < pairs) y[i] = gelu_tanh_pair(x[i]);
}

}  // namespace

int launch_quantize_act(const __half *x, int64_t M, int64_t K, int64_t ldx, float clip, int act, int fmt, uint8_t *qact,
                        __half *scale_h, hipStream_t s) {
    if (M == 0) return VDMQ_OK;
    if (act == VDMQ_ACT_GELU_TANH) return launch_quantize_act_impl<VDMQ_ACT_GELU_TANH>(x, M, K, ldx, clip, fmt, qact, scale_h, s);
    return launch_quantize_act_impl<VDMQ_ACT_NONE>(x, M, K, ldx, clip, fmt, qact, scale_h, s);
}

int launch_ln_quantize(const __half *x, int64_t M, int64_t K, int64_t ldx, float eps, int ln_mode, const __half *va, const __half *vb,
                       int64_t ldv, int64_t rows_per_vec, float clip, int fmt, uint8_t *qact, __half *scale_h, __half *h_out, int64_t ldh,
                       hipStream_t s) {
    if (M == 0) return VDMQ_OK;
    if (ln_mode == VDMQ_LN_MODULATE)
        return launch_ln_impl<VDMQ_LN_MODULATE>(x, M, K, ldx, eps, va, vb, ldv, rows_per_vec, clip, fmt, qact, scale_h, h_out, ldh, s);
    return launch_ln_impl<VDMQ_LN_AFFINE>(x, M, K, ldx, eps, va, vb, ldv, rows_per_vec, clip, fmt, qact, scale_h, h_out, ldh, s);
}

int launch_gelu_tanh(const __half *x, __half *y, int64_t n, hipStream_t s) {
    const int64_t pairs = n / 2;
    if (pairs == 0) return VDMQ_OK;
    hipLaunchKernelGGL(gelu_tanh_kernel, dim3(static_cast<unsigned>(ceil_div(pairs, 256))), dim3(256), 0, s,
                       reinterpret_cast<const uint32_t *>(x), reinterpret_cast<uint32_t *>(y), pairs);
    return check_launch("gelu_tanh_kernel");
}

int launch_row_scale(const __half *x, int64_t rows, int64_t K, float clip, __half *scale_h, hipStream_t s) {
    if (rows == 0) return VDMQ_OK;
    hipLaunchKernelGGL(row_scale_kernel, dim3(static_cast<unsigned>(ceil_div(rows, kRowsPerBlock))),
                       dim3(kRowsPerBlock * kWaveSize), 0, s, x, rows, static_cast<int>(K), clip, scale_h);
    return check_launch("row_scale_kernel");
}

int launch_pack_weight(const __half *w, const __half *scale_in, int64_t N, int64_t K, uint8_t *q_v1, __half *scales_v1, __half *scale_out,
                       uint8_t *native, hipStream_t s) {
    if (N == 0) return VDMQ_OK;
    const int64_t nch = ceil_div(k_padded(K), 512);
    using Kernel = void (*)(const __half *, const __half *, int, int, int, u32x4 *, u32x2 *, __half *, uint32_t *);
    // (a chunk that a row does not have is still loaded, converted and staged as zeros: 4608 x 4096 on 10 chunks 13.3 us, on 8
    // 12.3; 2048 x 16384 read twice 43, on 32 20.9)
    const Kernel kernel = nch <= 2 ? pack_weight_kernel<2> : nch <= 3 ? pack_weight_kernel<3> : nch <= 4 ? pack_weight_kernel<4> :
                          nch <= 6 ? pack_weight_kernel<6> : nch <= 8 ? pack_weight_kernel<8> : nch <= 10 ? pack_weight_kernel<10> :
                          nch <= 14 ? pack_weight_kernel<14> : nch <= 18 ? pack_weight_kernel<18> : nch <= 24 ? pack_weight_kernel<24> :
                          nch <= 28 ? pack_weight_kernel<28> : nch <= 32 ? pack_weight_kernel<32> : pack_weight_kernel<0>;
    const int units = static_cast<int>(N / kPackRows);
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(units)), dim3(kPackRows * kWaveSize), 0, s, w, scale_in, units, static_cast<int>(K),
                       static_cast<int>(k_padded(K)), reinterpret_cast<u32x4 *>(q_v1), reinterpret_cast<u32x2 *>(scales_v1), scale_out,
                       reinterpret_cast<uint32_t *>(native));
    return check_launch("pack_weight_kernel");
}

int launch_quantize_given_scale(const __half *x, const __half *scale_h, int64_t rows, int64_t K, uint8_t *q, hipStream_t s) {
    if (rows == 0) return VDMQ_OK;
    const int64_t total = rows * (k_padded(K) / 8);
    hipLaunchKernelGGL(quantize_given_scale_kernel, dim3(static_cast<unsigned>(ceil_div(total, 256))), dim3(256), 0, s, x, scale_h,
                       rows, static_cast<int>(K), static_cast<int>(k_padded(K)), q);
    return check_launch("quantize_given_scale_kernel");
}

}  // namespace vdmq
