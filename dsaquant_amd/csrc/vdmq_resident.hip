// Quantizer and W4A4 GEMM in one kernel for short rows: the workgroup quantizes its token rows into LDS, where they stay
// while the weights stream past them.
//
// A workgroup of eight waves owns 32 * MI token rows.  It reads them as fp16, quantizes them exactly as the quantizers of
// vdmq_quant.hip do (vdmq_rowops.h) and keeps them in LDS as bf6 operand blocks (vdmq_bf6.hip), all K of them: 128 rows of 1536
// are 144 KiB.  One barrier later every wave is on its own: it takes strips of 64 output columns in turn, streams their
// weight blocks from L2 straight into its registers, two K steps ahead, and reads the token operand from LDS, which nobody
// writes any more.  No barrier in the K loop, none between tiles: one wave's epilogue runs under its neighbours' matrix
// instructions.
//
// Against quantizer and tiled GEMM it saves a launch and the blocks' way to memory and back, and where tiles of 256 x 256 or 128 x 128
// leave CUs idle its units need not.  Measured as a call among others, us, two kernels -> here: 512 x 1536 -> 3072 19.9 -> 12.3 (the
// host's; the kernel takes 10.0), 3613 x 1024 -> 4096 25.1 -> 18.5, 4096 x 1536 -> 4608 32.7 -> 26.4, 32760 x 1536 -> 4608 151 -> 124,
// -> 1536 with gate and residual 98.7 -> 78.7.  What bounds it: at 32760 x 1536 -> 4608 the matrix cores, busy two thirds of the time at the
// 1.7 GHz the chip holds under them; taking instructions out of the K step or moving its loads changed nothing there.  At a few
// thousand rows the quantization, repeated in every column group (5 us of 26 at 4096 rows; half the vector instructions in its absmax
// changed nothing), and the weights' way into the registers for 64 or 32 rows at a time.
// Why 64 columns and two waves per SIMD: 32 x MI x 64 sums fill half of a wave's registers at MI = 4, and 64 columns are the 128-byte lines
// that an epilogue needs; weights through LDS would take the room of the rows and a barrier per step, and each weight byte is read once
// per CU as it is.  Non-temporal stores because the next kernel reads most outputs too late to find them in L2, where
// they push out the weights.  Ordinary / non-temporal, us, the kernel back to back on four sets of buffers in turn: 32760 x 1536 ->
// 4608 170 / 132, -> 8960 309 / 237, -> 1536 66.9 / 57.0 and with gate and residual 83.8 / 80.4 (80.0 / 61.6 on one set), 16000 x 1536 ->
// 4608 77.0 / 66.5, 3613 x 1024 -> 4096 21.1 / 18.9, 4096 x 1536 -> 4608 27.3 / 26.3, 512 x 1536 -> 3072 9.3 / 9.3.
#include <type_traits>

#include "vdmq_rowops.h"

namespace vdmq {
namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kWaves = 8, kStripCols = 64, kXcds = 8;
constexpr int kBlk = 1536;            /* 32 rows x 64 k in LDS: [2 x 32 x 16 bytes][2 x 32 x 8 bytes] */
constexpr int kStage = 2048;          /* epilogue staging of a wave: 16 rows x 64 fp16 columns */
[[maybe_unused]] constexpr float kAccScale = 256.0f;   /* the blocks hold q / 16 */

struct ResidentArgs {
    const __half *x;
    int64_t ldx;
    const uint8_t *w;
    const __half *wscale, *bias;
    __half *out;
    int64_t ldo;
    int M, N, K, kblocks;
    float clip;
    float eps;
    const __half *va, *vb;
    int64_t ldv;
    int rows_per_vec;
    int tiles, groups; /* row tiles; column groups a row tile is split into (a workgroup each) */
    int by_group;      /* order of the units */
    GemmTail tail;
};
enum { kPreNone, kPreLnModulate, kPreLnAffine };

// Where a string lies in its 1536-byte block: 16-byte part at 16 * place, 8-byte part at 1024 + 8 * place, place = 32 * h +
// (row ^ 8h ^ kb % 8).  The sixteen strings that a wave writes at once (one row, eight k-blocks, two halves) then meet 64
// different banks, and so do the reads, which take all 32 rows of a block.
[[maybe_unused]] __device__ __forceinline__ int string_place(int row, int h, int kb) { return 32 * h + (row ^ (8 * h) ^ (kb & 7)); }

// What one lane of a wave writes to LDS another one reads, without a barrier: the wave's LDS operations are executed in order.
// The compiler reasons about one lane alone and must not move them across, or reuse what it has read before.
[[maybe_unused]] __device__ __forceinline__ void lanes_meet() { asm volatile("" ::: "memory"); }

// the lane's number, worked out again where it is wanted instead of being held in a register
[[maybe_unused]] __device__ __forceinline__ int lane_again() {
    int l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(l));
    return l;
}

#if defined(__HIP_DEVICE_COMPILE__)
// Maximum over the wave's 64 lanes as a scalar (as wave_max, written so that every step is one v_max_u32 with a DPP operand).
__device__ __forceinline__ uint32_t row_max(uint32_t v) {
    auto step = [&](uint32_t o) { v = o > v ? o : v; };
    step(dpp<kDppSwap1, 0xF, true>(0u, v));
    step(dpp<kDppSwap2, 0xF, true>(0u, v));
    step(dpp<kDppHalfMirror, 0xF, true>(0u, v));
    step(dpp<kDppMirror, 0xF, true>(0u, v));
    step(dpp<kDppBcast15, 0xA, false>(0u, v));
    step(dpp<kDppBcast31, 0xC, false>(0u, v));
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 63));
}

// Four rows held in registers (v[i][c] = elements 512c + 8*lane ... +7 of row i, zero beyond K) into bf6 blocks in LDS.
// `rb`: the row-block they lie in, `row`: the first one's place in it, a multiple of four.  A conversion takes four chunks, of
// whichever rows.
template <int MI, int NCH>
__device__ __forceinline__ void quantize_four_rows(const u32x4 (&v)[4][NCH], int lane, int rb, int row, int kblocks, float clip, uint8_t *lds,
                                                   uint8_t *scales) {
    uint32_t m16[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t m2 = 0;
#pragma unroll
        for (int c = 0; c < NCH; ++c) m2 = absmax_bits(v[i][c], m2);
        m16[i] = (m2 & 0xFFFFu) > (m2 >> 16) ? (m2 & 0xFFFFu) : (m2 >> 16);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) m16[i] = row_max(m16[i]);
    // lane l works out the scale of row l % 4 (else: the same instructions in 64 equal lanes, four times)
    const int p = lane & 3;
    const uint32_t mine = p < 2 ? (p == 0 ? m16[0] : m16[1]) : (p == 2 ? m16[2] : m16[3]);
    const bool finite = mine < 0x7C00u;
    float mx = half_bits_to_float(mine);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!finite) != 0, 0)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (m16[i] < 0x7C00u) continue;
            float e = 0.0f;
#pragma unroll
            for (int c = 0; c < NCH; ++c) e = absmax_exact(v[i][c], e);
            e = wave_max(e);
            mx = p == i ? e : mx;
        }
    }
    const __half sh = scale_from_absmax(mx, clip);
    const bool fast = finite && scale_is_ordinary(sh);
    float rs = reciprocal_of_scale(__half2float(sh));
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!fast) != 0, 0)) rs = fast ? rs : 1.0f / __half2float(sh);
    // (the instruction rounds and needs |t| below 8.5, above -8.5 and t below 7.5: see vdmq_quant.hip; where one row has to be
    // clamped all four are, which changes nothing in the others)
    const bool clamp = __builtin_amdgcn_ballot_w64(!(fast && mx * rs < 7.5f)) != 0;
    if (lane < 4) *reinterpret_cast<__half *>(scales + (rb * 32 + row + lane) * 2) = sh;
    float rscale[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) rscale[i] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(rs), i));

    // the lane's quarter of a string (see vdmq_quant.hip): k-block lane / 8 of the chunk's eight, half lane / 4 % 2, bytes 6p ...
    // 6p + 5, p = lane % 4; a word and a half word, none of which crosses from the 16-byte into the 8-byte part
    const int h = (lane >> 2) & 1, kb = lane >> 3;
    const bool odd = (p & 1) != 0;
    const int blk = (kb * MI + rb) * kBlk, place = string_place(row & ~3, h, kb & ~3), twist = kb & 3; /* row i of the four: place + (i ^ twist) */
    const int word0 = blk + (p == 3 ? 1024 + place * 8 - 16 : place * 16) + p * 6 + (odd ? 2 : 0);
    const int half0 = blk + (p >= 2 ? 1024 + place * 8 - 16 : place * 16) + p * 6 + (odd ? 0 : 4);
    const int word_row = p == 3 ? 8 : 16, half_row = p >= 2 ? 8 : 16;
    int word_at[4], half_at[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        word_at[i] = word0 + (i ^ twist) * word_row;
        half_at[i] = half0 + (i ^ twist) * half_row;
    }
    const bool in = 8 * (NCH - 1) + kb < kblocks; /* strings beyond K go to a place that nobody reads, in the epilogue's staging behind the scales */
    const int nowhere = kblocks * MI * kBlk + 1024 + lane * 4;
#pragma unroll
    for (int j = 0; j < NCH; ++j) {
        f32x16 even, odds;
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {
            const int i = (4 * j + cc) / NCH, c = (4 * j + cc) % NCH;
            const uint32_t w[4] = {v[i][c].x, v[i][c].y, v[i][c].z, v[i][c].w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const f16x2 hh = __builtin_bit_cast(f16x2, w[e]);
                even[cc * 4 + e] = __builtin_fmaf(static_cast<float>(hh[0]), rscale[i], 0.0f);
                odds[cc * 4 + e] = __builtin_fmaf(static_cast<float>(hh[1]), rscale[i], 0.0f);
            }
        }
        if (__builtin_expect(clamp, 0)) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                even[e] = __builtin_amdgcn_fmed3f(even[e] == even[e] ? even[e] : 0.0f, -8.0f, 7.0f);
                odds[e] = __builtin_amdgcn_fmed3f(odds[e] == odds[e] ? odds[e] : 0.0f, -8.0f, 7.0f);
            }
        }
        const u32x6 str = to_bf6(even, odds);
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {
            const int i = (4 * j + cc) / NCH, c = (4 * j + cc) % NCH;
            const uint32_t lo = str[cc / 2 * 3 + cc % 2], hi = str[cc / 2 * 3 + cc % 2 + 1];
            const uint32_t joined = __builtin_amdgcn_alignbyte(hi, lo, 2);
            const uint32_t word = cc % 2 == 0 ? (odd ? joined : lo) : (odd ? hi : joined);
            const uint32_t half = cc % 2 == 0 ? (odd ? lo : hi) : (odd ? lo : hi) >> 16;
            int to_word = word_at[i] + 8 * c * MI * kBlk, to_half = half_at[i] + 8 * c * MI * kBlk;
            if (c == NCH - 1) {
                to_word = in ? to_word : nowhere;
                to_half = in ? to_half : nowhere;
            }
            *reinterpret_cast<uint32_t *>(lds + to_word) = word;
            *reinterpret_cast<uint16_t *>(lds + to_half) = static_cast<uint16_t>(half);
        }
    }
}
#endif

// TAIL: the gated residual update in the epilogue; ODD: an odd number of K steps
template <int MI, int NCH, int PRE, bool TAIL, bool ODD>
__global__ __launch_bounds__(kWaves * 64, 2) void resident_linear_kernel(const ResidentArgs args) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int ROWS = 32 * MI, kStepBytes = 2 * MI * kBlk;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, lh = lane >> 5;
    const int M = args.M, K = args.K, kblocks = args.kblocks, pairs = kblocks / 2;
    // Units (row tile, column group) in eight equal runs, one per XCD: row tile by row tile, so that the workgroups of a row tile
    // share an L2 and the rows are fetched once, or group by group, so that the weights are.
    const int units = args.tiles * args.groups, xcd = blockIdx.x % kXcds, slot = blockIdx.x / kXcds;
    const int first = static_cast<int>(static_cast<int64_t>(units) * xcd / kXcds), last = static_cast<int>(static_cast<int64_t>(units) * (xcd + 1) / kXcds);
    const int unit = first + slot;
    if (unit >= last) return;
    const int inner = args.by_group ? args.tiles : args.groups, outer_at = unit / inner, inner_at = unit - outer_at * inner;
    const int tile = args.by_group ? inner_at : outer_at, group = args.by_group ? outer_at : inner_at;
    const int strips = args.N / kStripCols;
    const int strip0 = static_cast<int>(static_cast<int64_t>(strips) * group / args.groups), strip1 = static_cast<int>(static_cast<int64_t>(strips) * (group + 1) / args.groups);
    const int m0 = tile * ROWS;
    uint8_t *const stage = lds + kblocks * MI * kBlk;

    // ---- weights: per K step (two k-blocks) and 32 columns three 16-byte loads per lane: the 16-byte parts of its two strings,
    // and the 8-byte parts of two neighbouring rows, an even lane those of the first k-block, an odd lane those of the second
    const int rb_bytes = 4 * kblocks * kBf6PanelKb;
    const uint32_t lane_a = (l32 >> 3) * kblocks * kBf6PanelKb + lh * 128 + (l32 & 7) * 16;
    const uint32_t lane_b = (l32 >> 3) * kblocks * kBf6PanelKb + 256 + lh * 64 + (l32 & 6) * 8 + (l32 & 1) * kBf6PanelKb;
    const bool odd_lane = (lane & 1) != 0;
    // a slot holds the weights of one K step: a[2 * k-block + columns], and the 8-byte parts as they arrive (raw) and as they are used (b)
    using PartsA = u32x4[4];
    using PartsB = u32x2[4];
    using PartsRaw = u32x4[2];
    // Where the next slot is loaded from: strip (the wave's next one when this one is through; behind the last one the same again,
    // never used) and K step.
    int load_strip = strip0 + wave < strip1 ? strip0 + wave : strip1 - 1, load_pair = 0, load_off = 0;
    const uint8_t *load_base = args.w + static_cast<int64_t>(load_strip) * 2 * rb_bytes;
    auto load16 = [&](uint32_t voff, int ni, int more = 0) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(load_base), 0, 2 * rb_bytes, 0x00020000);
        return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(src, voff, load_off + ni * rb_bytes + more, 0));
    };
    auto load_advance = [&]() __attribute__((always_inline)) { /* (no branch: it stands in the middle of a K step) */
        const bool through = load_pair + 1 == pairs, on = through && load_strip + kWaves < strip1;
        load_pair = through ? 0 : load_pair + 1;
        load_off = through ? 0 : load_off + 2 * kBf6PanelKb;
        load_strip += on ? kWaves : 0;
        load_base += on ? kWaves * 2 * rb_bytes : 0;
    };
    auto untangle = [&](PartsB &b, const PartsRaw &parts, int ni) __attribute__((always_inline)) { /* neighbouring lanes hand each other the parts they loaded for the other */
        const u32x4 raw = parts[ni];
        const uint32_t t0 = dpp<kDppSwap1, 0xF, true>(0u, odd_lane ? raw.x : raw.z), t1 = dpp<kDppSwap1, 0xF, true>(0u, odd_lane ? raw.y : raw.w);
        b[ni] = odd_lane ? u32x2{t0, t1} : u32x2{raw.x, raw.y};
        b[2 + ni] = odd_lane ? u32x2{raw.z, raw.w} : u32x2{t0, t1};
    };
    PartsA a0, a1;
    PartsB b0, b1;
    PartsRaw raw0, raw1;
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) {
        raw0[ni] = load16(lane_b, ni);
        a0[ni] = load16(lane_a, ni);
        a0[2 + ni] = load16(lane_a, ni, kBf6PanelKb);
    }
    load_advance();
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) {
        raw1[ni] = load16(lane_b, ni);
        a1[ni] = load16(lane_a, ni); /* (the rest: see step) */
    }

    uint32_t asked;
    // ---- the token rows: 4 * MI per wave, four at a time, the next four on their way
    {
        const int row0 = wave * 4 * MI, rb = row0 / 32;
        auto load_row = [&](u32x4 (&v)[NCH], int r) __attribute__((always_inline)) {
            const int m = m0 + r < M ? m0 + r : M - 1; /* rows beyond M: a copy of the last one, never stored */
            const __amdgpu_buffer_rsrc_t row = __builtin_amdgcn_make_buffer_rsrc(const_cast<__half *>(args.x + static_cast<int64_t>(m) * args.ldx), 0, K * 2, 0x00020000);
#pragma unroll
            for (int c = 0; c < NCH; ++c) /* (zeros beyond K) */
                v[c] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(row, lane * 16 + c * 1024, 0, 0));
        };
        u32x4 va[4][NCH], vb[4][NCH];
        auto load_group = [&](u32x4 (&v)[4][NCH], int g) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 4; ++i) load_row(v[i], row0 + 4 * g + i);
        };
        auto work_group = [&](u32x4 (&v)[4][NCH], int g) __attribute__((always_inline)) {
            const int r = row0 + 4 * g;
            if constexpr (PRE != kPreNone) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int m = m0 + r + i < M ? m0 + r + i : M - 1;
                    const int64_t vrow = args.rows_per_vec >= M ? 0 : (m / args.rows_per_vec) * args.ldv;
                    const u32x4 *pa = reinterpret_cast<const u32x4 *>(args.va + vrow), *pb = reinterpret_cast<const u32x4 *>(args.vb + vrow);
                    ln_row<NCH, PRE == kPreLnModulate ? VDMQ_LN_MODULATE : VDMQ_LN_AFFINE, NCH - 1>(v[i], lane, K, args.eps, pa, pb);
                }
            }
            quantize_four_rows<MI, NCH>(v, lane, rb, r % 32, kblocks, args.clip, lds, stage);
        };
        load_group(va, 0);
        // The weights, which the next call seldom shares, come from memory: a byte that no XCD has asked for yet takes longer than the two K
        // steps that it is loaded ahead, and since all workgroups want the same strips at the same time all would wait at every step.
        // So each wave asks for 64 lines of 128 bytes at once, all waves together for all of them (as far as that goes), behind its
        // first rows, which so need not wait for them; from then on they are in the memory-side cache.  (Every call with weights of
        // its own, us, without / with: 32760 x 1536 -> 4608 157 / 123, -> 8960 289 / 224, behind a LayerNorm 305 / 235, 32760 x 1024 ->
        // 4096 124 / 98, 4096 x 1536 -> 4608 35.5 / 27.1, 2500 x 640 -> 4096 16.2 / 13.4; always the same weights 118.6 / 118.8, 215 / 219,
        // 231 / 232, 92 / 87, 26.2 / 25.9, 12.0 / 12.0.)
        const __amdgpu_buffer_rsrc_t weights = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t *>(args.w), 0, static_cast<int>(min(static_cast<int64_t>(args.N / 32) * rb_bytes, static_cast<int64_t>(0x7FFFFFFF))), 0x00020000);
        asked = __builtin_amdgcn_raw_buffer_load_b32(weights, ((blockIdx.x * kWaves + wave) * 64 + lane) * 128, 0, 0);
        if constexpr (MI > 1) {
#pragma unroll 1
            for (int g = 0; g < MI; g += 2) {
                load_group(vb, g + 1);
                work_group(va, g);
                if (g + 2 < MI) load_group(va, g + 2);
                work_group(vb, g + 1);
            }
        } else {
            work_group(va, 0);
        }
    }
    asm volatile("" ::"v"(asked)); /* (has arrived: the rows were asked for later) */
    __syncthreads();
    // token scales, as they are used for one row-block at a time: fp16, row-blocks 0 and 1 in the lower and upper 32 lanes of the
    // low half, 2 and 3 of the high half (a register instead of four)
    uint32_t scales4 = *reinterpret_cast<const uint16_t *>(stage + (MI == 1 ? l32 : lane) * 2);
    if (MI == 4) scales4 |= static_cast<uint32_t>(*reinterpret_cast<const uint16_t *>(stage + (64 + lane) * 2)) << 16;
    __syncthreads(); /* the scales lie where the epilogue stages */

    // ---- one wave, its strips
    const uint32_t place8 = string_place(l32, lh, 0) * 8;
    auto frag = [&](uint32_t twisted, int base, int blk) __attribute__((always_inline)) { /* twisted: place8 ^ 8 * (kb % 8) of the block's kb */
        const u32x4 a = *reinterpret_cast<const u32x4 *>(lds + (base + (twisted << 1)) + blk * kBlk);
        const u32x2 b = *reinterpret_cast<const u32x2 *>(lds + (base + twisted) + (blk * kBlk + 1024));
        return v8i{(int)a.x, (int)a.y, (int)a.z, (int)a.w, (int)b.x, (int)b.y, 0, 0};
    };
    uint8_t *const stg = stage + wave * kStage;
    v16f acc[2][MI];
    v8i xf[MI];
    int xbase = 0, twist = 0; /* of the K step's first k-block: its blocks in LDS, 8 * (kb % 8) */
    // One K step: 2 x 2 x MI matrix instructions on one slot; the other is the next step's.  A token fragment is read again, for the
    // next k-block, as soon as the last instruction that uses it has been issued; the weight loads are spread over the step, each
    // as soon as its registers are free: the 16-byte parts of the second k-block for the next step, then everything else
    // for the step after that.  The 8-byte parts of the next step, which have arrived by then, are untangled here too, so
    // that a step begins with matrix instructions.
    auto step = [&](PartsA &a, PartsB &b, PartsRaw &raw, PartsA &a_next, PartsB &b_next, PartsRaw &raw_next, auto first_step, auto last_step) __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(first_step)::value, LAST = decltype(last_step)::value;
        if (FIRST) { /* (not held through the epilogue of the strip before) */
            xbase = twist = 0;
            asm volatile("" : "+s"(xbase), "+s"(twist)); /* (no addresses of its own for this step: they would be held all along) */
#pragma unroll
            for (int mi = 0; mi < MI; ++mi) xf[mi] = frag(place8 ^ twist, xbase, mi);
        }
        const uint32_t at[2] = {place8 ^ (twist + 8), place8 ^ ((twist + 16) & 63)}; /* of the two k-blocks that are read in this step */
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            v8i wf[2];
#pragma unroll
            for (int ni = 0; ni < 2; ++ni) {
                const u32x4 p = a[2 * kb + ni];
                const u32x2 q = b[2 * kb + ni];
                wf[ni] = v8i{(int)p.x, (int)p.y, (int)p.z, (int)p.w, (int)q.x, (int)q.y, 0, 0};
            }
#pragma unroll
            for (int mi = 0; mi < MI; ++mi) {
#pragma unroll
                for (int ni = 0; ni < 2; ++ni) {
                    const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                    acc[ni][mi] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wf[ni], xf[mi], FIRST && kb == 0 ? zero : acc[ni][mi], 3, 3, 0, 0, 0, 0);
                    // four turns of a k-block: behind every other instruction (MI = 4), every one (2), two behind each (1)
                    const int i = mi * 2 + ni;
                    if (kb == 0) {
                        if (i == 0) a_next[2] = load16(lane_a, 0, kBf6PanelKb);
                        if (i == MI / 2) {
                            a_next[3] = load16(lane_a, 1, kBf6PanelKb);
                            load_advance();
                        }
                        if (i == MI) raw[0] = load16(lane_b, 0);
                        if (i == MI * 3 / 2) raw[1] = load16(lane_b, 1);
                    } else {
                        if (i == 0) a[0] = load16(lane_a, 0);
                        if (i == MI / 2) a[1] = load16(lane_a, 1);
                        if (i == MI) untangle(b_next, raw_next, 0);
                        if (i == MI * 3 / 2) untangle(b_next, raw_next, 1);
                    }
                }
                if (kb == 0 || !LAST) xf[mi] = frag(at[kb], xbase, (kb + 1) * MI + mi);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        xbase += kStepBytes;
        twist = (twist + 16) & 63;
    };
    untangle(b0, raw0, 0);
    untangle(b0, raw0, 1);
    const int wave_rows = min(M - m0, ROWS), ldo = static_cast<int>(args.ldo);
    const GemmTail &tail = args.tail;
    auto vector_of = [&](const __half *p, int bytes) __attribute__((always_inline)) { /* (nothing to read: zeros) */
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<__half *>(p), 0, p != nullptr ? bytes : 0, 0x00020000);
    };
    // Of a SIMD's two waves the older one goes first wherever both could issue, and would be through its strips a fifth of the time
    // before the other.  The younger four (waves 4 ... 7: waves are placed round the four SIMDs) take precedence from two fifths of
    // their strips on.
    const int precedence_from = wave < kWaves / 2 ? strip1 : strip0 + (strip1 - strip0) * 2 / 5;
    auto work_strip = [&](int strip, PartsA &a, PartsB &b, PartsRaw &raw, PartsA &a_next, PartsB &b_next, PartsRaw &raw_next) __attribute__((always_inline)) {
        if (strip >= precedence_from) __builtin_amdgcn_s_setprio(1);
        const int n0 = strip * kStripCols;
        // channel scales, bias (none: -0, whose addition changes no bit) and gate (none: 1) of the strip, a column per lane; requested
        // under the last K step
        uint16_t ws = 0, bias = 0, gate = 0;
        auto request_vectors = [&]() __attribute__((always_inline)) {
            const int off = lane_again() * 2;
            ws = __builtin_amdgcn_raw_buffer_load_b16(vector_of(args.wscale + n0, 128), off, 0, 0);
            bias = __builtin_amdgcn_raw_buffer_load_b16(vector_of(args.bias != nullptr ? args.bias + n0 : nullptr, 128), off, 0, 0);
            if (TAIL) gate = __builtin_amdgcn_raw_buffer_load_b16(vector_of(tail.gate != nullptr ? tail.gate + n0 : nullptr, 128), off, 0, 0);
        };
        constexpr std::true_type yes{};
        constexpr std::false_type no{};
        step(a, b, raw, a_next, b_next, raw_next, yes, no);
        for (int p = ODD ? 3 : 2; p < pairs; p += 2) {
            step(a_next, b_next, raw_next, a, b, raw, no, no);
            step(a, b, raw, a_next, b_next, raw_next, no, no);
        }
        if constexpr (ODD) {
            step(a_next, b_next, raw_next, a, b, raw, no, no);
            request_vectors();
            step(a, b, raw, a_next, b_next, raw_next, no, yes);
        } else {
            request_vectors();
            step(a_next, b_next, raw_next, a, b, raw, no, yes);
        }

        // ---- epilogue: out = fp16(float(acc) * (float(as) * float(ws))) (+ bias) [then residual + y * gate], 16 rows of the strip at a
        // time through the wave's staging, so that rows leave as whole 128-byte lines
        const int el = lane_again();
        const int em = el & 31, eh = el >> 5, srow = el >> 3, piece = (el & 7) * 8;
        if (args.bias == nullptr) bias = 0x8000u;
        if (TAIL && tail.gate == nullptr) gate = 0x3C00u;
        // The strip of the output (and of the residual) is a buffer that ends with the last row below M: rows beyond are dropped by
        // the range check, which looks at the vector offset alone, so the row goes there.
        const int part = tail.split_cols != 0 ? n0 / tail.split_cols : 0;
        const __amdgpu_buffer_rsrc_t out_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            args.out + part * tail.part_stride + static_cast<int64_t>(m0) * args.ldo + (n0 - part * tail.split_cols), 0, wave_rows * ldo * 2, 0x00020000);
        const int out_voff = (srow * ldo + piece) * 2, ldr = static_cast<int>(tail.ldr), res_voff = (srow * ldr + piece) * 2;
        const __amdgpu_buffer_rsrc_t res_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<__half *>(tail.residual) + static_cast<int64_t>(m0) * tail.ldr + n0, 0,
                                                                                  TAIL ? wave_rows * ldr * 2 : 0, 0x00020000);
        f16x8 rv[2][2];
        auto fetch = [&](int t) __attribute__((always_inline)) { /* the residual of rows 16t ... 16t + 15, a turn ahead of its use */
#pragma unroll
            for (int it = 0; it < 2; ++it)
                rv[t & 1][it] = __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(res_rsrc, res_voff + (t * 16 + it * 8) * ldr * 2, 0, 0));
        };
        if (TAIL) fetch(0);
        *reinterpret_cast<uint16_t *>(stg + el * 2) = ws;
        *reinterpret_cast<uint16_t *>(stg + 128 + el * 2) = bias;
        if (TAIL) *reinterpret_cast<uint16_t *>(stg + 256 + el * 2) = gate;
        lanes_meet();
        f16x4 w4[2][4];
#pragma unroll
        for (int ni = 0; ni < 2; ++ni)
#pragma unroll
            for (int rg = 0; rg < 4; ++rg) w4[ni][rg] = *reinterpret_cast<const f16x4 *>(stg + (ni * 32 + rg * 8 + eh * 4) * 2);
        const f16x8 bv = *reinterpret_cast<const f16x8 *>(stg + 128 + piece * 2);
        const f16x8 gv = *reinterpret_cast<const f16x8 *>(stg + 256 + piece * 2);
        lanes_meet();
        // staging: 16 rows of 128 bytes, the 16-byte pieces of a row swizzled by the row so that neither side meets a bank twice
        uint8_t *const to = stg + (em & 15) * 128 + eh * 8;
        const int swz = (em & 15) >> 1;
        f16x4 hv[2][2][4]; /* [row-block, in turns][columns][...] */
        auto convert = [&](int mi, int ni) __attribute__((always_inline)) {
            const u32x2 both = __builtin_amdgcn_permlane32_swap(scales4, scales4, false, false);
            const float as = half_bits_to_float((mi % 2 == 0 ? both.x : both.y) >> (mi / 2 * 16) & 0xFFFFu) * kAccScale; /* exact: a power of two */
#pragma unroll
            for (int rg = 0; rg < 4; ++rg)
#pragma unroll
                for (int e = 0; e < 4; ++e) /* (fma(as, ws, -0) = fl(as * ws), the sign of a zero included: one v_fma_mix_f32, which reads the fp16 value as it lies) */
                    hv[mi & 1][ni][rg][e] = static_cast<_Float16>(acc[ni][mi][rg * 4 + e] * __builtin_fmaf(as, static_cast<float>(w4[ni][rg][e]), -0.0f));
        };
        convert(0, 0);
        convert(0, 1);
#pragma unroll
        for (int t = 0; t < 2 * MI; ++t) { /* rows 16t ... 16t + 15; the next row-block is converted while they come back from LDS */
            const int mi = t >> 1, half = t & 1;
            if ((em >> 4) == half) {
#pragma unroll
                for (int ni = 0; ni < 2; ++ni)
#pragma unroll
                    for (int rg = 0; rg < 4; ++rg) *reinterpret_cast<f16x4 *>(to + (((ni * 4 + rg) ^ swz) << 4)) = hv[mi & 1][ni][rg];
            }
            lanes_meet();
            if (TAIL && t + 1 < 2 * MI) fetch(t + 1);
            f16x8 o[2];
#pragma unroll
            for (int it = 0; it < 2; ++it) {
                const int row = it * 8 + srow;
                o[it] = *reinterpret_cast<const f16x8 *>(stg + row * 128 + (((el & 7) ^ (row >> 1)) << 4));
            }
            lanes_meet();
            __builtin_amdgcn_sched_barrier(0);
            if (mi + 1 < MI) convert(mi + 1, half);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int it = 0; it < 2; ++it) {
                o[it] += bv;
                if (TAIL) o[it] = rv[t & 1][it] + o[it] * gv;
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o[it]), out_rsrc, out_voff + (t * 16 + it * 8) * ldo * 2, 0, 2 /* nt */);
            }
        }
    };
    if constexpr (!ODD) {
        for (int strip = strip0 + wave; strip < strip1; strip += kWaves) work_strip(strip, a0, b0, raw0, a1, b1, raw1);
    } else { /* an odd number of K steps: every other strip starts with the other slot */
        for (int strip = strip0 + wave; strip < strip1; strip += 2 * kWaves) {
            work_strip(strip, a0, b0, raw0, a1, b1, raw1);
            if (strip + kWaves >= strip1) break;
            work_strip(strip + kWaves, a1, b1, raw1, a0, b0, raw0);
        }
    }
#endif
}

template <int MI, int NCH, int PRE>
int launch_cfg(const ResidentArgs &args, bool tail, hipStream_t s) {
    using Kernel = void (*)(const ResidentArgs);
    constexpr bool kTail = PRE == kPreNone; /* (see resident_takes) */
    const Kernel kernels[4] = {resident_linear_kernel<MI, NCH, PRE, false, false>, resident_linear_kernel<MI, NCH, PRE, kTail, false>,
                               resident_linear_kernel<MI, NCH, PRE, false, true>, resident_linear_kernel<MI, NCH, PRE, kTail, true>};
    const int which = (tail ? 1 : 0) + (args.kblocks / 2 % 2 ? 2 : 0);
    const int lds_bytes = args.kblocks * MI * kBlk + kWaves * kStage;
    constexpr int kMaxDevices = 64;
    static bool attr_done[kMaxDevices][4] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return fail(VDMQ_ELAUNCH, "no current HIP device");
    if (!attr_done[dev][which]) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernels[which]), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return fail(VDMQ_ELAUNCH, "hipFuncSetAttribute: %s", hipGetErrorString(e));
        attr_done[dev][which] = true;
    }
    const int64_t units = static_cast<int64_t>(args.tiles) * args.groups;
    const dim3 grid(static_cast<unsigned>(ceil_div(units, kXcds) * kXcds));
    hipLaunchKernelGGL(kernels[which], grid, dim3(kWaves * 64), lds_bytes, s, args);
    const int rc = check_launch("resident_linear_kernel");
    if (rc == VDMQ_OK) record_gemm_launch({VDMQ_KERNEL_LINEAR_RESIDENT, 32 * MI, kStripCols, 1, args.groups, 1, static_cast<int64_t>(grid.x)});
    return rc;
}

template <int MI, int NCH>
int launch_pre(const ResidentArgs &args, int pre, bool tail, hipStream_t s) {
    if constexpr (MI == 4) { /* (see resident_takes) */
        if (pre == kPreLnModulate) return launch_cfg<MI, NCH, kPreLnModulate>(args, tail, s);
        if (pre == kPreLnAffine) return launch_cfg<MI, NCH, kPreLnAffine>(args, tail, s);
    }
    return launch_cfg<MI, NCH, kPreNone>(args, tail, s);
}

// Token rows per workgroup (32 * mi) and column groups per row tile.  A unit -- the rows of a tile, quantized, against a group's
// strips -- takes, at K = 1536, about 2.5 us per 32 rows for the first part (8 with the LayerNorm, which is bound by its
// instructions) and, for the second, a pass of its eight waves over eight strips 10.6 / 8 / 6 us with 128 / 64 / 32 rows (32 rows load
// as many weight bytes as 128), half of them (a wave per SIMD) 6.3 / 5 / 4.  Fewer rows suit problems that give the chip's CUs no
// 128 each; among equals the fewer groups, each of which quantizes the tile again.  On 120 shapes of 64 ... 75637 rows, K 640 ...
// 1536, every candidate timed, the choice takes 1.2 % more than the best one in the geometric mean, 12 % at most.  (Figures fitted to 75 of
// them: 0.7 and 6 % there, 0.8 and 7 % on the others, but narrow outputs of many rows went to 32 rows at a time.)
struct ResidentShape {
    int mi, tiles, groups;
    int64_t rounds; /* of units on a CU */
    int64_t time;   /* estimate at K = 1536, in units of 0.1 us */
};
ResidentShape resident_shape(int64_t M, int64_t N, bool ln) {
    constexpr int64_t kCus = 256;
    const int64_t strips = N / kStripCols, quantize = ln ? 80 : 25;
    ResidentShape best = {0, 0, 0, 0, 0};
    const int mis[3] = {4, 2, 1}, full[3] = {106, 80, 60}, part[3] = {63, 50, 40};
    for (int i = 0; i < 3; ++i) {
        const int64_t tiles = ceil_div(M, 32 * mis[i]);
        // groups: around what makes one round of units, or 1 ... 4 where that is more than one
        const int64_t fill = kCus / tiles, most = fill > 4 ? (fill < strips ? fill : strips) : (4 < strips ? 4 : strips);
        for (int64_t g = fill > 4 && most > 5 ? most - 4 : 1; g <= most; ++g) {
            const int64_t per = ceil_div(strips, g), rest = per % kWaves, second = rest - kWaves / 2; /* of the last pass: waves that share a SIMD */
            const int64_t last = rest == 0 ? 0 : part[i] + (second > 0 ? (full[i] - part[i]) * second / (kWaves / 2) : 0);
            const int64_t unit = quantize * mis[i] + per / kWaves * full[i] + last;
            const int64_t rounds = ceil_div(tiles * g, kCus), time = rounds * unit;
            if (best.mi == 0 || time < best.time) best = {mis[i], static_cast<int>(tiles), static_cast<int>(g), rounds, time};
        }
    }
    return best;
}

}  // namespace

// The one-kernel linear's time at K = 1280 ... 1536, us: quantization and strips of its units as resident_shape counts them, output (and
// residual), what the XCDs fetch.  A residual that comes from memory -- rows in, residual and output together more than 500 MB; up to
// 450 MB the terms without it gave 1.04 ... 1.09 of what was measured, beyond 0.78 -- is waited for at every turn of the epilogue.  Fitted to
// the timings of bf6_two_kernels_us, within 0.91 ... 1.07 at 90 % of them.
static double resident_us(int64_t M, int64_t N, int64_t K, bool has_tail, const ResidentShape &s) {
    const double k = K / 1536.0, rows = M * K * 2e-6, w = N * K * 0.75e-6, out = M * N * 1e-6;
    const double quantize = 2.5 * s.mi * s.rounds, strips = s.time * 0.1 - quantize;
    const double by_rows = w + rows * (s.groups < kXcds ? s.groups : kXcds), by_weights = rows + w * (s.tiles < kXcds ? s.tiles : kXcds);
    const double fetch = by_rows < by_weights ? by_rows : by_weights;
    const double waits = M * (2 * K + 4 * N) > 500000000 ? strips : 0.0;
    if (!has_tail) {
        if (s.mi == 1) return 1.77 * quantize + 0.75 * strips * k + 0.83 * out + 0.022 * fetch;
        if (s.mi == 2) return 1.16 * quantize + 0.50 * strips * k + 0.41 * out + 0.119 * fetch;
        return 1.32 * quantize + 0.61 * strips * k + 0.26 * out + 0.035 * fetch;
    }
    if (s.mi == 1) return 1.50 * quantize + 0.84 * strips * k + 0.99 * out + 0.042 * fetch;
    if (s.mi == 2) return 1.30 * quantize + 0.39 * strips * k + 0.65 * out + 0.116 * fetch + 0.27 * waits;
    return 1.30 * quantize + 0.57 * strips * k + 0.48 * out + 0.045 * fetch + 0.47 * waits;
}

bool resident_takes(const ResidentProblem &p) {
    // Rows of up to 1536 elements fit LDS; shorter ones than VDMQ_LINEAR_BF6_MIN_K are the int8 path's.  In front of it no GELU, in its epilogue
    // what the models' blocks ask for (a residual, with one gate vector or none, without a LayerNorm): the rest is left to the quantizers'
    // and the GEMM's kernels.
    const GemmTail &t = p.tail;
    const bool tail = t.residual == nullptr ? t.gate == nullptr : (t.gate == nullptr || t.rows_per_gate >= p.M) && t.ldr <= (1 << 22) && p.ln_mode == 0;
    if (p.K < VDMQ_LINEAR_BF6_MIN_K || p.K > 1536 || p.M > (1 << 24) || p.out_dtype != VDMQ_OUT_F16 || p.act != VDMQ_ACT_NONE || !tail) return false;
    if (p.ln_mode == 0) {
        // Against quantizer and tiled GEMM it takes 0.5 ... 0.95 of the time as a rule, but it loses where their tiles fill the CUs exactly
        // and its units do not (2459 x 1536 -> 6144 with a residual 33.4 / 26.7 us, 679 x 1472 -> 13056 22.4 / 20.8), and with a residual
        // from memory in front of a wide output (11450 x 1536 -> 11136 203 / 164): so both are estimated.  Not slower, so not asked:
        // K < 1280 than the int8 path, which served those (6500 timings, 0.995 at most), N <= 384 (550, 1.03), few tiles with K divided
        // (vdmq_bf6_ksplit.hip; as calls 0.77 ... 0.83 of that one's time on 320 shapes).  On 2300 shapes of 2.5 ... 400 million outputs, each
        // timed with one set of buffers and with rows and weights of its own in every call, the choice takes 1.0035 of the faster
        // form's time in the geometric mean, over 1.06 at 2.3 % (always one kernel 1.0061 and 4.4 %, always two 1.20).
        // Two kernels count as never faster than 16 us, with gate and residual 20.5, which the host took for them when the line was drawn.  It
        // takes 11.5 now (one: 8.2), but the line stays: with 11.5 and 12 in its place 12 of 4000 problems of up to 40 million outputs
        // would be two kernels, and as one they take 0.87 ... 1.09 of that time on the GPU, 0.98 in the mean (1166 x 1472 -> 3200 with a residual 13.8 us as
        // one, 15.1 as two; the choice knowingly loses 205 x 1280 -> 30336, 16.3 and 15.0, and 230 x 1536 -> 14848, 13.9 and 12.9).  The tiled GEMM
        // stands for two kernels here, also where K = 1536 with a residual would be the pair kernel's (vdmq_bf6_pair.hip).  Up to 2.5
        // million outputs the estimates always say one kernel (2.8 million is the least where they do not), and the call waits for the
        // host, whom they cost 0.2 us each time.
        if (p.K < 1280 || p.N <= 384 || p.M * p.N <= 2500000 || ksplit_takes(p.M, p.N, p.K, p.out_dtype) || p.M * p.N > (int64_t(1) << 40)) return true;
        const ResidentShape shape = resident_shape(p.M, p.N, false);
        const double two = bf6_two_kernels_us(p.M, p.N, p.K, t.residual != nullptr), host = t.residual != nullptr ? 20.5 : 16.0;
        return resident_us(p.M, p.N, p.K, t.residual != nullptr, shape) < (two > host ? two : host);
    }
    // Behind a LayerNorm only where its instructions, repeated in each column group, cost less than the second launch and the
    // blocks' way through memory: in effect where a row tile is one workgroup's (K = 1536, us, here / as two kernels: 28000 -> 4608 128 /
    // 147, 32760 -> 1536 73 / 85, -> 8960 233 / 289; 4680 -> 4608 47 / 40, 40000 -> 4608 245 / 203).  Two kernels: 29 us for the
    // quantizer of 32760 rows, 13.4 us per 512 columns for the GEMM, 6 us for both launches, 12 us at least.
    const int64_t two = p.M * (290 + p.N * 134 / 512) / 32760 + 60;
    const ResidentShape shape = resident_shape(p.M, p.N, true);
    return shape.mi == 4 && shape.time + 30 < (two > 120 ? two : 120);
}

int launch_linear_resident(const ResidentProblem &p, hipStream_t s) {
    ResidentArgs a;
    a.x = p.x;
    a.ldx = p.ldx;
    a.w = p.wblocks;
    a.wscale = p.wscale;
    a.bias = p.bias;
    a.out = static_cast<__half *>(p.out);
    a.ldo = p.ldo;
    a.M = static_cast<int>(p.M);
    a.N = static_cast<int>(p.N);
    a.K = static_cast<int>(p.K);
    a.kblocks = static_cast<int>(bf6_kblocks(p.K));
    a.clip = p.clip;
    a.eps = p.eps;
    a.va = p.va;
    a.vb = p.vb;
    a.ldv = p.ldv;
    a.rows_per_vec = static_cast<int>(p.rows_per_vec);
    a.tail = p.tail;
    const int pre = p.ln_mode == VDMQ_LN_MODULATE ? kPreLnModulate : p.ln_mode == VDMQ_LN_AFFINE ? kPreLnAffine : kPreNone;
    const ResidentShape shape = resident_shape(p.M, p.N, p.ln_mode != 0);
    a.tiles = shape.tiles;
    a.groups = shape.groups;
    // Bytes that the XCDs fetch: the rows once and the weights on every XCD that has a row tile of its own, or the other way round
    // (140 x 1472 -> 12032: 15.8 us row tile by row tile, 9.4 group by group; 4096 x 1536 -> 4608 28.5 and 32.3).
    const int64_t x_bytes = 2 * p.M * p.K, w_bytes = p.N * p.K * 3 / 4;
    a.by_group = w_bytes + x_bytes * (a.groups < kXcds ? a.groups : kXcds) < x_bytes + w_bytes * (a.tiles < kXcds ? a.tiles : kXcds) ? 1 : 0;
    const bool tail = p.tail.residual != nullptr;
    if (p.K <= 1024) return shape.mi == 4 ? launch_pre<4, 2>(a, pre, tail, s) : shape.mi == 2 ? launch_pre<2, 2>(a, pre, tail, s) : launch_pre<1, 2>(a, pre, tail, s);
    return shape.mi == 4 ? launch_pre<4, 3>(a, pre, tail, s) : shape.mi == 2 ? launch_pre<2, 3>(a, pre, tail, s) : launch_pre<1, 3>(a, pre, tail, s);
}

}  // namespace vdmq
