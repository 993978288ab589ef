// W4A4 GEMM on bf6 blocks (vdmq_bf6.hip) for problems between few tiles and many, fp16 outputs: one output tile per CU, of the smallest of
// five sizes that gives the chip's 256 CUs at most one each, and two groups of four waves that take the tile's K in turns.
//
// 257 ... 512 tiles of 128 x 128 (vdmq_bf6.hip) are two on some CUs, which take two tiles' time however few they are, and just above
// that 256 x 256 tiles leave half the CUs idle.  A tile's operands go through LDS, in once and out again once for each wave that wants them.
// With K divided between two groups a wave owns a quarter of the tile and four waves instead of eight read a unit of 128 k; eight waves
// because four fetch only 30 ... 47 bytes per clock from L2, eight 60.  Cycles per unit by the counters (K = 7680 ... 15360), in brackets those in
// which the matrix pipes work: 128 x 160 562 (320), 128 x 192 624 (384), 192 x 160 819 (480), 192 x 192 927 (576); the tiled kernel's 128 x
// 128 with four waves 590 (256).  No pipe is full: of the 562 LDS works 216 for 55 KB of fragments, without a bank conflict, and 28 KB come in,
// 49 bytes per clock.  The sums of the two groups meet in LDS at the end (integers: exact in any order); with launch, first loads and
// stores what is not K loop takes 7.5 us of a 128 x 160 tile, 10 of a 192 x 192 one.  GEMM alone, us, tiled / here: 512 x 10240, K 5120 25.6 / 21.4; 1021 x 4224, K 7680 36.3 /
// 27.0; 3589 x 1152, K 10432 48.9 / 33.4; 4355 x 1408, K 8640 42.4 / 35.6; 5579 x 1536, K 11072 81.7 / 56.5.
#include <type_traits>

#include "vdmq_internal.h"

namespace vdmq {
namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kWaves = 8, kXcds = 8;
constexpr int kFrag = 1536; /* 16 rows x 128 k: [64 lanes x 16 bytes][64 lanes x 8 bytes] */

struct PairArgs {
    const uint8_t *x, *w;
    const __half *ascale, *wscale, *bias;
    __half *out;
    int64_t ldo;
    int M, N, kblocks;
    int tiles_m, tiles_n;
    int strip; /* tile rows of a strip */
    GemmTail tail;
};

// MB x NB blocks of 16 tokens x 16 channels per wave; 2 x 2 waves of a group make the tile.  SETS: of registers for a wave's fragments (one
// where two do not fit).
template <int MB_, int NB_, int SETS_>
struct Pair {
    static constexpr int kSets = SETS_;
    static constexpr int MB = MB_, NB = NB_, BM = 32 * MB, BN = 32 * NB, OB = MB / 2; /* OB: token blocks a wave keeps */
    static constexpr int kUnit = (2 * MB + 2 * NB) * kFrag;                            /* bytes of 128 k of the tile's operands */
    static constexpr int kLdsMax = 160 * 1024, S = (kLdsMax - 2048) / kUnit; /* units the ring holds */
    static constexpr int kMinUnits = S + 1; /* the K loop fills the ring in front and refills it at least once */
    static constexpr int kLoadsAll = kUnit / 1024, kLoads = (kLoadsAll + kWaves - 1) / kWaves;
    static constexpr int kArea = OB * NB * 1024, kStageRow = NB * 32 + 16;
    static constexpr int kSideBytes = (BM + 2 * BN) * 2; /* fp16 token scales, channel scales and bias */
    static constexpr int kSideAt = S * kUnit > kWaves * kArea ? S * kUnit : kWaves * kArea, kLds = kSideAt + kSideBytes;
    static_assert(MB % 2 == 0 && kUnit % 1024 == 0 && S >= 4 && S <= 5 && kLds <= kLdsMax, "the ring, the sums and the side vectors fit LDS");
    static_assert(OB * 16 * kStageRow <= kArea, "a wave's outputs are staged where it received its sums");
    static_assert(kLoads * (S - 2) < 64, "vmcnt is a 6-bit counter");
};

#if defined(__HIP_DEVICE_COMPILE__)
// The K loop.  A phase is the time between two barriers.  Unit u (128 k) belongs to group u % 2, whose waves read it from LDS in phase u, while
// they finish their previous unit, and work on it in phases u + 1 and u + 2: in every phase one group is in its first half and
// the other, which reads, in its second.  The loads of phase p fill the slot that unit p - 1 has left.
template <class Cfg>
struct PairKLoop {
    static constexpr int MB = Cfg::MB, NB = Cfg::NB, OB = Cfg::OB, S = Cfg::S, kSets = Cfg::kSets, kHalf = (NB + 1) / 2, kRing = S * Cfg::kUnit;
    using Acc = v4f[NB][MB];
    using XFrags = v8i[MB];
    using WFrags = v8i[NB - 1];
    uint8_t *lds;
    const __amdgpu_buffer_rsrc_t (&src)[Cfg::kLoads];
    const uint32_t (&lane_off)[Cfg::kLoads];
    int wave;
    int lane_a, lane_b, at_w, at_x0, at_x1; /* bytes within a unit */
    int units;

    struct Place { /* phase, and the bytes in the ring of the slots of its unit and of the one before */
        int p, cur, fill;
    };
    static __device__ __forceinline__ void advance(Place &at) {
        ++at.p;
        at.fill = at.cur;
        at.cur = at.cur + Cfg::kUnit == kRing ? 0 : at.cur + Cfg::kUnit;
    }
    __device__ __forceinline__ void load_one(int i, int u, int slot) const {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(src[i], (__attribute__((address_space(3))) void *)(lds + slot + (i * kWaves + wave) * 1024), 16, lane_off[i],
                                                 u * (2 * kBf6PanelKb), 0, 0);
    }
    // End of a phase: unit p + 1 has landed (STEADY: the loads of S - 2 younger units are in flight), and this wave's reads of the slot that
    // is filled next are done.
    template <int L, bool STEADY, bool READ>
    __device__ __forceinline__ void end_phase(Place &at) const {
        constexpr int lgkm = READ ? 0 : 15;
        const int n = units - 2 - at.p;
        if (STEADY || n >= S - 2) __builtin_amdgcn_s_waitcnt(waitcnt_imm((S - 2) * L, lgkm));
        else if (S == 5 && n == 2) __builtin_amdgcn_s_waitcnt(waitcnt_imm(2 * L, lgkm));
        else if (n == 1) __builtin_amdgcn_s_waitcnt(waitcnt_imm(L, lgkm));
        else __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, lgkm));
        lds_barrier();
        advance(at);
    }
    __device__ __forceinline__ v8i frag(uint32_t a, uint32_t b, int f) const {
        b += f * kFrag;
        asm volatile("" : "+v"(b)); /* (the compiler would read two fragments' second parts at once and move them into place) */
        const u32x4 va = *reinterpret_cast<const u32x4 *>(lds + a + f * kFrag);
        const u32x2 vb = *reinterpret_cast<const u32x2 *>(lds + b);
        return v8i{(int)va.x, (int)va.y, (int)va.z, (int)va.w, (int)vb.x, (int)vb.y, 0, 0};
    }
    // One phase: SECOND half of the wave's present unit.  WORK: matrix instructions on it; READ: the wave's next unit into registers, a
    // weight fragment when the present one has had its last use, the token fragments and the last weight fragment into registers
    // of their own (kSets == 2), so that no read is issued behind the phase's last matrix instructions, or, with larger tiles, as the
    // present ones have had theirs.
    template <int L, bool STEADY, bool SECOND, bool READ, bool WORK>
    __device__ __forceinline__ void phase(Place &at, Acc &acc, WFrags &wf, v8i &wl, XFrags &x, v8i &wln, XFrags &xn) const {
        const int u = at.p - 1 + S;
        const bool load = STEADY || (at.p >= 1 && u < units);
        constexpr bool ahead = kSets == 2 || !WORK;
        constexpr int j0 = SECOND ? kHalf : 0, j1 = SECOND ? NB : kHalf, turns = j1 - j0;
        const uint32_t wa = at.cur + at_w + lane_a, wb = at.cur + at_w + lane_b, xa = at.cur + lane_a, xb = at.cur + lane_b;
        auto read_x = [&](int i) __attribute__((always_inline)) { xn[i] = i < OB ? frag(xa + at_x0, xb + at_x0, i) : frag(xa + at_x1, xb + at_x1, i - OB); };
        if (READ) {
            if (ahead) {
#pragma unroll
                for (int i = 0; i < MB; ++i) read_x(i);
            }
#pragma unroll
            for (int j = 0; j < kHalf; ++j) wf[j] = frag(wa, wb, j);
            if (ahead) wln = frag(wa, wb, NB - 1);
        }
        if (WORK) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = j0; j < j1; ++j) {
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                if (WORK) acc[j][i] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(j == NB - 1 ? wl : wf[j < NB - 1 ? j : 0], x[i], acc[j][i], 3, 3, 0, 0, 0, 0);
                if (READ && !ahead && j == NB - 1) read_x(i);
            }
            if (READ && j < NB - 1) wf[j < NB - 1 ? j : 0] = frag(wa, wb, j);
            if (READ && !ahead && j == NB - 1) wln = frag(wa, wb, j);
            if (load) {
#pragma unroll
                for (int i = 0; i < L; ++i)
                    if (i * turns / L == j - j0) load_one(i, u, at.fill);
            }
            if (WORK) __builtin_amdgcn_sched_barrier(0);
        }
        end_phase<L, STEADY, READ>(at);
    }
    template <int L, bool STEADY>
    __device__ __forceinline__ void unit(Place &at, Acc &acc, WFrags &wf, v8i &wl, XFrags &x, v8i &wln, XFrags &xn) const {
        phase<L, STEADY, false, false, true>(at, acc, wf, wl, x, wln, xn);
        phase<L, STEADY, true, true, true>(at, acc, wf, wl, x, wln, xn);
    }
    template <int L, class Hook>
    __device__ __forceinline__ void run(Acc &acc, int group, Hook &&first_read) const {
#pragma unroll
        for (int u = 0; u < S; ++u)
#pragma unroll
            for (int i = 0; i < L; ++i) load_one(i, u, u * Cfg::kUnit);
        __builtin_amdgcn_s_waitcnt(waitcnt_imm((S - 1) * L, 15));
        lds_barrier();
        Place at = {0, 0, kRing - Cfg::kUnit};
        if (group == 1) end_phase<L, false, false>(at);
        WFrags wf;
        XFrags x0;
        v8i w0;
        phase<L, false, true, true, false>(at, acc, wf, w0, x0, w0, x0);
        first_read();
        if constexpr (kSets == 2) {
            XFrags x1;
            v8i w1;
            for (; at.p + S + 3 <= units;) { /* two units: the sets of registers in turn */
                unit<L, true>(at, acc, wf, w0, x0, w1, x1);
                unit<L, true>(at, acc, wf, w1, x1, w0, x0);
            }
            for (; at.p + 1 < units;) {
                unit<L, false>(at, acc, wf, w0, x0, w1, x1);
#pragma unroll
                for (int i = 0; i < MB; ++i) x0[i] = x1[i];
                w0 = w1;
            }
        } else {
            for (; at.p + S + 1 <= units;) unit<L, true>(at, acc, wf, w0, x0, w0, x0);
            for (; at.p + 1 < units;) unit<L, false>(at, acc, wf, w0, x0, w0, x0);
        }
        // the wave's last unit; the other group may still have one to read
        const bool other = at.p < units;
        auto last = [&](int j0, int j1) __attribute__((always_inline)) {
#pragma unroll
            for (int j = j0; j < j1; ++j)
#pragma unroll
                for (int i = 0; i < MB; ++i)
                    acc[j][i] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(j == NB - 1 ? w0 : wf[j < NB - 1 ? j : 0], x0[i], acc[j][i], 3, 3, 0, 0, 0, 0);
        };
        last(0, kHalf);
        if (other) end_phase<L, false, false>(at);
        last(kHalf, NB);
    }
};
#endif

template <class Cfg, bool TAIL>
__global__ __launch_bounds__(kWaves * 64, 2) void gemm_bf6_pair_kernel(const PairArgs args) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int MB = Cfg::MB, NB = Cfg::NB, OB = Cfg::OB, L = Cfg::kLoads;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int group = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1; /* (waves w and w + 4 share a SIMD) */
    // tiles: strips of `strip` tile rows, column by column; an eighth of the sequence for each XCD
    const int tiles = args.tiles_m * args.tiles_n, xcd = blockIdx.x % kXcds, slot0 = blockIdx.x / kXcds;
    const int first = static_cast<int>(static_cast<int64_t>(tiles) * xcd / kXcds), last = static_cast<int>(static_cast<int64_t>(tiles) * (xcd + 1) / kXcds);
    const int tile = first + slot0;
    if (tile >= last) return;
    const int in_strips = args.strip * args.tiles_n, st = tile / in_strips, at = tile - st * in_strips;
    const int strip_rows = min(args.strip, args.tiles_m - st * args.strip), tile_n = at / strip_rows, tile_m = st * args.strip + at - tile_n * strip_rows;
    const int m0 = tile_m * Cfg::BM, n0 = tile_n * Cfg::BN;
    const int kblocks = args.kblocks, units = kblocks / 2;

    // global -> LDS: a unit is NB weight and MB token row-blocks of 32 rows x 128 k, 3 KiB each; this wave's i-th load fills KiB
    // i * 8 + wave of it.  Rows beyond the last row-block: that one again, never stored.
    __amdgpu_buffer_rsrc_t src[L];
    uint32_t lane_off[L];
    const int last_rb_m = (args.M + 31) / 32 - 1, last_rb_n = args.N / 32 - 1;
#pragma unroll
    for (int i = 0; i < L; ++i) {
        const int idx = i * kWaves + wave, q = idx / 3;
        const int off = (idx % 3) * 1024 + lane * 16, frag = off / kFrag, in = off % kFrag;
        const bool part_b = in >= 1024;
        const int l = part_b ? (in - 1024) / 8 : in / 16; /* lane of the operand: row % 16 + 16 * (k / 32) */
        const int64_t rb = q < NB ? min(tile_n * NB + q, last_rb_n) : min(tile_m * MB + q - NB, last_rb_m);
        src[i] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>((q < NB ? args.w : args.x) + bf6_piece(rb * 32, 0, 0, false, kblocks)), 0,
                                                   4 * kblocks * kBf6PanelKb, 0x00020000);
        lane_off[i] = static_cast<uint32_t>(bf6_piece(frag * 16 + (l & 15), l >> 5, (l >> 4) & 1, part_b, kblocks));
    }
    // The tile's token scales, channel scales and bias, fp16, for the epilogue: asked for in front of the operands
    constexpr int kSide = Cfg::BM + 2 * Cfg::BN, kSideLoads = (kSide + kWaves * 64 - 1) / (kWaves * 64);
    _Float16 side[kSideLoads];
#pragma unroll
    for (int i = 0; i < kSideLoads; ++i) {
        const int at = i * kWaves * 64 + static_cast<int>(threadIdx.x), n = n0 + (at - Cfg::BM) % Cfg::BN;
        const __half *from = at < Cfg::BM ? args.ascale + min(m0 + at, args.M - 1) : at < Cfg::BM + Cfg::BN ? args.wscale + min(n, args.N - 1) : args.bias + min(n, args.N - 1);
        side[i] = static_cast<_Float16>(-0.0f); /* no bias: the one value whose addition changes no bit */
        if (at < Cfg::BM + Cfg::BN || (at < kSide && args.bias != nullptr)) side[i] = *reinterpret_cast<const _Float16 *>(from);
    }
    v4f acc[NB][MB];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int i = 0; i < MB; ++i) acc[j][i] = v4f{0.f, 0.f, 0.f, 0.f};
    // Token blocks: the wave of the second group starts its own numbering with the second half, so that what it keeps and what it hands
    // over in the end has the same place in either group's registers.
    const PairKLoop<Cfg> loop{lds, src, lane_off, wave, lane * 16, 1024 + lane * 8, wn * NB * kFrag, (2 * NB + wm * MB + group * OB) * kFrag,
                              (2 * NB + wm * MB + (1 - group) * OB) * kFrag, units};
    _Float16 *const side_lds = reinterpret_cast<_Float16 *>(lds + Cfg::kSideAt);
    auto keep_side = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kSideLoads; ++i) {
            const int at = i * kWaves * 64 + static_cast<int>(threadIdx.x);
            if (kSide % (kWaves * 64) == 0 || at < kSide) side_lds[at] = side[i];
        }
    };
    if (Cfg::kLoadsAll % kWaves == 0 || (L - 1) * kWaves + wave < Cfg::kLoadsAll) loop.template run<L>(acc, group, keep_side);
    else loop.template run<L - 1>(acc, group, keep_side);

    // ---- the groups' sums: a wave keeps its first OB token blocks and takes those of its partner in the other group, which takes
    // the rest; meanwhile the vectors of the epilogue are on their way
    const GemmTail &tail = args.tail;
    constexpr int P = Cfg::BN / 8, kPieces = Cfg::BM * P, kTurns = (kPieces + kWaves * 64 - 1) / (kWaves * 64); /* 16-byte pieces of a row, of the tile; a thread's */
    f16x8 gv[kTurns], rv[kTurns];
    auto place = [&](int it, int &row, int &piece) __attribute__((always_inline)) {
        const int idx = it * kWaves * 64 + static_cast<int>(threadIdx.x);
        row = idx / P;
        piece = idx % P;
        return (kPieces % (kWaves * 64) == 0 || idx < kPieces) && m0 + row < args.M && n0 + piece * 8 < args.N;
    };
    if (TAIL) {
#pragma unroll
        for (int it = 0; it < kTurns; ++it) {
            int row, piece;
            if (!place(it, row, piece)) continue;
            const int m = m0 + row, n = n0 + piece * 8;
            if (tail.gate != nullptr) {
                const int64_t grow = tail.rows_per_gate == 1 ? m : tail.rows_per_gate >= args.M ? 0 : m / tail.rows_per_gate;
                gv[it] = *reinterpret_cast<const f16x8 *>(tail.gate + grow * tail.ldg + n);
            }
            if (tail.residual != nullptr) rv[it] = *reinterpret_cast<const f16x8 *>(tail.residual + m * tail.ldr + n);
        }
    }
    uint8_t *const to = lds + (wave ^ 4) * Cfg::kArea + lane * 16, *const mine = lds + wave * Cfg::kArea;
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int i = 0; i < OB; ++i) *reinterpret_cast<v4f *>(to + (j * OB + i) * 1024) = acc[j][OB + i];
    __syncthreads();
    float as[OB];
    f16x4 w4[NB], b4[NB];
    const int l16 = lane & 15, l4 = lane >> 4;
#pragma unroll
    for (int i = 0; i < OB; ++i) as[i] = static_cast<float>(side_lds[(wm * MB + group * OB + i) * 16 + l16]) * 256.0f; /* the blocks hold q / 16 */
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const _Float16 *const at = side_lds + Cfg::BM + (wn * NB + j) * 16 + l4 * 4;
        w4[j] = *reinterpret_cast<const f16x4 *>(at);
        b4[j] = *reinterpret_cast<const f16x4 *>(at + Cfg::BN);
    }
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int i = 0; i < OB; ++i) acc[j][i] += *reinterpret_cast<const v4f *>(mine + (j * OB + i) * 1024 + lane * 16);
    asm volatile("" ::: "memory"); /* (the compiler reasons about one lane alone: every lane has read before one writes) */
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int i = 0; i < OB; ++i) {
            f16x4 h;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                h[e] = static_cast<_Float16>(acc[j][i][e] * (as[i] * static_cast<float>(w4[j][e])));
            *reinterpret_cast<f16x4 *>(mine + (i * 16 + l16) * Cfg::kStageRow + (j * 16 + l4 * 4) * 2) = h + b4[j];
        }
    __syncthreads();
    // ---- the tile's rows leave as a whole
#pragma unroll
    for (int it = 0; it < kTurns; ++it) {
        int row, piece;
        if (!place(it, row, piece)) continue;
        const int owner = (row / (OB * 16) % 2) * 4 + row / (MB * 16) * 2 + piece / (NB * 2);
        const int m = m0 + row, n = n0 + piece * 8;
        f16x8 hv = *reinterpret_cast<const f16x8 *>(lds + owner * Cfg::kArea + row % (OB * 16) * Cfg::kStageRow + piece % (NB * 2) * 16);
        if (TAIL && tail.gate != nullptr) hv *= gv[it];
        if (TAIL && tail.residual != nullptr) hv = rv[it] + hv;
        const int part = tail.split_cols != 0 ? n / tail.split_cols : 0;
        *reinterpret_cast<f16x8 *>(args.out + part * tail.part_stride + static_cast<int64_t>(m) * args.ldo + (n - part * tail.split_cols)) = hv;
    }
#endif
}

template <class Cfg>
int launch_cfg(PairArgs &args, hipStream_t s) {
    using Kernel = void (*)(const PairArgs);
    const Kernel kernels[2] = {gemm_bf6_pair_kernel<Cfg, false>, gemm_bf6_pair_kernel<Cfg, true>};
    const bool has_tail = args.tail.gate != nullptr || args.tail.residual != nullptr;
    if (args.kblocks / 2 < Cfg::kMinUnits) return fail(VDMQ_ESHAPE, "gemm_bf6_pair_kernel needs K >= %d", 128 * Cfg::kMinUnits - 127);
    args.tiles_m = static_cast<int>(ceil_div(args.M, Cfg::BM));
    args.tiles_n = static_cast<int>(ceil_div(args.N, Cfg::BN));
    const int tiles = args.tiles_m * args.tiles_n, per_xcd = static_cast<int>(ceil_div(tiles, kXcds));
    // strip height: the fewest operand rows that an XCD's run of tiles takes in
    int best = 1;
    int64_t least = -1;
    for (int strips = 1; strips <= args.tiles_m; ++strips) {
        const int rows = static_cast<int>(ceil_div(args.tiles_m, strips));
        const int64_t cost = static_cast<int64_t>(rows < per_xcd ? rows : per_xcd) * Cfg::BM * 2 + (2 * per_xcd + rows) / rows * Cfg::BN;
        if (least < 0 || cost < least) {
            least = cost;
            best = rows;
        }
        if (rows == 1) break;
    }
    args.strip = best;
    constexpr int kMaxDevices = 64;
    static bool attr_done[kMaxDevices][2] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return fail(VDMQ_ELAUNCH, "no current HIP device");
    if (!attr_done[dev][has_tail]) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernels[has_tail]), hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::kLds);
        if (e != hipSuccess) return fail(VDMQ_ELAUNCH, "hipFuncSetAttribute: %s", hipGetErrorString(e));
        attr_done[dev][has_tail] = true;
    }
    const dim3 grid(static_cast<unsigned>(per_xcd * kXcds));
    hipLaunchKernelGGL(kernels[has_tail], grid, dim3(kWaves * 64), Cfg::kLds, s, args);
    const int rc = check_launch("gemm_bf6_pair_kernel");
    if (rc == VDMQ_OK) record_gemm_launch({VDMQ_KERNEL_GEMM_BF6_PAIR, Cfg::BM, Cfg::BN, args.strip, 1, 1, static_cast<int64_t>(grid.x)});
    return rc;
}

}  // namespace

// Tile by the number of workgroups.  The smaller the tile, the less a CU has to do, so: the smallest of which the chip holds all; K has
// to be long enough for what the sums' exchange costs.  Time here over that of the tiled kernel's choice, 300 problems of 3 ... 10
// million outputs and K 1536 ... 13824, without / with a residual: 128 x 160 from K = 1984 (1536) on 0.68 ... 0.98, below 1.0 ... 1.04;
// 128 x 192 and 192 x 128 from 3328 (2600) 0.71 ... 0.97, 1.0 ... 1.14; 192 x 160 from 7424 0.87 ... 0.95, 1.0 ... 1.18; 192 x 192, in place of
// the 256 x 256 tiles of more than 512 small ones, from 2600 0.69 ... 0.97, 0.95 ... 1.01.  256 small tiles or fewer, a CU each, are 0.97 ... 1.2.
static int pair_tile(int64_t M, int64_t N, int64_t K, bool has_tail) {
    constexpr int64_t kCus = 256;
    const int64_t small = ceil_div(M, 128) * ceil_div(N, 128);
    if (small <= kCus || M > (1 << 20)) return 0;
    if (ceil_div(M, 128) * ceil_div(N, 160) <= kCus) return K >= (has_tail ? 1536 : 1984) ? 1 : 0;
    const bool wide = ceil_div(M, 128) * ceil_div(N, 192) <= kCus;
    if (wide || ceil_div(M, 192) * ceil_div(N, 128) <= kCus) return K < (has_tail ? 2600 : 3328) ? 0 : wide ? 2 : 3;
    if (ceil_div(M, 192) * ceil_div(N, 160) <= kCus && small <= 2 * kCus) return K >= 7424 ? 4 : 0;
    return small > 2 * kCus && ceil_div(M, 192) * ceil_div(N, 192) <= kCus && K >= 2600 ? 5 : 0;
}

bool pair_takes(int64_t M, int64_t N, int64_t K, int out_dtype, const GemmTail &tail) {
    return out_dtype == VDMQ_OUT_F16 && pair_tile(M, N, K, tail.gate != nullptr || tail.residual != nullptr) != 0;
}

int launch_gemm_bf6_pair(const uint8_t *xblocks, const __half *ascale, const uint8_t *wblocks, const __half *wscale, const __half *bias, void *out, int64_t M,
                         int64_t N, int64_t K, int64_t ldo, const GemmTail &tail, hipStream_t s) {
    PairArgs a;
    a.x = xblocks;
    a.w = wblocks;
    a.ascale = ascale;
    a.wscale = wscale;
    a.bias = bias;
    a.out = static_cast<__half *>(out);
    a.ldo = ldo;
    a.M = static_cast<int>(M);
    a.N = static_cast<int>(N);
    a.kblocks = static_cast<int>(bf6_kblocks(K));
    a.tail = tail;
    switch (pair_tile(M, N, K, tail.gate != nullptr || tail.residual != nullptr)) {
        case 1: return launch_cfg<Pair<4, 5, 2>>(a, s);
        case 2: return launch_cfg<Pair<4, 6, 2>>(a, s);
        case 3: return launch_cfg<Pair<6, 4, 2>>(a, s);
        case 4: return launch_cfg<Pair<6, 5, 1>>(a, s);
        default: return launch_cfg<Pair<6, 6, 1>>(a, s);
    }
}

}  // namespace vdmq
