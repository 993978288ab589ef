// W4A4 GEMM on bf6 blocks (vdmq_bf6.hip) for problems that give the chip's 256 CUs at most one output tile each, fp16 outputs: small
// tiles, whose four waves all work on the whole tile and divide K among themselves.
//
// Such a problem takes as long as one tile does, and the 128 x 128 tiles of vdmq_bf6.hip walk their K in steps of two k-blocks with a
// barrier and 620 cycles each, LDS passing every operand byte twice and twice again (512 x 13824 -> 5120 and 100 x 13824 -> 5120 both
// 33 ... 35 us: 108 such steps).  Here a k-block's strings are wanted by one wave alone, so they go from L2 straight into its
// registers, three k-blocks ahead, without LDS and without a barrier; the waves meet once, to add up their sums (integers: exact in
// any order).  What bounds it is that way into the registers, at 44 bytes per clock and CU of 64 (a 128 x 128 tile of this form would
// take as long as one of the others; its first loads, its sums' exchange and its epilogue cost 5 us).  Smaller tiles fetch less
// per CU as long as each CU has at most one: GEMM alone, us, 128 x 128 tiles -> here: 100 x 13824 -> 5120 32.6 / 18.6, 300 x 8960 ->
// 1536 21.1 / 12.1, 256 x 5120 -> 4096 12.4 / 8.9 (64 x 64); 537 x 12544 -> 2944 31.0 / 25.7, 512 x 5120 -> 4096 15.0 / 13.9 (128 x 64).
#include <type_traits>

#include "vdmq_internal.h"

namespace vdmq {
namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kWaves = 4, kXcds = 8, kTileBytes = 4096; /* one 32 x 32 block of fp32 sums */

struct KsplitArgs {
    const uint8_t *x, *w;
    const __half *ascale, *wscale, *bias;
    __half *out;
    int64_t ldo;
    int M, N, kblocks;
    int tiles_m, tiles_n;
    int by_column; /* order of the units */
    GemmTail tail;
};

// MI x NJ blocks of 32 tokens x 32 channels per workgroup; at the end wave w owns OJ of them, of row w % MI, column group w / MI.
template <int MI_, int NJ_>
struct Ksplit {
    static constexpr int MI = MI_, NJ = NJ_, RN = kWaves / MI, OJ = NJ / RN;
    static constexpr int kAreaBytes = kWaves * OJ * kTileBytes, kLdsBytes = 3 * kAreaBytes;
    static constexpr int kStageRow = OJ * 64 + 16;
    static_assert(MI % 2 == 0 && kWaves % MI == 0 && NJ % RN == 0 && NJ % 2 == 0 && 128 % (NJ * 32) == 0, "the blocks divide among the waves, the columns among the tiles");
    static_assert(32 * kStageRow <= OJ * kTileBytes && kLdsBytes <= 160 * 1024, "a wave's staging lies in its part of an area");
};

#if defined(__HIP_DEVICE_COMPILE__)
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_mov(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, 0xF, 0xF, true));
}
// (the compiler reasons about one lane alone and must not move LDS accesses of one wave's lanes across this)
__device__ __forceinline__ void lanes_meet() { asm volatile("" ::: "memory"); }

#endif

template <class Cfg, bool TAIL>
__global__ __launch_bounds__(kWaves * 64, 1) void gemm_bf6_ksplit_kernel(const KsplitArgs args) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int MI = Cfg::MI, NJ = Cfg::NJ, RM = MI, RN = Cfg::RN, OJ = Cfg::OJ;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, lh = lane >> 5;
    const bool odd = (lane & 1) != 0;
    const int units = args.tiles_m * args.tiles_n, xcd = blockIdx.x % kXcds, slot = blockIdx.x / kXcds;
    const int first = static_cast<int>(static_cast<int64_t>(units) * xcd / kXcds), last = static_cast<int>(static_cast<int64_t>(units) * (xcd + 1) / kXcds);
    const int unit = first + slot;
    if (unit >= last) return;
    const int inner = args.by_column ? args.tiles_m : args.tiles_n, outer_at = unit / inner, inner_at = unit - outer_at * inner;
    const int tile_m = args.by_column ? inner_at : outer_at, tile_n = args.by_column ? outer_at : inner_at;
    const int kblocks = args.kblocks, rb_bytes = 4 * kblocks * kBf6PanelKb;
    // Row-blocks: wave w starts its own numbering at its own ones, so that what it keeps and what it hands to whom in the
    // end has the same place in every wave's registers.  Rows beyond the last block: that one again, never stored.
    const int rot_m = wave % RM, rot_n = (wave / RM) * OJ;
    const int last_m = min((args.M + 31) / 32 - 1 - tile_m * MI, MI - 1);
    auto block_m = [&](int i) __attribute__((always_inline)) { const int b = i + rot_m; return min(b >= MI ? b - MI : b, last_m); };
    auto block_n = [&](int j) __attribute__((always_inline)) { const int b = j + rot_n; return b >= NJ ? b - NJ : b; };
    const uint8_t *const xbase = args.x + static_cast<int64_t>(tile_m) * MI * rb_bytes, *const wbase = args.w + static_cast<int64_t>(tile_n) * NJ * rb_bytes;
    const uint32_t panel = (l32 >> 3) * kblocks * kBf6PanelKb;
    const uint32_t lane_a = panel + lh * 128 + (l32 & 7) * 16;
    const uint32_t lane_pair = panel + 256 + lh * 64 + (l32 & 6) * 8;
    uint32_t pair_m[MI / 2], pair_n[NJ / 2];
#pragma unroll
    for (int p = 0; p < MI / 2; ++p) pair_m[p] = lane_pair + (odd ? block_m(2 * p + 1) : block_m(2 * p)) * rb_bytes;
#pragma unroll
    for (int p = 0; p < NJ / 2; ++p) pair_n[p] = lane_pair + (odd ? block_n(2 * p + 1) : block_n(2 * p)) * rb_bytes;

    // the wave's k-blocks: wave, wave + 4, ...; beyond the last one nothing is read and the strings are zeros
    int load_kb = wave;
    auto rsrc = [&](const uint8_t *base, int blocks) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(base), 0, load_kb < kblocks ? blocks * rb_bytes : 0, 0x00020000);
    };
    auto load_x = [&](u32x4 &v, int i) __attribute__((always_inline)) {
        v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc(xbase, last_m + 1), lane_a, block_m(i) * rb_bytes + load_kb * kBf6PanelKb, 0));
    };
    auto load_w = [&](u32x4 &v, int j) __attribute__((always_inline)) {
        v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc(wbase, NJ), lane_a, block_n(j) * rb_bytes + load_kb * kBf6PanelKb, 0));
    };
    auto load_x_rest = [&](u32x4 (&pair)[MI / 2]) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < MI / 2; ++p) pair[p] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc(xbase, last_m + 1), pair_m[p], load_kb * kBf6PanelKb, 0));
    };
    auto load_w_rest = [&](u32x4 (&pair)[NJ / 2]) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < NJ / 2; ++p) pair[p] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc(wbase, NJ), pair_n[p], load_kb * kBf6PanelKb, 0));
    };
    auto untangle = [&](u32x2 &b0, u32x2 &b1, const u32x4 &raw) __attribute__((always_inline)) { /* neighbouring lanes hand each other the parts they loaded for the other */
        const uint32_t t0 = dpp_mov<0xB1>(odd ? raw.x : raw.z), t1 = dpp_mov<0xB1>(odd ? raw.y : raw.w);
        b0 = odd ? u32x2{t0, t1} : u32x2{raw.x, raw.y};
        b1 = odd ? u32x2{raw.z, raw.w} : u32x2{t0, t1};
    };
    using XA = u32x4[MI];
    using WA = u32x4[NJ];
    using XP = u32x4[MI / 2];
    using WP = u32x4[NJ / 2];
    v16f acc[NJ][MI];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[j][i][r] = 0.f;
    XA xa0, xa1, xa2;
    WA wa0, wa1, wa2;
    XP xp0, xp1, xp2;
    WP wp0, wp1, wp2;
    auto fill = [&](XA &xa, WA &wa, XP &xp, WP &wp) __attribute__((always_inline)) {
        load_x_rest(xp);
        load_w_rest(wp);
#pragma unroll
        for (int i = 0; i < MI; ++i) load_x(xa[i], i);
#pragma unroll
        for (int j = 0; j < NJ; ++j) load_w(wa[j], j);
        load_kb += kWaves;
    };
    // One k-block: MI * NJ matrix instructions on one slot, which is filled again, for the wave's third k-block after it, as its registers
    // become free.
    auto work = [&](XA &xa, WA &wa, XP &xp, WP &wp) __attribute__((always_inline)) {
        u32x2 xb[MI], wb[NJ];
#pragma unroll
        for (int p = 0; p < NJ / 2; ++p) untangle(wb[2 * p], wb[2 * p + 1], wp[p]);
#pragma unroll
        for (int p = 0; p < MI / 2; ++p) untangle(xb[2 * p], xb[2 * p + 1], xp[p]);
        load_x_rest(xp);
        load_w_rest(wp);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const v8i wf = {(int)wa[j].x, (int)wa[j].y, (int)wa[j].z, (int)wa[j].w, (int)wb[j].x, (int)wb[j].y, 0, 0};
                const v8i xf = {(int)xa[i].x, (int)xa[i].y, (int)xa[i].z, (int)xa[i].w, (int)xb[i].x, (int)xb[i].y, 0, 0};
                acc[j][i] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wf, xf, acc[j][i], 3, 3, 0, 0, 0, 0);
                if (j == NJ - 1) load_x(xa[i], i);
            }
            load_w(wa[j], j);
            __builtin_amdgcn_sched_barrier(0);
        }
        load_kb += kWaves;
    };
    fill(xa0, wa0, xp0, wp0);
    fill(xa1, wa1, xp1, wp1);
    fill(xa2, wa2, xp2, wp2);
    __builtin_amdgcn_sched_barrier(0);
    for (int left = (kblocks + kWaves - 1) / kWaves; left > 0; left -= 3) { /* (past the wave's last one: zeros) */
        work(xa0, wa0, xp0, wp0);
        work(xa1, wa1, xp1, wp1);
        work(xa2, wa2, xp2, wp2);
    }

    // ---- the waves' sums: each collects those of the blocks it owns (local row-block 0, columns 0 ... OJ - 1) from the three
    // others, while the vectors of its epilogue are on their way
    const int m0 = (tile_m * MI + rot_m) * 32, n0 = (tile_n * NJ + rot_n) * 32, rows = args.M - m0; /* (rows <= 0: nothing is stored) */
    const GemmTail &tail = args.tail;
    constexpr int P = OJ * 4, kTurns = P / 2; /* 16-byte pieces of a row; passes of the wave over 32 rows */
    const int srow = lane / P, piece = (lane % P) * 8;
    const float as = static_cast<float>(reinterpret_cast<const _Float16 *>(args.ascale)[min(m0 + l32, args.M - 1)]) * 256.0f; /* the blocks hold q / 16 */
    f16x4 w4[OJ][4];
#pragma unroll
    for (int j = 0; j < OJ; ++j)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) w4[j][rg] = *reinterpret_cast<const f16x4 *>(args.wscale + n0 + j * 32 + rg * 8 + lh * 4);
    f16x8 bv = {0, 0, 0, 0, 0, 0, 0, 0}, gv[kTurns], rv[kTurns];
    if (args.bias != nullptr) bv = *reinterpret_cast<const f16x8 *>(args.bias + n0 + piece);
    else bv = -bv; /* the one value whose addition changes no bit */
    if (TAIL) {
#pragma unroll
        for (int it = 0; it < kTurns; ++it) {
            const int64_t m = min(m0 + it * (64 / P) + srow, args.M - 1);
            if (tail.gate != nullptr) gv[it] = *reinterpret_cast<const f16x8 *>(tail.gate + (tail.rows_per_gate == 1 ? m : static_cast<int>(m) / tail.rows_per_gate) * tail.ldg + n0 + piece);
            if (tail.residual != nullptr) rv[it] = *reinterpret_cast<const f16x8 *>(tail.residual + m * tail.ldr + n0 + piece);
        }
    }
    auto area = [&](int r, int owner) __attribute__((always_inline)) { return lds + ((r - 1) * kWaves + owner) * OJ * kTileBytes + lane * 16; };
    auto send = [&](auto rc) __attribute__((always_inline)) {
        constexpr int r = decltype(rc)::value, ri = r % RM, rj = r / RM;
        const int to_m = wave % RM + ri, to_n = wave / RM + rj;
        uint8_t *const to = area(r, (to_n >= RN ? to_n - RN : to_n) * RM + (to_m >= RM ? to_m - RM : to_m));
#pragma unroll
        for (int j = 0; j < OJ; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const v16f &a = acc[rj * OJ + j][ri];
                *reinterpret_cast<v4f *>(to + (j * 4 + q) * 1024) = v4f{a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
            }
    };
    auto collect = [&](int r) __attribute__((always_inline)) {
        const uint8_t *const from = area(r, wave);
#pragma unroll
        for (int j = 0; j < OJ; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const v4f v = *reinterpret_cast<const v4f *>(from + (j * 4 + q) * 1024);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[j][0][4 * q + e] += v[e];
            }
    };
    using R1 = std::integral_constant<int, 1>;
    using R2 = std::integral_constant<int, 2>;
    using R3 = std::integral_constant<int, 3>;
    send(R1{});
    send(R2{});
    send(R3{});
    __syncthreads();
    collect(1);
    collect(2);
    collect(3);

    // ---- epilogue (as bf6_epilogue in vdmq_bf6.hip): the 32 rows through the wave's own part of an area
    uint8_t *const stg = area(1, wave) - lane * 16;
    lanes_meet();
#pragma unroll
    for (int j = 0; j < OJ; ++j)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
            f16x4 h;
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = static_cast<_Float16>(acc[j][0][rg * 4 + e] * (as * static_cast<float>(w4[j][rg][e])));
            *reinterpret_cast<f16x4 *>(stg + l32 * Cfg::kStageRow + (j * 32 + rg * 8 + lh * 4) * 2) = h;
        }
    lanes_meet();
    // (the wave's corner of the output is a buffer that ends with the last row below M; its columns lie in one part of a split output)
    const int part = tail.split_cols != 0 ? n0 / tail.split_cols : 0, ldo = static_cast<int>(args.ldo);
    const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(
        args.out + part * tail.part_stride + static_cast<int64_t>(m0) * args.ldo + (n0 - part * tail.split_cols), 0, max(min(rows, 32), 0) * ldo * 2, 0x00020000);
#pragma unroll
    for (int it = 0; it < kTurns; ++it) {
        const int row = it * (64 / P) + srow;
        f16x8 hv = *reinterpret_cast<const f16x8 *>(stg + row * Cfg::kStageRow + piece * 2) + bv;
        if (TAIL && tail.gate != nullptr) hv *= gv[it];
        if (TAIL && tail.residual != nullptr) hv = rv[it] + hv;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, hv), out, (row * ldo + piece) * 2, 0, 0);
    }
#endif
}

template <class Cfg>
int launch_cfg(const KsplitArgs &args, bool has_tail, hipStream_t s) {
    using Kernel = void (*)(const KsplitArgs);
    const Kernel kernels[2] = {gemm_bf6_ksplit_kernel<Cfg, false>, gemm_bf6_ksplit_kernel<Cfg, true>};
    constexpr int kMaxDevices = 64;
    static bool attr_done[kMaxDevices][2] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return fail(VDMQ_ELAUNCH, "no current HIP device");
    if (!attr_done[dev][has_tail]) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernels[has_tail]), hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::kLdsBytes);
        if (e != hipSuccess) return fail(VDMQ_ELAUNCH, "hipFuncSetAttribute: %s", hipGetErrorString(e));
        attr_done[dev][has_tail] = true;
    }
    const int64_t units = static_cast<int64_t>(args.tiles_m) * args.tiles_n;
    const dim3 grid(static_cast<unsigned>(ceil_div(units, kXcds) * kXcds));
    hipLaunchKernelGGL(kernels[has_tail], grid, dim3(kWaves * 64), Cfg::kLdsBytes, s, args);
    const int rc = check_launch("gemm_bf6_ksplit_kernel");
    if (rc == VDMQ_OK) record_gemm_launch({VDMQ_KERNEL_GEMM_BF6_KSPLIT, Cfg::MI * 32, Cfg::NJ * 32, 1, 1, 1, static_cast<int64_t>(grid.x)});
    return rc;
}

}  // namespace

// Tile by the number of workgroups, none where the chip would not hold them all at once, a CU each.  GEMM alone, time here over
// that of 128 x 128 tiles: 64 x 64, 46 shapes of 1 ... 1560 rows, K 640 ... 11712, 0.51 ... 0.83; with more than 256 of them (two on a
// CU) 0.93 ... 1.13.  128 x 64 and 64 x 128, 30 shapes: from K = 3328 on 0.79 ... 0.97, 0.96 ... 1.04 below; with more than 256 1.3 ... 1.8.
static int ksplit_tile(int64_t M, int64_t N, int64_t K) {
    constexpr int kCus = 256;
    if (ceil_div(M, 64) * (N / 64) <= kCus) return 1;
    if (K < 3328) return 0;
    return ceil_div(M, 128) * (N / 64) <= kCus ? 2 : ceil_div(M, 64) * (N / 128) <= kCus ? 3 : 0;
}

bool ksplit_takes(int64_t M, int64_t N, int64_t K, int out_dtype) { return out_dtype == VDMQ_OUT_F16 && ksplit_tile(M, N, K) != 0; }

int launch_gemm_bf6_ksplit(const uint8_t *xblocks, const __half *ascale, const uint8_t *wblocks, const __half *wscale, const __half *bias, void *out, int64_t M,
                           int64_t N, int64_t K, int64_t ldo, const GemmTail &tail, hipStream_t s) {
    KsplitArgs a;
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
    const bool has_tail = tail.gate != nullptr || tail.residual != nullptr;
    const int tile = ksplit_tile(M, N, K), mi = tile == 2 ? 4 : 2, nj = tile == 3 ? 4 : 2;
    a.tiles_m = static_cast<int>(ceil_div(M, 32 * mi));
    a.tiles_n = static_cast<int>(ceil_div(N, 32 * nj));
    // (the order in which the XCDs fetch fewer bytes, see vdmq_resident.hip)
    const int64_t x_bytes = M * K, w_bytes = N * K;
    a.by_column = w_bytes + x_bytes * (a.tiles_n < kXcds ? a.tiles_n : kXcds) < x_bytes + w_bytes * (a.tiles_m < kXcds ? a.tiles_m : kXcds) ? 1 : 0;
    return tile == 1 ? launch_cfg<Ksplit<2, 2>>(a, has_tail, s) : tile == 2 ? launch_cfg<Ksplit<4, 2>>(a, has_tail, s) : launch_cfg<Ksplit<2, 4>>(a, has_tail, s);
}

}  // namespace vdmq
