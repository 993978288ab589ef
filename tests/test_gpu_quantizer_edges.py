"""Edges of the A4 quantizers: every fp16 absmax through the scale arithmetic, rounding ties and the clamp through the
6-bit conversion, and the rows that decide where the fused GELU takes its absmax from."""
import numpy as np
import pytest
import torch

import oracle as O
from tests.test_gpu_parity import gpu_gelu_table, pack_native, rows_of_blocks, special_rows, t16, unpack_native, vk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("clip", [1.0, 0.95, 0.9, 0.3, 1e-5])
def test_scale_and_codes_for_every_fp16_absmax(clip):
    """One row per positive fp16 value, that value its absmax: the scale (absmax / 7 and 1 / scale are each one correction
    step, not a division) and the codes are the oracle's, in both operand forms.  The other elements lie on the fifteen
    rounding ties of the row's grid and next to them (fp16 neighbours), and beyond the clamp for small clip ratios."""
    v = vk()
    K = 64
    amax = np.arange(1, 0x7C00, dtype=np.uint16).view(np.float16)
    step = amax.astype(np.float64) / 7 * clip
    ties = np.arange(-7.5, 8.0)[None, :16] * step[:, None]
    ties = np.clip(ties, -amax.astype(np.float64)[:, None], amax.astype(np.float64)[:, None]).astype(np.float16)
    with np.errstate(over="ignore"):
        up, down = np.nextafter(ties, np.float16(np.inf)), np.nextafter(ties, np.float16(-np.inf))
    x = np.concatenate([ties, up, down, np.zeros_like(ties)], axis=1)
    x = np.where(np.abs(x.astype(np.float32)) > amax.astype(np.float32)[:, None], ties[:, :1] * np.float16(0), x).astype(np.float16)
    x[np.arange(len(amax)), np.arange(len(amax)) % K] = np.where(np.arange(len(amax)) % 2 == 0, amax, -amax)
    want_s = O.np_row_scale(x, clip)
    want_q = O.np_quantize_rows(x, want_s)
    blocks, sc = v.quantize_activation_bf6(t16(x), clip)
    assert np.array_equal(sc.cpu().numpy().view(np.uint16), want_s.view(np.uint16))
    assert np.array_equal(rows_of_blocks(blocks, len(amax), K), want_q.astype(np.float64))
    qn, sc = v.quantize_activation_native(t16(x), clip)
    assert np.array_equal(sc.cpu().numpy().view(np.uint16), want_s.view(np.uint16))
    assert np.array_equal(unpack_native(qn.cpu().numpy(), K), want_q)


def test_gelu_table_has_the_order_the_row_maximum_relies_on():
    """On fp16 values >= 0 the library's GELU does not decrease, and on negative ones its magnitude stays below 0x3180."""
    allh, got = gpu_gelu_table()
    positive = got[:0x7C01].view(np.uint16)
    assert (np.diff(positive.astype(np.int32)) >= 0).all()
    negative = got[0x8000:0xFC00]
    assert np.isfinite(negative).all() and ((negative.view(np.uint16) & 0x7FFF) < 0x3180).all()


@pytest.mark.parametrize("K", [512, 5120, 7168, 7168 + 64, 8192 + 64, 9216, 9216 + 128, 13824, 16384])
@pytest.mark.parametrize("clip", [1.0, 0.5, 1e-6])
def test_gelu_quantizer_row_kinds(K, clip):
    """Rows whose absmax comes from a large positive element, from the negative branch, from a positive element just
    around the negative branch's peak, and rows with NaN / Inf of either sign, on both sides of the row lengths where
    the kernel changes form."""
    v = vk()
    _, table = gpu_gelu_table()
    rng = np.random.default_rng(K)
    x = rng.standard_normal((37, K)).astype(np.float16)
    x[1] = 0
    x[2] = -np.abs(x[2])                       # no positive element: |gelu| <= 0.17
    x[3] = np.minimum(x[3], np.float16(0.05))  # small positive ones: the negative branch decides
    x[4] = np.minimum(x[4], np.float16(0.284))
    x[5] = np.minimum(x[5], np.float16(0.29))
    x[6, 3], x[7, 5], x[8, 7], x[9, 9] = np.inf, -np.inf, np.nan, 65504
    x[10] = np.float16(-65504)
    x[11] = np.float16(6e-8)
    x[12, 1] = np.array(0xFE00, np.uint16).view(np.float16)  # NaN with the sign bit
    x[13] = -np.abs(x[13])
    x[13, K - 1] = -np.inf
    g = table[x.view(np.uint16)]
    want_s = O.np_row_scale(g, clip)
    want_q = O.np_quantize_rows(g, want_s)
    blocks, sc = v.quantize_activation_bf6(t16(x), clip, act="gelu_tanh")
    assert np.array_equal(sc.cpu().numpy().view(np.uint16), want_s.view(np.uint16))
    assert np.array_equal(rows_of_blocks(blocks, len(x), K), want_q.astype(np.float64))


def codes_of_blocks(blocks, rows, K):
    """The six-bit codes of a bf6 operand, strings in memory order, minus zero as zero (the quantizers keep the sign of what
    they round to zero, the conversion from native rows has none)."""
    panels = blocks.view(rows // 8, -1, 384)
    a, b = panels[..., :256].unflatten(2, (2, 8, 16)), panels[..., 256:].unflatten(2, (2, 8, 8))
    w = torch.cat([a, b], dim=-1).unflatten(-1, (8, 3)).int()
    w = w[..., 0] | w[..., 1] << 8 | w[..., 2] << 16
    codes = torch.stack([w >> 6 * i & 63 for i in range(4)], dim=-1).to(torch.uint8)
    return torch.where(codes == 32, 0, codes)


def by_row(blocks, rows):
    """The two planes of a bf6 operand's first rows, [row, k-block, half, byte] each."""
    panels = blocks.view(-(-rows // 32) * 4, -1, 384)
    planes = [panels[..., :256].unflatten(2, (2, 8, 16)), panels[..., 256:].unflatten(2, (2, 8, 8))]
    return [p.movedim(3, 1).flatten(0, 1)[:rows] for p in planes]


@pytest.mark.parametrize("M,K,producer", [(5121, 1536, None), (5121, 3584, None), (5123, 3648, None), (12999, 13824, None), (20001, 9216, None),
                                          (3073, 6208, None), (4096, 13824, None), (5633, 5184, None), (7041, 8960, None), (7681, 8960, None), (8192, 10304, None), (8705, 10304, None),
                                          (5121, 1536, "gelu_tanh"), (20001, 9216, "gelu_tanh"), (20001, 9280, "gelu_tanh"), (40005, 8960, "gelu_tanh")])
def test_whole_and_half_panel_workgroups(M, K, producer):
    """A workgroup takes a panel of eight rows or half of one, by the number of rows, their length, the producer in front and the
    size of the output: on both sides of those lines the rows' codes and scales are those of the same rows in slices of 2048, which
    workgroups of four or fewer rows serve (and which the other tests compare with the oracle)."""
    v = vk()
    g = torch.Generator("cuda").manual_seed(M)
    x = torch.randn(M, K, generator=g, device="cuda").half()
    blocks, scales = v.quantize_activation_bf6(x, 0.95, act=producer)
    whole = by_row(blocks, M)
    for r in range(0, M, 2048):
        rows = x[r:r + 2048]
        part, part_scales = v.quantize_activation_bf6(rows, 0.95, act=producer)
        assert torch.equal(scales[r:r + 2048], part_scales)
        assert all(torch.equal(w[r:r + 2048], p) for w, p in zip(whole, by_row(part, len(rows))))


@pytest.mark.parametrize("mode", ["modulate", "affine"])
@pytest.mark.parametrize("M,K", [(517, 64), (517, 1536), (517, 1600), (517, 3072), (517, 5120), (517, 8960), (517, 13824), (517, 16384), (2347, 1536),
                                 (2347, 8960), (35005, 5120)])
def test_layer_norm_with_two_and_four_rows_per_workgroup(M, K, mode):
    """Behind a LayerNorm up to 512 rows go by twos and more by fours (the last group of either not full): the first and the last rows
    of a call have the codes and scales that they have in calls of their own, of either kind."""
    from dsaquant_amd import fused_ops

    g = torch.Generator("cuda").manual_seed(K)
    x = torch.randn(M, K, generator=g, device="cuda").half()
    x[3::41] = 0
    x[5, K - 1], x[8, 3], x[511, 0] = float("inf"), float("nan"), 65504
    vectors = [0.1 * torch.randn(M, K, generator=g, device="cuda").half() for _ in range(2)]

    def quantize(rows):
        return fused_ops.LnInput(x[rows], *(t[rows] for t in vectors), 1e-6, mode).quantize(0.95, bf6=True)

    blocks, scales = quantize(slice(M))
    by_fours = by_row(blocks, M)
    for n in (1, 2, 13, 511, 512, 513):
        for rows in (slice(n), slice(M - n, M)):
            part, part_scales = quantize(rows)
            assert torch.equal(scales[rows].view(torch.int16), part_scales.view(torch.int16))
            assert all(torch.equal(w[rows], p) for w, p in zip(by_fours, by_row(part, n)))


@pytest.mark.parametrize("act", [None, "gelu_tanh"])
@pytest.mark.parametrize("K", [1600, 2560, 2624, 4096, 4160, 6208, 7168, 8256, 9216, 12288, 13824, 14400, 16384])
def test_rows_shared_by_four_waves(K, act):
    """Few rows go to four waves each: the codes and scales are those of the same rows among many, which have a wave each, with rows of
    every kind (the largest element and NaN or Inf in any part, zeros, the GELU's negative branch) and numbers of rows around the line."""
    v = vk()
    g = torch.Generator("cuda").manual_seed(K)
    x = torch.randn(1600, K, generator=g, device="cuda").half()
    x[torch.arange(1600), torch.arange(1600) * 131 % K] *= 20
    x[1::11] = -x[1::11].abs()
    x[2::97] = 0
    x[3::101, K - 1], x[5::103, K // 2], x[7::107, 3], x[8::109, K // 4] = float("inf"), float("nan"), float("-inf"), 65504
    many, many_scales = v.quantize_activation_bf6(x, 0.95, act=act)
    want = by_row(many, 1600)
    for rows in (1, 2, 31, 513, 1536) if K > 2560 else (1, 2, 31, 511, 512):
        blocks, scales = v.quantize_activation_bf6(x[:rows], 0.95, act=act)
        assert torch.equal(scales.view(torch.int16), many_scales[:rows].view(torch.int16))
        assert all(torch.equal(w[:rows], p) for w, p in zip(want, by_row(blocks, rows)))


@pytest.mark.parametrize("act", [None, "gelu_tanh"])
@pytest.mark.parametrize("M,K", [(25600, 1536), (17408, 2048), (4320, 9216 + 64), (4320, 13824), (4320, 16384)])
def test_walking_quantizers_over_several_rounds(M, K, act):
    """Row lengths whose workgroups walk row groups, with more than two groups each: rows of every kind -- the GELU's absmax
    from the largest element, from the negative branch, NaN, Inf, zeros -- follow one another in a workgroup's sequence,
    every row against the oracle's integers (brought into blocks by the conversion from native rows)."""
    v = vk()
    _, table = gpu_gelu_table()
    rng = np.random.default_rng(M + K)
    kinds = rng.standard_normal((61, K)).astype(np.float16)
    kinds[1::7] = -np.abs(kinds[1::7])                          # the negative branch decides
    kinds[2::7] = np.minimum(kinds[2::7], np.float16(0.284))
    kinds[3], kinds[17] = 0, np.float16(6e-8)
    kinds[4, 3], kinds[18, K - 1], kinds[32, 7], kinds[46, 9] = np.inf, -np.inf, np.nan, 65504
    kinds[5::7, :: K // 9] *= np.float16(20)
    x = kinds if act is None else table[kinds.view(np.uint16)]
    scale = O.np_row_scale(x, 0.95)
    native = t16(pack_native(O.np_quantize_rows(x, scale), v.k_padded(K)))
    row = torch.arange(M, device="cuda") * 23 % 61
    blocks, sc = v.quantize_activation_bf6(t16(kinds)[row], 0.95, act=act)
    assert torch.equal(sc.view(torch.int16), t16(scale)[row].view(torch.int16))
    assert torch.equal(codes_of_blocks(blocks, M, K), codes_of_blocks(v.bf6_blocks(native[row], K), M, K))


@pytest.mark.parametrize("N,K", [(128, 64), (256, 1088), (128, 5120 + 64), (128, 16384 + 64)])
def test_row_scale_and_given_scale_entry_points(N, K):
    """vdmq_row_scale and vdmq_quantize_weight_native of the C interface, rows with NaN / Inf / zeros, given scales of zero,
    Inf and NaN among ordinary ones."""
    from dsaquant_amd import _lib

    lib, v = _lib.load(), vk()
    rng = np.random.default_rng(N + K)
    w = special_rows((0.05 * rng.standard_normal((N, K))).astype(np.float16))
    wt, s = t16(w), torch.cuda.current_stream().cuda_stream
    for clip in (1.0, 0.95, 1e-5):
        scale = torch.empty(N, dtype=torch.float16, device="cuda")
        _lib.check(lib.vdmq_row_scale(wt.data_ptr(), N, K, clip, scale.data_ptr(), s))
        want = O.np_row_scale(w, clip)
        assert np.array_equal(scale.cpu().numpy().view(np.uint16), want.view(np.uint16))
    given = np.where(want == 1, want, O.np_row_scale(w, 0.75)).astype(np.float16)
    given[20:25] = np.array([0.0, -1e-3, np.inf, 6e-8, np.nan], np.float16)
    native = torch.empty((N, v.k_padded(K) // 2), dtype=torch.uint8, device="cuda")
    _lib.check(lib.vdmq_quantize_weight_native(wt.data_ptr(), t16(given).data_ptr(), native.data_ptr(), N, K, s))
    assert np.array_equal(unpack_native(native.cpu().numpy(), K), O.np_quantize_rows(w, given))


def _round_fma(a, b, c):
    """fl32(a * b + c) of float32 arrays: the sum in double, its last bit made odd where the addition was inexact, so that
    the second rounding cannot tie."""
    p, c = a.astype(np.float64) * b.astype(np.float64), c.astype(np.float64)
    s = p + c
    t = s - p
    err = (p - (s - t)) + (c - t)
    even = (s.view(np.int64) & 1) == 0
    return np.where((err != 0) & even, np.nextafter(s, np.where(err > 0, np.inf, -np.inf)), s).astype(np.float32)


def _wave_sum(lanes):
    for distance in (32, 16, 8, 4, 2, 1):
        lanes = lanes + lanes[:, np.arange(64) ^ distance]
    assert (lanes == lanes[:, :1]).all()
    return lanes[:, 0]


def layer_norm_as_defined(x, a, b, eps, mode):
    """The fused LayerNorm's fp32 arithmetic, operation by operation: lane l of a row holds elements 512 c + 8 l ... + 7 and
    adds them in that order, lanes are added at distances 32, 16, 8, 4, 2, 1, every division and square root is rounded
    correctly."""
    M, K = x.shape
    xf = x.astype(np.float32)
    total, sq = np.zeros((M, 64), np.float32), np.zeros((M, 64), np.float32)
    places = [(np.arange(64) * 8 + 512 * c + e) for c in range((K + 511) // 512) for e in range(8)]
    for k in places:
        total[:, k < K] += xf[:, k[k < K]]
    mean = _wave_sum(total) / np.float32(K)
    d = xf - mean[:, None]
    for k in places:
        sq[:, k < K] = _round_fma(d[:, k[k < K]], d[:, k[k < K]], sq[:, k < K])
    rstd = np.float32(1) / np.sqrt(_wave_sum(sq) / np.float32(K) + np.float32(eps))
    n = d * rstd[:, None]
    if mode == "affine":
        return (n * a.astype(np.float32) + b.astype(np.float32)).astype(np.float16)
    return n.astype(np.float16) * (np.float16(1) + a) + b


@pytest.mark.parametrize("mode", ["modulate", "affine"])
@pytest.mark.parametrize("K", [64, 192, 512, 1088, 1536, 2048, 3072, 5120, 8192 + 64, 13824])
def test_layer_norm_sums_in_its_defined_order(K, mode):
    """Bit for bit, rows with and without a mean: a sum in another order moves the last bits, and int4 codes with them."""
    from dsaquant_amd import fused_ops

    rng = np.random.default_rng(K)
    x = (rng.standard_normal((300, K)) * 3 + rng.standard_normal((300, 1))).astype(np.float16)
    x[:, rng.permutation(K)[: max(1, K // 100)]] *= np.float16(20)
    a, b = ((0.1 * rng.standard_normal((1, K))).astype(np.float16) for _ in range(2))
    want = layer_norm_as_defined(x, a, b, 1e-6, mode)
    pre = fused_ops.LnInput(t16(x), t16(a), t16(b), 1e-6, mode)
    assert np.array_equal(pre.materialize().cpu().numpy().view(np.uint16), want.view(np.uint16))
    want_s = O.np_row_scale(want, 0.95)
    want_q = O.np_quantize_rows(want, want_s)
    blocks, sc = pre.quantize(0.95, bf6=True)
    assert np.array_equal(sc.cpu().numpy().view(np.uint16), want_s.view(np.uint16))
    assert np.array_equal(rows_of_blocks(blocks, len(x), K), want_q.astype(np.float64))


@pytest.mark.parametrize("N,K", [(128, 64), (128, 1088), (1152, 448), (640, 2112), (256, 5120 + 64), (128, 9216), (128, 9216 + 64), (1024 + 128, 13824),
                                 (128, 1536), (128, 1600), (128, 4096), (128, 4160), (128, 7168), (128, 7232), (128, 12288), (128, 12352),
                                 (128, 14336), (128, 14400), (2048, 16384), (128, 16448)])
def test_pack_weight_edges(N, K):
    """One-pass weight packing: row tiles beyond and within a full group of eight 128-row blocks, rows on both sides of
    every register form and the two-pass one, rows with NaN / Inf, zero rows and scales of zero, negative and Inf; the
    int8 path's form, made in the same pass for short rows, holds the same integers."""
    v = vk()
    rng = np.random.default_rng(N + K)
    w = special_rows((0.05 * rng.standard_normal((N, K))).astype(np.float16))
    q, ps, s = v.quantize_weight_per_channel(t16(w))
    want_s = O.np_row_scale(w, 1.0)
    want_q = O.np_quantize_rows(w, want_s)
    assert np.array_equal(s.cpu().numpy().view(np.uint16), want_s.view(np.uint16))
    assert np.array_equal(q.cpu().numpy(), O.np_pack_wgt_v1(want_q))
    assert np.array_equal(ps.cpu().numpy().view(np.uint16), O.np_pack_wscales_v1(want_s, K).view(np.uint16))
    if K < 1280:
        assert np.array_equal(unpack_native(v._native_weights(q, ps)[0].cpu().numpy(), K), want_q)
    scale = np.where(want_s == 1, want_s, want_s * np.float16(0.75)).astype(np.float16)
    scale[20:24] = np.array([0.0, -1e-3, np.inf, 6e-8], np.float16)
    q, ps, s = v.pack_weight_with_scale(t16(w), t16(scale))
    assert np.array_equal(q.cpu().numpy(), O.np_pack_wgt_v1(O.np_quantize_rows(w, scale)))
    assert np.array_equal(ps.cpu().numpy().view(np.uint16), O.np_pack_wscales_v1(scale, K).view(np.uint16))
