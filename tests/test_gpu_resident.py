"""The forms of a linear that vdmq_linear_bf6 chooses by size -- one kernel for short rows, K divided among a workgroup's waves for few
tiles, between two groups of them for a tile per CU --: the bits of the quantizer and the tiled GEMM in every form they take, at the
edges of their tiles, strips and K steps,
and what they leave to those two."""
import pytest
import torch

from tests.test_gpu_parity import vk

pytestmark = pytest.mark.gpu

RESIDENT, KSPLIT, PAIR = 4, 5, 6  # VDMQ_KERNEL_* of include/vdmq.h
F16 = torch.float16
TILED = (2, 3)


@pytest.fixture(scope="module")
def weight():
    v, cache = vk(), {}

    def make(N, K):
        if (N, K) not in cache:
            g = torch.Generator(device="cuda").manual_seed(N + K)
            s = 1e-3 + 9e-3 * torch.rand(N, 1, generator=g, device="cuda")
            q = torch.randint(-7, 8, (N, K), generator=g, device="cuda")
            qw, ws, _ = v.pack_weight_with_scale((q * s).half(), s.half().view(-1))
            cache[N, K] = (qw, ws, torch.randn(N, generator=g, device="cuda").half())
        return cache[N, K]

    return make


def rows(M, K, seed=0):
    """Rows of every kind: ordinary, zero, tiny, beyond the clamp at small clip ratios, infinite and NaN."""
    g = torch.Generator(device="cuda").manual_seed(seed + 7 * M + K)
    x = torch.randn(M, K, generator=g, device="cuda").half()
    x[:, ::97] *= 20
    for i, value in enumerate((0.0, 6e-8, 65504.0, float("inf"), float("-inf"), float("nan"))):
        at = 5 * i + 1
        if at < M - 1:
            if value == 0.0:
                x[at] = 0
            else:
                x[at, (i * 331 + 3) % K] = value
                x[at, K - 1 - i] = -1.0
    return x


def tiled(f):
    """``f()`` as quantizer and tiled GEMM."""
    from dsaquant_amd import _lib

    v = vk()
    before = v.matrix_path()
    try:
        v.set_matrix_path("bf6")
        want = f()
        assert _lib.last_gemm_launch().kernel in TILED
        return want
    finally:
        v.set_matrix_path(before)


def both(f, kernel=RESIDENT):
    """``f()`` by the library's choice and as quantizer and tiled GEMM."""
    from dsaquant_amd import _lib

    v = vk()
    before = v.matrix_path()
    try:
        v.set_matrix_path("auto")
        got = f()
        info = _lib.last_gemm_launch()
        assert info.kernel in kernel if isinstance(kernel, tuple) else info.kernel == kernel, info.kernel
    finally:
        v.set_matrix_path(before)
    want = tiled(f)
    # NaN rows: the same positions; everything else bit for bit
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    got, want = (torch.where(torch.isnan(t), torch.zeros_like(t), t) for t in (got, want))
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    return info


# K: an even and an odd number of K steps (128 elements), one and two chunks of 512 with and without a remainder, the limits
@pytest.mark.parametrize("K", [640, 704, 960, 1024, 1088, 1472, 1536])
@pytest.mark.parametrize("M,N,tile", [(1, 128, 32), (33, 4608, 32), (300, 12032, 32), (700, 2944, 32), (2049, 1536, 32), (2500, 4096, 64),
                                      (4097, 4608, 128), (33000, 128, 64)])
def test_plain_linear(weight, M, N, tile, K):
    v = vk()
    qw, ws, b = weight(N, K)
    x = rows(M, K)
    info = both(lambda: v.linear_vdm_w4a4(x, qw, ws, b, 0.95))
    assert info.tile_m == tile, info.tile_m
    both(lambda: v.linear_vdm_w4a4(x, qw, ws, None, 1e-3 if M % 2 else 1.0))


@pytest.mark.parametrize("value", [0.0, 65504.0, float("inf"), float("nan")])
@pytest.mark.parametrize("M,N,K", [(33, 4608, 1536), (2500, 4096, 1024), (4097, 4608, 1088), (200, 512, 4096), (500, 4096, 3328)])
def test_special_rows_at_the_ends_of_tiles(weight, M, N, K, value):
    """The last row, which the kernels read again where a tile has none, and the ones at tile ends."""
    v = vk()
    qw, ws, b = weight(N, K)
    x = rows(M, K, 20)
    for at in {31, 63, 127, M - 2, M - 1} & set(range(M)):
        if value == 0.0:
            x[at] = 0
        else:
            x[at, at % K] = value
    both(lambda: v.linear_vdm_w4a4(x, qw, ws, b, 0.95), (RESIDENT, KSPLIT))


@pytest.mark.parametrize("M,N,K", [(679, 13056, 1472), (720, 10880, 1536)])
def test_left_to_two_kernels_where_they_are_faster(weight, M, N, K):
    from dsaquant_amd import fused_ops as F

    v = vk()
    qw, ws, b = weight(N, K)
    x = rows(M, K)
    both(lambda: v.linear_vdm_w4a4(x, qw, ws, b, 0.95), TILED)
    both(lambda: F.linear_fused(x, qw, ws, b, 0.95, split_cols=64), TILED)
    res = torch.randn(M, N, device="cuda").half()
    both(lambda: F.linear_fused(x, qw, ws, b, 0.95, residual=res), TILED if K == 1536 else RESIDENT)


@pytest.mark.parametrize("K", [640, 1472, 1536])
@pytest.mark.parametrize("M,N", [(1, 128), (257, 1536), (1500, 1536), (4100, 1536)])
def test_gated_residual_and_split(weight, M, N, K):
    from dsaquant_amd import fused_ops as F

    qw, ws, b = weight(N, K)
    x = rows(M, K, 1)
    g = torch.Generator(device="cuda").manual_seed(3)
    res, gate = torch.randn(M, N, generator=g, device="cuda").half(), torch.randn(1, N, generator=g, device="cuda").half()
    both(lambda: F.linear_fused(x, qw, ws, b, 0.95, residual=res, gate=gate))
    both(lambda: F.linear_fused(x, qw, ws, None, 0.95, residual=res))
    both(lambda: F.linear_fused(x, qw, ws, b, 0.95, split_cols=64))
    both(lambda: F.linear_fused(x, qw, ws, b, 0.95, split_cols=N))
    both(lambda: F.linear_fused(x, qw, ws, b, 0.95, gate=gate), kernel=TILED + (KSPLIT,))
    both(lambda: F.linear_fused(x, qw, ws, b, 0.95, act="gelu_tanh"), kernel=TILED + (KSPLIT,))
    if M > 1:
        token_gate = torch.randn(M, N, generator=g, device="cuda").half()
        both(lambda: F.linear_fused(x, qw, ws, b, 0.95, residual=res, gate=token_gate), kernel=TILED + (KSPLIT,))


# every instantiation the library chooses: 32, 64 and 128 rows to a workgroup, one and two or three chunks of 512, an odd and an even number
# of K steps each, with the residual and without; a ragged last tile
@pytest.mark.parametrize("K", [640, 960, 1088, 1472])
@pytest.mark.parametrize("M,tile", [(257, 32), (4100, 64), (32700, 128)])
def test_every_tile_with_residual_and_split(weight, M, tile, K):
    from dsaquant_amd import fused_ops as F

    N = 1536
    qw, ws, b = weight(N, K)
    x = rows(M, K, 1)
    g = torch.Generator(device="cuda").manual_seed(3)
    res, gate = torch.randn(M, N, generator=g, device="cuda").half(), torch.randn(1, N, generator=g, device="cuda").half()
    for kw in (dict(), dict(split_cols=N // 3), dict(residual=res), dict(residual=res, gate=gate)):
        info = both(lambda: F.linear_fused(x, qw, ws, b, 0.95, **kw))
        assert info.tile_m == tile, (info.tile_m, kw.keys())


@pytest.mark.parametrize("mode", ["modulate", "affine"])
@pytest.mark.parametrize("B,L,N,K", [(1, 32700, 1536, 640), (2, 16001, 1536, 1088), (1, 32760, 1536, 1536), (1, 31001, 2560, 1472), (2, 16001, 1536, 960), (1, 32700, 1536, 1024)])
def test_layer_norm_in_front(weight, B, L, N, K, mode):
    from dsaquant_amd import fused_ops as F

    qw, ws, b = weight(N, K)
    g = torch.Generator(device="cuda").manual_seed(5)
    x = rows(B * L, K, 2).view(B, L, K)
    vec = (K,) if mode == "affine" else (B, 1, K)
    s, t = ((0.1 * torch.randn(vec, generator=g, device="cuda")).half() for _ in range(2))
    both(lambda: F.linear_ln_vdm_w4a4(F.LnInput(x, s, t, 1e-6, mode), qw, ws, b, 0.95))
    few = x[:, :40].contiguous()
    both(lambda: F.linear_ln_vdm_w4a4(F.LnInput(few, s, t, 1e-6, mode), qw, ws, b, 0.95), kernel=TILED + (KSPLIT,))


def test_strides_workspace_and_refusals_through_the_c_abi(weight):
    """Row strides beyond the row on both sides, no byte written outside the rows; where a workspace is needed and where not."""
    from dsaquant_amd import _lib

    lib, v = _lib.load(), vk()
    M, N, K, ldx, ldo = 129, 384, 1088, 1088 + 72, 384 + 40
    qw, ws, b = weight(N, K)
    pw = v.PreparedWeight([(qw, ws)])
    w = pw.operand(True)
    x = torch.full((M + 1, ldx), float("nan"), device="cuda", dtype=F16)
    x[:M, :K] = rows(M, K, 4).nan_to_num(0.5, 9.0, -9.0)
    out = torch.full((M + 1, ldo), 3.0, device="cuda", dtype=F16)
    s = torch.cuda.current_stream().cuda_stream

    def call(k=K, dtype=0, lx=ldx, lo=ldo, n=N, act=0, workspace=None, nbytes=0):
        return lib.vdmq_linear_bf6(x.data_ptr(), M, k, lx, 0.95, act, w.data_ptr(), pw.wscale.data_ptr(), b.data_ptr(), out.data_ptr(), dtype, n, lo,
                                   workspace, nbytes, s)

    assert lib.vdmq_linear_bf6_workspace(M, N, K, 0, 0, 0, 0, 0) == 0
    _lib.check(call())
    assert _lib.last_gemm_launch().kernel == RESIDENT
    want = tiled(lambda: v.linear_vdm_w4a4(x[:M, :K].contiguous(), qw, ws, b, 0.95))
    assert torch.equal(out[:M, :N], want)
    assert (out[:M, N:] == 3.0).all() and (out[M] == 3.0).all()
    need = lib.vdmq_linear_bf6_workspace(M, N, K, 0, 0, 0, 0, 1)
    assert need == lib.vdmq_workspace_bytes_bf6(M, K) > 0  # bf16: quantizer and GEMM
    assert lib.vdmq_linear_bf6_workspace(M, N, K, 1, 0, 0, 0, 0) == need and lib.vdmq_linear_bf6_workspace(M, N, 1600, 0, 0, 0, 0, 0) > 0
    assert call(dtype=1) == -1 and call(act=1) == -1 and call(act=9) == -1  # no workspace
    for bad in (dict(lx=K - 8), dict(lx=ldx + 4), dict(lo=N - 8), dict(lo=ldo + 4), dict(n=N + 32), dict(k=K + 32), dict(dtype=7)):
        assert call(**bad) < 0, bad


def test_replays_from_a_hip_graph(weight):
    from dsaquant_amd import fused_ops as F

    v = vk()
    N = K = 1536
    qw, ws, b = weight(N, K)
    x = rows(1000, K, 6).nan_to_num(0.5, 9.0, -9.0)
    res = torch.randn(1000, N, device="cuda").half()
    gate = torch.randn(1, N, device="cuda").half()

    def step():
        return F.linear_fused(v.linear_vdm_w4a4(x, qw, ws, b, 0.95), qw, ws, b, 0.95, residual=res, gate=gate)

    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for turn in range(4):
        x.copy_(torch.randn(1000, K, device="cuda").half() * (turn + 1))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, tiled(step))


# K: k-blocks (64 elements, rounded up to an even number) from fewer than the four waves keep in flight to several times as many, each
# remainder; M, N: one row, the edges of 64 x 64, 128 x 64 and 64 x 128 tiles, the last problems of one tile per CU and the first beyond
@pytest.mark.parametrize("M,N,K,tile", [(1, 128, 1600, (64, 64)), (63, 256, 1664, (64, 64)), (65, 384, 1792, (64, 64)), (200, 128, 2048, (64, 64)),
                                        (256, 4096, 2176, (64, 64)), (256, 4096, 13824, (64, 64)), (257, 4096, 4096, (128, 64)),
                                        (500, 4096, 3328, (128, 64)), (385, 4096, 16384, (128, 64)), (289, 6400, 5120, (64, 128)),
                                        (512, 4096, 3264, None), (513, 4096, 4096, None)])
def test_few_tiles(weight, M, N, K, tile):
    from dsaquant_amd import fused_ops as F

    v = vk()
    qw, ws, b = weight(N, K)
    x = rows(M, K, 8)
    kernel = TILED if tile is None else KSPLIT
    info = both(lambda: v.linear_vdm_w4a4(x, qw, ws, b, 0.95), kernel)
    assert tile is None or (info.tile_m, info.tile_n) == tile
    both(lambda: v.linear_vdm_w4a4(x, qw, ws, None, 1e-3), kernel)
    both(lambda: v._linear_2d(x, v._prepared_weight(qw, ws), b, 0.95, out_dtype=torch.bfloat16), TILED)
    g = torch.Generator(device="cuda").manual_seed(11)
    res = torch.randn(M, N, generator=g, device="cuda").half()
    gates = [torch.randn(n, N, generator=g, device="cuda").half() for n in {1, M, 2 if M % 2 == 0 else 1}]
    for gate in gates:
        both(lambda: F.linear_fused(x, qw, ws, b, 0.95, residual=res, gate=gate), kernel)
    both(lambda: F.linear_fused(x, qw, ws, None, 0.95, act="gelu_tanh", gate=gates[0]), kernel)
    both(lambda: F.linear_fused(x, qw, ws, b, 0.95, residual=res), kernel)
    for split in (64, 128, N):
        both(lambda: F.linear_fused(x, qw, ws, b, 0.95, split_cols=split), kernel)


@pytest.mark.parametrize("K", [640, 704, 768, 896, 1024])
def test_few_tiles_short_rows(weight, K):
    """... with fewer k-blocks than twelve or a remainder of each size, where the one-kernel form is not taken."""
    from dsaquant_amd import fused_ops as F

    qw, ws, b = weight(256, K)
    both(lambda: F.linear_fused(rows(100, K, 9), qw, ws, b, 0.95, act="gelu_tanh"), KSPLIT)


# each tile, the last rows and columns of a ragged one, an odd and an even number of 128 k steps with and without a half one, the
# first K each is taken at, and problems next to the rule's lines
@pytest.mark.parametrize("M,N,K,tile", [(1021, 4224, 1984, (128, 160)), (257, 13568, 2112, (128, 160)), (2151, 2432, 3328, (128, 192)),
                                        (11473, 512, 3392, (192, 128)), (4680, 1536, 7424, (192, 160)), (2881, 2944, 2624, (192, 192)),
                                        (5579, 1536, 11072, (192, 192)), (1021, 4224, 1920, None), (1024, 4096, 4096, None), (2880, 2944, 2560, None)])
def test_between_few_tiles_and_many(weight, M, N, K, tile):
    from dsaquant_amd import fused_ops as F

    v = vk()
    qw, ws, b = weight(N, K)
    x = rows(M, K, 21)
    kernel = TILED if tile is None else PAIR
    info = both(lambda: v.linear_vdm_w4a4(x, qw, ws, b, 0.95), kernel)
    assert tile is None or (info.tile_m, info.tile_n) == tile
    both(lambda: F.linear_fused(x, qw, ws, None, 1e-3, split_cols=64), kernel)
    both(lambda: v._linear_2d(x, v._prepared_weight(qw, ws), b, 0.95, out_dtype=torch.bfloat16), TILED)
    if tile is not None:
        g = torch.Generator(device="cuda").manual_seed(11)
        res = torch.randn(M, N, generator=g, device="cuda").half()
        for n in {1, M, 2 if M % 2 == 0 else 1}:
            gate = torch.randn(n, N, generator=g, device="cuda").half()
            both(lambda: F.linear_fused(x, qw, ws, b, 0.95, residual=res, gate=gate), PAIR)
        both(lambda: F.linear_fused(x, qw, ws, b, 0.95, residual=res), PAIR)
        both(lambda: F.linear_fused(x, qw, ws, None, 0.95, act="gelu_tanh", gate=gate), PAIR)


@pytest.mark.parametrize("M,N,K", [(129, 1536, 1536), (2100, 1536, 1472), (200, 512, 4096), (500, 4096, 3328), (1021, 4224, 1984)])
def test_residual_updated_in_place_through_the_c_abi(weight, M, N, K):
    """``out`` is the residual: each element is read by the lane that writes it, before."""
    from dsaquant_amd import _lib, fused_ops as F

    lib, v = _lib.load(), vk()
    qw, ws, b = weight(N, K)
    x = rows(M, K, 12).nan_to_num(0.5, 9.0, -9.0)
    g = torch.Generator(device="cuda").manual_seed(13)
    out, gate = torch.randn(M, N, generator=g, device="cuda").half(), torch.randn(1, N, generator=g, device="cuda").half()
    want = tiled(lambda: F.linear_fused(x, qw, ws, b, 0.95, residual=out, gate=gate))
    pw = v._prepared_weight(qw, ws)
    nbytes = lib.vdmq_linear_bf6_workspace(M, N, K, 0, 0, M, N, 0)
    workspace = torch.empty(max(nbytes, 1), dtype=torch.uint8, device="cuda")
    _lib.check(lib.vdmq_linear_bf6_ex(x.data_ptr(), M, K, K, 0.95, 0, 0, 0.0, None, None, 0, 1, pw.operand(True).data_ptr(), pw.wscale.data_ptr(),
                                      b.data_ptr(), gate.data_ptr(), N, M, out.data_ptr(), N, 0, 0, out.data_ptr(), 0, N, N, workspace.data_ptr(),
                                      nbytes, torch.cuda.current_stream().cuda_stream))
    assert _lib.last_gemm_launch().kernel in (RESIDENT, KSPLIT, PAIR)
    assert torch.equal(out, want)


# resident (32, 64, 128 rows; LayerNorm), K split (64 x 64, 128 x 64)
@pytest.mark.parametrize("M,N,K,kind", [(257, 1536, 1088, "tail"), (4100, 1536, 960, "tail"), (32700, 1536, 1472, "tail"), (200, 512, 4096, "tail"),
                                        (500, 4096, 3328, "tail"), (300, 768, 1536, "split"), (4100, 1536, 1024, "split"), (200, 768, 4096, "split"),
                                        (32700, 1536, 1088, "ln"), (1021, 4224, 1984, "tail"), (1021, 4224, 2112, "split")])
def test_strides_beyond_the_rows_through_the_c_abi(weight, M, N, K, kind):
    """Row strides of input, residual, gate, LayerNorm vectors and output beyond their rows, a part stride beyond the part: the
    bits of the dense call, no byte written outside the rows."""
    from dsaquant_amd import _lib, fused_ops as F

    lib, v = _lib.load(), vk()
    qw, ws, b = weight(N, K)
    g = torch.Generator(device="cuda").manual_seed(17)

    def wide(n, k, pad, fill=7.0):
        t = torch.full((n + 1, k + pad), fill, device="cuda", dtype=F16)
        return t, t[:n, :k]

    xw, x = wide(M, K, 72, float("nan"))
    x.copy_(rows(M, K, 14).nan_to_num(0.5, 9.0, -9.0))
    split, cols = (N // 3, N // 3) if kind == "split" else (0, N)
    parts, part_stride = (3, (M + 2) * (cols + 40)) if split else (1, 0)
    flat = torch.full((parts, M + 2, cols + 40), 3.0, device="cuda", dtype=F16)
    gate_p, ldg, rpg, res_p, ldr, ln = None, 0, 1, None, 0, (0, 0.0, None, None, 0, 1)
    kw = dict(split_cols=split) if split else {}
    if kind == "tail":
        resw, res = wide(M, N, 56)
        res.copy_(torch.randn(M, N, generator=g, device="cuda"))
        gatew, gate = wide(1, N, 24)
        gate.copy_(torch.randn(1, N, generator=g, device="cuda"))
        kw = dict(residual=res.contiguous(), gate=gate.clone().view(-1).view(1, N))
        gate_p, ldg, rpg, res_p, ldr = gatew.data_ptr(), gatew.stride(0), M, resw.data_ptr(), resw.stride(0)
    dense = x.contiguous()
    source = dense
    if kind == "ln":  # one vector for each half of the rows
        (aw, a), (cw, c) = wide(2, K, 48), wide(2, K, 48)
        a.copy_(0.1 * torch.randn(2, K, generator=g, device="cuda"))
        c.copy_(0.1 * torch.randn(2, K, generator=g, device="cuda"))
        source = F.LnInput(dense.view(2, M // 2, K), a.contiguous(), c.contiguous(), 1e-6)
        ln = (_lib.VDMQ_LN_MODULATE, 1e-6, aw.data_ptr(), cw.data_ptr(), aw.stride(0), M // 2)
    want = tiled(lambda: F.linear_fused(source, qw, ws, b, 0.95, **kw)).view(parts, M, cols)
    pw = v._prepared_weight(qw, ws)
    nbytes = lib.vdmq_linear_bf6_workspace(M, N, K, 0, ln[0], rpg if gate_p else 0, ldr, 0)
    workspace = torch.empty(max(nbytes, 1), dtype=torch.uint8, device="cuda")
    _lib.check(lib.vdmq_linear_bf6_ex(xw.data_ptr(), M, K, xw.stride(0), 0.95, 0, *ln, pw.operand(True).data_ptr(), pw.wscale.data_ptr(), b.data_ptr(),
                                      gate_p, ldg, rpg, res_p, ldr, split, part_stride, flat.data_ptr(), 0, N, cols + 40, workspace.data_ptr(), nbytes,
                                      torch.cuda.current_stream().cuda_stream))
    assert _lib.last_gemm_launch().kernel == (PAIR if N == 4224 else KSPLIT if K > 1536 else RESIDENT)
    assert torch.equal(flat[:, :M, :cols].contiguous().view(torch.int16), want.contiguous().view(torch.int16))
    assert (flat[:, :M, cols:] == 3.0).all() and (flat[:, M:] == 3.0).all()
