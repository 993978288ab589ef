"""The one-kernel form of the linear for short rows (vdmq_linear_bf6): the bits of the quantizer and the tiled GEMM in every
form it takes, at the edges of its row tiles, column strips and K steps, and the forms it leaves to those two."""
import pytest
import torch

from tests.test_gpu_parity import vk

pytestmark = pytest.mark.gpu

RESIDENT = 4  # VDMQ_KERNEL_LINEAR_RESIDENT of include/vdmq.h
F16 = torch.float16


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
    """Rows of every kind: ordinary, zero, tiny, beyond the clamp at small clip ratios, infinite and NaN; none of the special ones
    comes last, since the kernel reads that one again where it has no row."""
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


def both(f, resident=True):
    """``f()`` by the library's choice and as quantizer and tiled GEMM."""
    from dsaquant_amd import _lib

    v = vk()
    before = v.matrix_path()
    try:
        v.set_matrix_path("auto")
        got = f()
        info = _lib.last_gemm_launch()
        assert (info.kernel == RESIDENT) == resident, info.kernel
        v.set_matrix_path("bf6")
        want = f()
        assert _lib.last_gemm_launch().kernel != RESIDENT
    finally:
        v.set_matrix_path(before)
    # NaN rows: the same positions; everything else bit for bit
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.nan_to_num(got).view(torch.int16), torch.nan_to_num(want).view(torch.int16))
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
    both(lambda: F.linear_fused(x, qw, ws, b, 0.95, gate=gate), resident=False)
    both(lambda: F.linear_fused(x, qw, ws, b, 0.95, act="gelu_tanh"), resident=False)
    if M > 1:
        token_gate = torch.randn(M, N, generator=g, device="cuda").half()
        both(lambda: F.linear_fused(x, qw, ws, b, 0.95, residual=res, gate=token_gate), resident=False)


@pytest.mark.parametrize("mode", ["modulate", "affine"])
@pytest.mark.parametrize("B,L,N,K", [(1, 32760, 1536, 1536), (1, 31001, 2560, 1472), (2, 16001, 1536, 960), (1, 32700, 1536, 1024)])
def test_layer_norm_in_front(weight, B, L, N, K, mode):
    from dsaquant_amd import fused_ops as F

    qw, ws, b = weight(N, K)
    g = torch.Generator(device="cuda").manual_seed(5)
    x = rows(B * L, K, 2).view(B, L, K)
    vec = (K,) if mode == "affine" else (B, 1, K)
    s, t = ((0.1 * torch.randn(vec, generator=g, device="cuda")).half() for _ in range(2))
    both(lambda: F.linear_ln_vdm_w4a4(F.LnInput(x, s, t, 1e-6, mode), qw, ws, b, 0.95))
    few = x[:, :40].contiguous()
    both(lambda: F.linear_ln_vdm_w4a4(F.LnInput(few, s, t, 1e-6, mode), qw, ws, b, 0.95), resident=False)


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
    want = v.linear_vdm_w4a4(x[:M, :K].contiguous(), qw, ws, b, 0.95)
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
        assert torch.equal(out, step())
