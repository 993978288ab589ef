"""Calls served whole by the extension module (vdmq_host.cpp): results and errors are the general code's, and operands that are not
plain are left to it."""
import pytest
import torch

from tests.test_gpu_parity import vk

pytestmark = pytest.mark.gpu

N, K = 384, 704


@pytest.fixture(scope="module")
def operands():
    g = torch.Generator(device="cuda").manual_seed(3)
    s = (1e-3 + 9e-3 * torch.rand(N, generator=g, device="cuda")).half()
    w = (torch.randint(-7, 8, (N, K), generator=g, device="cuda") * s.view(-1, 1)).half()
    qw, ws, _ = vk().pack_weight_with_scale(w, s)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device="cuda").half()  # noqa: E731
    return dict(w=w, s=s, qw=qw, ws=ws, b=rnd(N), x=rnd(2, 33, K), res=rnd(2, 33, N), gate=rnd(2, 1, N), a=rnd(2, 1, K), shift=rnd(2, 1, K))


class Spy:
    """The extension module, counting what it served; ``off``: serving nothing."""

    def __init__(self, host, off):
        self.host, self.off, self.served = host, off, 0

    def __getattr__(self, name):
        def call(*args):
            out = None if self.off else getattr(self.host, name)(*args)
            self.served += out is not None
            return out

        return call


def outcome(f, off):
    from dsaquant_amd import _lib

    host = _lib.load() and _lib.host
    _lib.host = spy = Spy(host, off)
    try:
        out = f()
        out = out if isinstance(out, (tuple, list)) else (out,)
        return [(t.shape, t.stride(), t.dtype, t.device, t.requires_grad, t.clone()) for t in out], spy.served
    except Exception as e:
        return (type(e), str(e)), spy.served
    finally:
        _lib.host = host


def same(f, served):
    (got, n), (want, _) = outcome(f, False), outcome(f, True)
    assert (n > 0) == served
    assert len(got) == len(want)
    if isinstance(want, tuple):
        assert got == want
    else:
        for g, w in zip(got, want):
            assert g[:-1] == w[:-1] and torch.equal(g[-1].view(torch.uint8), w[-1].view(torch.uint8))
    return want


def test_served_calls(operands):
    from dsaquant_amd import fused_ops as F

    v, o = vk(), operands
    x, qw, ws, b = o["x"], o["qw"], o["ws"], o["b"]
    pw = v._prepared_weight(qw, ws)
    parts = [t for pair in zip(qw.chunk(3), ws.chunk(3)) for t in pair]
    same(lambda: v.linear_vdm_w4a4(x, qw, ws, b, 0.95), True)
    same(lambda: v.linear_vdm_w4a4(x[0, 0], qw, ws, None, 1), True)
    same(lambda: v.linear_vdm_w4a4(x, qw, ws, b.float(), 0.95, bias_half=b), True)
    same(lambda: v.linear_vdm_w4a4_qkv(x, *parts, clip_ratio=0.95, w_qkv_packed=qw, w_qkv_scale=ws, qkv_bias_half=b), True)
    same(lambda: v.linear_vdm_w4a4_qkv(x, *parts, clip_ratio=0.95, w_qkv_packed=qw, w_qkv_scale=ws, contiguous_outputs=True), True)
    same(lambda: v.linear_vdm_w4a4_prepared(x, pw, b, 0.95), True)
    same(lambda: v.linear_vdm_w4a4_prepared(x, pw, b, 0.95, split_cols=128), True)
    same(lambda: F.linear_fused(x, qw, ws, b, 0.95, residual=o["res"], gate=o["gate"]), True)
    same(lambda: F.linear_fused(x, qw, ws, b, 0.95, act="gelu_tanh", gate=o["gate"][:1]), True)
    same(lambda: F.linear_fused(x, pw, None, None, 0.95, residual=o["res"]), True)
    for a, s in ((o["a"], o["shift"]), (o["a"][0, 0], o["shift"][0, 0])):
        same(lambda: F.linear_ln_vdm_w4a4(F.LnInput(x, a, s, 1e-6), qw, ws, b, 0.95), True)
    same(lambda: F.linear_fused(F.LnInput(x.float(), o["a"], o["shift"], 1e-6, "affine"), qw, ws, b, 0.95, residual=o["res"]), True)
    pre = F.LnInput(x, o["a"], o["a"], 1e-6)
    pre.b = o["shift"].view(2, K)
    same(lambda: F.linear_ln_vdm_w4a4(pre, qw, ws, b, 0.95), True)
    assert torch.equal(F.linear_ln_vdm_w4a4(pre, qw, ws, b, 0.95), F.linear_ln_vdm_w4a4(F.LnInput(x, o["a"], o["shift"], 1e-6), qw, ws, b, 0.95))
    same(lambda: v.quantize_weight_per_channel(o["w"]), True)
    same(lambda: v.pack_weight_with_scale(o["w"], o["s"].view(-1, 1)), True)
    with torch.inference_mode():
        same(lambda: v.linear_vdm_w4a4(x, qw, ws, b, 0.95), True)
    with torch.enable_grad():
        same(lambda: v.linear_vdm_w4a4(torch.nn.Parameter(x), qw, ws, b, 0.95), True)


def test_calls_left_to_the_general_code(operands):
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from dsaquant_amd import fused_ops as F

    v, o = vk(), operands
    x, qw, ws, b = o["x"], o["qw"], o["ws"], o["b"]

    class Sub(torch.Tensor):
        pass

    same(lambda: v.linear_vdm_w4a4(x.float(), qw, ws, b, 0.95), False)
    same(lambda: v.linear_vdm_w4a4(x.transpose(0, 1), qw, ws, b, 0.95), False)
    same(lambda: v.linear_vdm_w4a4(x[:, :0], qw, ws, b, 0.95), False)
    same(lambda: v.linear_vdm_w4a4(x, qw, ws, b.float(), 0.95), False)
    same(lambda: v.linear_vdm_w4a4(x.as_subclass(Sub), qw, ws, b, 0.95).as_subclass(torch.Tensor), False)
    same(lambda: v.linear_vdm_w4a4(x, qw.t().contiguous().t(), ws, b, 0.95), False)
    same(lambda: F.linear_fused(x, qw, ws, b, 0.95, residual=o["res"].transpose(0, 1).contiguous().transpose(0, 1)), False)
    same(lambda: v.quantize_weight_per_channel(o["w"].float()), False)
    same(lambda: v.quantize_weight_per_channel(o["w"][:, :512]), False)
    for bad in (lambda: v.linear_vdm_w4a4(x.cpu(), qw, ws, b, 0.95), lambda: v.linear_vdm_w4a4(x[..., :640], qw, ws, b, 0.95),
                lambda: v.linear_vdm_w4a4(x, qw, ws, b[:128], 0.95), lambda: v.linear_vdm_w4a4(x, qw, ws[:, 1:], b, 0.95),
                lambda: F.linear_fused(x, qw, ws, b, 0.95, residual=o["res"][:1]), lambda: F.linear_fused(x, qw, ws, b, 0.95, gate=o["gate"][..., :128]),
                lambda: F.linear_fused(x[:, :32], qw, ws, b, 0.95, gate=o["res"][0, :3]), lambda: F.linear_fused(x, qw, ws, b, 0.95, split_cols=96),
                lambda: F.linear_fused(x, qw, ws, b, 0.95, split_cols=0), lambda: v.linear_vdm_w4a4(x, qw, ws, b, "much"),
                lambda: F.LnInput(x, o["a"], o["shift"][:1], 1e-6), lambda: F.LnInput(x, o["a"][..., :64], o["shift"][..., :64], 1e-6),
                lambda: torch.func.vmap(lambda t: v.linear_vdm_w4a4(t, qw, ws, b, 0.95))(x)):
        assert isinstance(same(bad, False), tuple)
    pw = v._prepared_weight(qw, ws)  # the packed entries take packed weights only, with their scales
    for refused in (lambda: v.linear_vdm_w4a4(x, pw, None, b, 0.95), lambda: v.linear_vdm_w4a4(x, qw, None, b, 0.95),
                    lambda: F.linear_fused(x, qw, None, b, 0.95), lambda: v.linear_vdm_w4a4(x, pw, ws, b, 0.95)):
        assert same(refused, False)[0] is AttributeError
    for path in ("int8", "bf6"):
        before = v.matrix_path()
        try:
            v.set_matrix_path(path)
            same(lambda: v.linear_vdm_w4a4(x, qw, ws, b, 0.95), False)
        finally:
            v.set_matrix_path(before)
    for mode in (TorchFunctionMode, TorchDispatchMode):

        class Seen(mode):
            calls = 0

            def __torch_function__(self, func, types, args=(), kwargs=None):
                Seen.calls += 1
                return func(*args, **(kwargs or {}))

            def __torch_dispatch__(self, func, types, args=(), kwargs=None):
                Seen.calls += 1
                return func(*args, **(kwargs or {}))

        with Seen():
            same(lambda: v.linear_vdm_w4a4(x, qw, ws, b, 0.95), False)
        assert Seen.calls > 0


@pytest.mark.parametrize("other", [K - 64, K + 64])
def test_rows_of_another_length_than_a_prepared_weights(operands, other):
    """Shorter rows would multiply by the wrong weights, longer ones read behind the last: refused, with the general code's error,
    before the weight's form is asked for."""
    from types import SimpleNamespace

    from dsaquant_amd import fused_ops as F
    from dsaquant_amd.fused_qkv import get_qkv_projections

    v, o = vk(), operands
    qw, ws = o["qw"].clone(), o["ws"].clone()
    x, a = torch.ones((2, 33, other), device="cuda").half(), torch.ones((2, 1, other), device="cuda").half()
    pw = v._prepared_weight(qw, ws)
    for call in (lambda: v.linear_vdm_w4a4_prepared(x, pw, o["b"], 0.95), lambda: v.linear_vdm_w4a4_prepared(x, pw, o["b"], 0.95, split_cols=128),
                 lambda: F.linear_fused(x, pw, None, o["b"], 0.95), lambda: F.linear_fused(x, pw, None, o["b"], 0.95, act="gelu_tanh"),
                 lambda: F.linear_fused(x, pw, None, o["b"], 0.95, residual=o["res"], gate=o["gate"]), lambda: F.linear_fused(x, pw, None, split_cols=128),
                 lambda: F.linear_fused(F.LnInput(x, a, a, 1e-6), pw, None, o["b"], 0.95),
                 lambda: F.linear_fused(F.LnInput(x.float(), a, a, 1e-6, "affine"), pw, None, o["b"], 0.95)):
        assert same(call, False) == (ValueError, "qweight shape must be [N, K/2]")
    assert pw.bf6 is None
    layer = lambda: SimpleNamespace(vdm_weight_packed=qw.clone(), vdm_weight_scale_packed=ws.clone(), _bias_half=None, kernel_clip_ratio=0.95)  # noqa: E731
    for contiguous in (False, True):
        for cross in (None, 128):
            attn = SimpleNamespace(to_q=lambda t: t, to_k=layer(), to_v=layer(), cross_attention_dim_head=cross, use_fused_qkv_kernel=True,
                                   qkv_kernel_backend="vdm", qkv_contiguous_outputs=contiguous)
            if cross is None:
                attn.to_q = layer()
                calls = [lambda: get_qkv_projections(attn, x, None), lambda: F.qkv_projections_ln(attn, F.LnInput(x, a, a, 1e-6))]
            else:
                calls = [lambda: get_qkv_projections(attn, x, x), lambda: F.kv_projections(attn, x)]
            for call in calls:
                assert same(call, False) == (ValueError, "qweight shape must be [N, K/2]")
    # a cached concatenation of another row length than the projections it is said to be of
    g = torch.Generator(device="cuda").manual_seed(5)
    part = v.pack_weight_with_scale(torch.randn((128, other), generator=g, device="cuda").half(), torch.ones(128, device="cuda").half())[:2]
    for contiguous in (False, True):
        assert same(lambda: v.linear_vdm_w4a4_qkv(x, *part, *part, *part, clip_ratio=0.95, w_qkv_packed=qw, w_qkv_scale=ws, contiguous_outputs=contiguous),
                    False) == (ValueError, "qweight shape must be [N, K/2]")


def test_refused_calls_leave_a_prepared_weight_as_it_was(operands):
    """A call that is refused for another operand has made no form of the weight and dropped none that was made ahead."""
    from dsaquant_amd import fused_ops as F

    v, o = vk(), operands
    x, b = o["x"], o["b"]
    qw, ws = o["qw"].clone(), o["ws"].clone()
    pw = v._prepared_weight(qw, ws)
    native = pw.operand(False, eager=True)
    for refused in (lambda: v.linear_vdm_w4a4_prepared(x, pw, b[:128], 0.95), lambda: v.linear_vdm_w4a4_prepared(x, pw, b, 0.95, split_cols=96),
                    lambda: F.linear_fused(x, pw, None, b, 0.95, gate=o["gate"][..., :128]), lambda: F.linear_fused(x[:, :32], pw, None, b, 0.95, gate=o["res"][0, :3]),
                    lambda: F.linear_fused(x, pw, None, b, 0.95, residual=o["res"][:1]), lambda: F.linear_fused(x, pw, None, b[:128], 0.95),
                    lambda: F.linear_fused(x, pw, None, b, 0.95, gate=o["gate"], split_cols=128), lambda: v.linear_vdm_w4a4(x, qw, ws, b[:128], 0.95),
                    lambda: v.linear_vdm_w4a4(x, qw, ws, b, "much")):
        assert isinstance(same(refused, False), tuple)
        assert pw.native is native and pw.bf6 is None
    same(lambda: v.linear_vdm_w4a4_prepared(x, pw, b, 0.95), True)
    assert pw.native is None and pw.bf6 is not None


def test_calls_without_the_extension_module(operands, monkeypatch):
    from dsaquant_amd import _lib, fused_ops as F

    v, o = vk(), operands
    x, qw, ws, b = o["x"], o["qw"], o["ws"], o["b"]
    parts = [t for pair in zip(qw.chunk(3), ws.chunk(3)) for t in pair]
    calls = (lambda: v.linear_vdm_w4a4(x, qw, ws, b, 0.95), lambda: v.linear_vdm_w4a4_prepared(x, v._prepared_weight(qw, ws), b, 0.95, split_cols=128),
             lambda: torch.cat(v.linear_vdm_w4a4_qkv(x, *parts, clip_ratio=0.95, w_qkv_packed=qw, w_qkv_scale=ws, qkv_bias_half=b)),
             lambda: F.linear_fused(x, qw, ws, b, 0.95, act="gelu_tanh", residual=o["res"], gate=o["gate"]),
             lambda: F.linear_ln_vdm_w4a4(F.LnInput(x, o["a"], o["shift"], 1e-6), qw, ws, b, 0.95),
             lambda: v.quantize_weight_per_channel(o["w"])[0], lambda: v.pack_weight_with_scale(o["w"], o["s"])[1])
    want = [c() for c in calls]
    monkeypatch.setattr(_lib, "host", None)
    for c, w in zip(calls, want):
        assert torch.equal(c().view(torch.uint8), w.view(torch.uint8))


def test_on_the_current_stream_and_in_a_graph(operands):
    v, o = vk(), operands
    x = o["x"].clone()
    want = v.linear_vdm_w4a4(x, o["qw"], o["ws"], o["b"], 0.95)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = v.linear_vdm_w4a4(x, o["qw"], o["ws"], o["b"], 0.95)
    side.synchronize()
    assert torch.equal(got, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = v.linear_vdm_w4a4(x, o["qw"], o["ws"], o["b"], 0.95)
    for i in range(3):
        x.copy_(o["x"] * (i + 1))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, v.linear_vdm_w4a4(x, o["qw"], o["ws"], o["b"], 0.95))
