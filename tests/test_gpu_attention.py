"""The kernels between the W4A4 linears -- attention, q/k RMS-norm with the rotary embedding, its table -- against
64-bit references and the harness's torch operations, at the sizes where their tiles have edges."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _reference(q, k, v):
    q, k, v = (t.cpu().double().transpose(1, 2) for t in (q, k, v))
    scores = q @ k.transpose(-1, -2).contiguous() * q.shape[-1] ** -0.5
    return (scores.softmax(-1) @ v).transpose(1, 2)


def _operand(g, B, L, H, layout):
    if layout == "packed":  # rows of a wider tensor, as a fused projection's strided views are
        return torch.randn((B, L, 3 * H * 128), generator=g, device=DEV).half()[..., H * 128 : 2 * H * 128].unflatten(2, (H, 128))
    if layout == "heads_first":
        return torch.randn((B, H, L, 128), generator=g, device=DEV).half().transpose(1, 2)
    return torch.randn((B, L, H, 128), generator=g, device=DEV).half()


# query tiles of 128 (32 per wave), key steps of 64: both sides of each edge, one key, one query, several heads and batches
@pytest.mark.parametrize("B,lq,lk,H,layout", [(1, 1, 1, 1, "plain"), (1, 31, 63, 2, "packed"), (2, 33, 64, 3, "heads_first"), (1, 127, 65, 1, "plain"),
                                              (1, 129, 127, 2, "packed"), (2, 128, 200, 5, "plain"), (1, 300, 512, 12, "heads_first"),
                                              (1, 257, 8192, 1, "plain"), (1, 257, 8193, 1, "packed")])  # (from 8193 keys on: tiles of 256 queries)
def test_attention_against_64_bits(B, lq, lk, H, layout):
    from dsaquant_amd import fused_ops as f

    g = torch.Generator(device=DEV).manual_seed(lq * 1000 + lk)
    q, k, v = 2.0 * _operand(g, B, lq, H, layout), _operand(g, B, lk, H, layout), _operand(g, B, lk, H, layout)
    assert f.attention_supported(q, k, v)
    got = f.attention(q, k, v)
    want = _reference(q, k, v)
    assert got.shape == want.shape and got.is_contiguous()
    # two roundings to fp16 of relative size 2^-11, of every probability and of the result, and fp32 sums
    bound = 2.0 ** -11 * (1 + v.float().abs().max().item()) * 1.25
    assert (got.cpu().double() - want).abs().max().item() <= bound
    assert ((got.cpu().double() - want).norm() / want.norm()).item() <= 2.0 ** -11


def test_attention_keeps_small_probabilities_large_scores_and_the_tail():
    from dsaquant_amd import fused_ops as f

    # 4096 keys of a probability of about 2^-16 (an fp16 denormal: half a step of its grid is 2^-25, 2^-9 of the value)
    # beside one of probability 1: a 17th of the sum
    q, k = torch.zeros((1, 5, 1, 128), device=DEV).half(), torch.zeros((1, 4097, 1, 128), device=DEV).half()
    q[..., 0] = 8
    k[:, 1:, :, 0] = -16 * 128 ** 0.5 / 1.4426950408889634 / 8
    v = torch.ones_like(k)
    v[:, 0] = 0
    want = _reference(q, k, v)[0, 0, 0, 0].item()
    assert abs(f.attention(q, k, v)[0, 0, 0, 0].item() - want) <= (2.0 ** -9 + 2.0 ** -11) * want
    # the maximum grows in every step of 64 keys (each rescales what was accumulated); the last step has one key
    k = (torch.arange(193, device=DEV) // 64 * 3.0).half().view(1, -1, 1, 1).expand(1, 193, 1, 128).contiguous()
    q = torch.ones((1, 40, 1, 128), device=DEV).half()
    v = torch.randn((1, 193, 1, 128), device=DEV).half()
    assert (f.attention(q, k, v).cpu().double() - _reference(q, k, v)).abs().max().item() <= 2.0 ** -10 * 4
    # an infinite value beside the unused part of the last step; a score that is NaN stays in its row
    v[:, -1, :, 0] = float("inf")
    out = f.attention(q, k, v)
    assert torch.isinf(out[..., 0]).all() and torch.isfinite(out[..., 1:]).all()
    q[:, 3, :, 0] = float("nan")
    out = f.attention(q, k, v)
    assert torch.isnan(out[:, 3]).all() and torch.isfinite(out[:, 4:, :, 1:]).all()


@pytest.mark.parametrize("exponent", [-20.5, -23.5, -25.5, -28.0])
def test_attention_keeps_many_tiny_probabilities(exponent):
    """One key of probability about 1 and 32000 of 2^exponent each: denormal in fp16 or below it, but what v has is theirs."""
    from dsaquant_amd import fused_ops as f

    q, k = torch.zeros((1, 3, 1, 128), device=DEV).half(), torch.zeros((1, 32001, 1, 128), device=DEV).half()
    q[..., 0] = 8
    k[:, 1:, :, 0] = exponent * 128 ** 0.5 / 1.4426950408889634 / 8
    v = torch.ones_like(k)
    v[:, 0] = 0
    want = _reference(q, k, v)[0, 0, 0, 0].item()
    # the probabilities round alike, by 2^-11 at most, and so does the result (fp16, normal); the sums are fp32
    assert abs(f.attention(q, k, v)[0, :, 0, 0].double().cpu() - want).max().item() <= 1.05 * 2.0 ** -10 * want


def test_attention_with_scores_that_fp32_holds_coarsely():
    """Scores around 2^20 and 2^25 (times log2 e): a step of fp32 there is up to 4, no probability may leave fp16's range."""
    from dsaquant_amd import fused_ops as f

    for size in (2048.0, 3000.0, 4096.0, 20000.0):
        q, k = torch.zeros((1, 33, 1, 128), device=DEV).half(), torch.zeros((1, 70, 1, 128), device=DEV).half()
        q[..., :4], k[..., :4] = size, size / 2
        k[:, 37, :, :4] = size
        v = torch.randn((1, 70, 1, 128), device=DEV).half()
        assert torch.equal(f.attention(q, k, v), v[:, 37:38].expand(1, 33, 1, 128))


def test_attention_refuses_what_it_is_not_for():
    from dsaquant_amd import _lib
    from dsaquant_amd import fused_ops as f

    t = torch.zeros((1, 8, 2, 128), device=DEV).half()
    assert not f.attention_supported(t.float(), t.float(), t.float())
    assert not f.attention_supported(t[..., :64], t[..., :64], t[..., :64])
    assert not f.attention_supported(t, t[:, :0], t[:, :0])
    with pytest.raises(_lib.VdmqError):
        f.attention(t[..., :64], t[..., :64], t[..., :64])


# one to sixteen chunks of 512, rows that are not a multiple of a workgroup's four, strided inputs
@pytest.mark.parametrize("B,fhw,K,H", [(1, (1, 1, 1), 128, 1), (1, (2, 3, 5), 512, 4), (2, (1, 3, 7), 1536, 12), (1, (3, 4, 6), 3072, 24),
                                       (1, (1, 5, 7), 5120, 40), (1, (2, 2, 3), 8192, 64)])
def test_norm_and_rope_against_the_torch_operations(B, fhw, K, H):
    from dsaquant_amd import fused_ops as f
    from dsaquant_amd import wan_harness as W

    L = fhw[0] * fhw[1] * fhw[2]
    g = torch.Generator(device=DEV).manual_seed(K)
    wide = (3 * torch.randn((B, L, 2 * K), generator=g, device=DEV)).half()
    xs, ws = wide.split(K, dim=-1), [(1 + 0.1 * torch.randn(K, generator=g, device=DEV)).half() for _ in range(2)]
    host = W.rope_frequencies(K // H, *fhw, "cpu")
    freqs = f.rope_table(K // H, *fhw, DEV)
    # double precision on both sides, rounded to float: equal but for a rounding boundary between two double results
    assert (torch.view_as_real(freqs).cpu() - torch.view_as_real(host)).abs().max().item() <= 2.0 ** -23
    assert f.rms_norm_rope_supported(xs, ws, freqs, H)
    turned = f.rms_norm_rope(xs, ws, 1e-6, freqs, H)
    for i in range(2):
        norm = W.RMSNormAcrossHeads(K, 1e-6).to(DEV).half()
        norm.weight.data.copy_(ws[i])
        with torch.no_grad():
            plain = norm(xs[i])
            want = W.apply_rope(plain.unflatten(2, (H, -1)), freqs).flatten(2, 3)
        got = f.rms_norm_rope((xs[i],), (ws[i],), 1e-6, None, H)[0]
        # the mean of squares in another order: isolated values round the other way, by one fp16 step of theirs and one behind
        # the weight; the rotation mixes the two of a pair and rounds once more
        pair = plain.float().unflatten(2, (-1, 2)).norm(dim=-1, keepdim=True).expand(-1, -1, -1, 2).flatten(2, 3)
        for a, b, bound in ((got, plain, 2.0 ** -9 * plain.float().abs() + 2.0 ** -24), (turned[i], want, 3 * 2.0 ** -10 * pair + 2.0 ** -23)):
            assert (a != b).float().mean().item() <= 5e-3
            assert ((a.float() - b.float()).abs() <= bound).all()


def test_harness_attention_runs_on_the_kernels():
    """Same module, same inputs: the library's kernels between the linears against the torch operations."""
    from dataclasses import replace

    from dsaquant_amd import fused_ops
    from dsaquant_amd import wan_harness as W

    args = replace(W.WAN21_1P3B, num_layers=1, num_heads=2, ffn_dim=512, text_dim=128)
    model = W.build_quantized(args, DEV, seed=3)
    for module in (model.blocks[0].attn1, model.blocks[0].attn2):
        module.fuse_attention = True
    g = torch.Generator(device=DEV).manual_seed(4)
    latent = torch.randn((1, 16, 3, 10, 14), generator=g, device=DEV).half()
    ctx, t = torch.randn((1, 77, args.text_dim), generator=g, device=DEV).half(), torch.tensor([500.0], device=DEV)
    calls = []
    kernel = fused_ops.attention
    fused_ops.attention = lambda *a: (calls.append(1), kernel(*a))[1]
    supported = fused_ops.attention_supported, fused_ops.rms_norm_rope_supported
    try:
        with torch.no_grad():
            got = model(latent, t, ctx)
            assert len(calls) == 2
            fused_ops.attention_supported = fused_ops.rms_norm_rope_supported = lambda *a: False
            want = model(latent, t, ctx)
            assert len(calls) == 2
    finally:
        fused_ops.attention = kernel
        fused_ops.attention_supported, fused_ops.rms_norm_rope_supported = supported
    # rounding steps of the following int4 quantizers, as between any two correct implementations
    assert ((got.float() - want.float()).norm() / want.float().norm()).item() <= 0.03


@pytest.mark.parametrize("freq_dim,dtype,n", [(256, torch.float32, 1), (2, torch.float64, 3), (514, torch.float16, 5), (255, torch.int64, 257)])
def test_timestep_embedding_against_the_tensor_operations(freq_dim, dtype, n):
    from dsaquant_amd import fused_ops as f
    from dsaquant_amd import wan_harness as W

    t = torch.linspace(0, 1000, 2 * n, dtype=torch.float64, device=DEV).to(dtype)[::2]
    want = W.timestep_embedding(freq_dim, t).half()
    got = f.timestep_embedding(freq_dim, t)
    assert got.shape == want.shape and got.dtype == torch.float16
    # double on both sides: apart from a result next to a rounding boundary the same fp16 value, there one step of at most 2^-11
    assert (got != want).float().mean().item() <= 1e-3
    assert (got.float() - want.float()).abs().max().item() <= 2.0 ** -11


def test_harness_head_runs_on_the_layernorm_kernel():
    """The last LayerNorm and its modulation, and the timestep embedding, against the tensor operations on one model: no
    quantizer follows the first, and the second gives the same fp16 values."""
    from dataclasses import replace

    from dsaquant_amd import fused_ops
    from dsaquant_amd import wan_harness as W

    args = replace(W.WAN21_1P3B, num_layers=1, num_heads=2, ffn_dim=512, text_dim=128)
    model = W.build_quantized(args, DEV, seed=5)
    for block in model.blocks:
        block.fuse_ln = True
    model.fuse_head = True
    g = torch.Generator(device=DEV).manual_seed(6)
    latent = torch.randn((1, 16, 1, 6, 10), generator=g, device=DEV).half()
    ctx, t = torch.randn((1, 77, args.text_dim), generator=g, device=DEV).half(), torch.tensor([500.0], device=DEV)
    calls = []
    materialize, plain = fused_ops.LnInput.materialize, W._plain_fp16
    fused_ops.LnInput.materialize = lambda self: (calls.append(1), materialize(self))[1]
    try:
        with torch.no_grad():
            got = model(latent, t, ctx)
            assert len(calls) == 1
            W._plain_fp16 = lambda x: False
            want = model(latent, t, ctx)
            assert len(calls) == 1
    finally:
        fused_ops.LnInput.materialize, W._plain_fp16 = materialize, plain
    # statistics in another order: isolated fp16 steps of the normalised tokens
    assert ((got.float() - want.float()).norm() / want.float().norm()).item() <= 2.0 ** -11


def test_harness_without_quantized_linears_needs_nothing_from_the_library(monkeypatch):
    """A model whose linears are torch's runs on the GPU without the library, and with the same table of rotations."""
    from dataclasses import replace

    from dsaquant_amd import _lib, fused_ops
    from dsaquant_amd import wan_harness as W
    from dsaquant_amd.kernels import vdm_w4a4 as v

    for shape in ((3, 30, 52), (21, 1, 1), (1, 5, 7)):
        assert torch.equal(fused_ops.rope_table(128, *shape, DEV), W.rope_frequencies(128, *shape, DEV))

    def refuse(*args, **kwargs):
        raise RuntimeError("the library was asked for")

    monkeypatch.setattr(v, "_load_ext", refuse)
    monkeypatch.setattr(_lib, "load", refuse)
    args = replace(W.WAN21_1P3B, num_layers=1, num_heads=2, ffn_dim=512, text_dim=128)
    torch.manual_seed(8)
    model = W.WanDiT(args).half().to(DEV)
    latent, ctx = torch.randn((1, 16, 1, 6, 10), device=DEV).half(), torch.randn((1, 9, args.text_dim), device=DEV).half()
    with torch.no_grad():
        assert torch.isfinite(model(latent, torch.tensor([500.0], device=DEV), ctx)).all()


def test_harness_keeps_the_torch_operations_between_the_linears_unless_asked(monkeypatch):
    """Norms, rotation, attention and the head's LayerNorm on the library's kernels are as exact as the torch operations but not
    their bits, which the quantizers after them amplify: a forward takes them only with the module's switch, whatever else
    is fused."""
    from dataclasses import replace

    from dsaquant_amd import fused_ops
    from dsaquant_amd import wan_harness as W

    args = replace(W.WAN21_1P3B, num_layers=2, num_heads=2, ffn_dim=512, text_dim=128)
    model = W.build_quantized(args, DEV, seed=9)
    for block in model.blocks:
        block.fuse_ln = block.fuse_residual = block.ffn.fuse_gelu = True
    g = torch.Generator(device=DEV).manual_seed(10)
    latent = torch.randn((1, 16, 2, 10, 14), generator=g, device=DEV).half()
    ctx, t = torch.randn((1, 77, args.text_dim), generator=g, device=DEV).half(), torch.tensor([500.0], device=DEV)

    calls = []
    for owner, name in ((fused_ops, "attention"), (fused_ops, "rms_norm_rope"), (fused_ops.LnInput, "materialize")):
        kernel = getattr(owner, name)
        monkeypatch.setattr(owner, name, lambda *a, kernel=kernel, name=name: (calls.append(name), kernel(*a))[1])
    with torch.no_grad():
        model(latent, t, ctx)
        assert calls == []
        model.fuse_head = True
        for block in model.blocks:
            block.attn1.fuse_attention = block.attn2.fuse_attention = True
        model(latent, t, ctx)
    assert calls == ["rms_norm_rope", "attention", "rms_norm_rope", "rms_norm_rope", "attention"] * 2 + ["materialize"]


@pytest.mark.parametrize("hook", ["forward", "forward_pre", "global", "replaced"])
def test_harness_calls_norms_that_carry_hooks(hook):
    """With the kernels switched on, a norm that more than its own forward hangs on is still called."""
    from dataclasses import replace

    from dsaquant_amd import wan_harness as W

    args = replace(W.WAN21_1P3B, num_layers=1, num_heads=2, ffn_dim=512, text_dim=128)
    model = W.build_quantized(args, DEV, seed=11)
    attn = model.blocks[0].attn1
    attn.fuse_attention = model.blocks[0].attn2.fuse_attention = True
    seen, handle = [], None
    if hook == "forward":
        handle = attn.norm_k.register_forward_hook(lambda m, i, o: seen.append(m))
    elif hook == "forward_pre":
        handle = attn.norm_k.register_forward_pre_hook(lambda m, i: seen.append(m))
    elif hook == "global":
        handle = torch.nn.modules.module.register_module_forward_hook(lambda m, i, o: seen.append(m))
    else:
        plain = attn.norm_k.forward
        attn.norm_k.forward = lambda x: (seen.append(attn.norm_k), plain(x))[1]
    try:
        with torch.no_grad():
            model(torch.randn((1, 16, 1, 6, 10), device=DEV).half(), torch.tensor([500.0], device=DEV), torch.randn((1, 7, args.text_dim), device=DEV).half())
    finally:
        if handle is not None:
            handle.remove()
    assert attn.norm_k in seen


def _same_bits(a, b):
    assert a.shape == b.shape and a.dtype == b.dtype and a.is_contiguous() == b.is_contiguous()
    assert torch.equal(torch.isnan(a), torch.isnan(b))
    zero = torch.zeros((), dtype=a.dtype, device=a.device)
    ints = torch.int16 if a.dtype == torch.float16 else torch.int32
    assert torch.equal(torch.where(torch.isnan(a), zero, a).view(ints), torch.where(torch.isnan(b), zero, b).view(ints))


# one piece of eight, rows that fill no workgroup, more rows than one; row strides beyond the row
@pytest.mark.parametrize("B,L,K,pad", [(1, 1, 8, 0), (1, 7, 1536, 0), (2, 33, 5120, 0), (1, 513, 4104, 64), (1, 4680, 1536, 3072)])
def test_norm_around_its_means_has_the_bits_of_the_tensor_operations(B, L, K, pad):
    from dsaquant_amd import fused_ops as f
    from dsaquant_amd import wan_harness as W

    g = torch.Generator(device=DEV).manual_seed(B + L + K)
    xs = [torch.randn((B, L, K + pad), generator=g, device=DEV).half()[..., :K] for _ in range(2)]
    for x in xs:  # subnormals, zeros, an overflowing square's row, infinities, a NaN
        x[:, ::5] *= 1e-6
        x[0, 0, :4] = torch.tensor([0.0, -0.0, 6e-8, 65504.0], device=DEV).half()
        if L > 6:
            x[0, 2] = 65504.0
            x[0, 3, 1], x[0, 4, 2], x[0, 5] = float("inf"), float("nan"), 0.0
    norms = [W.RMSNormAcrossHeads(K, 1e-6).half().to(DEV) for _ in xs]
    with torch.no_grad():
        for n in norms:
            n.weight.copy_(torch.randn(K, generator=g, device=DEV))
            n.weight[:2] = torch.tensor([6e-8, 0.0], device=DEV)
        assert f.rms_norm_rope_supported(xs, [n.weight for n in norms], None, 1)
        want = [n(x) for n, x in zip(norms, xs)]
        weights = [n.weight for n in norms]
        for got, w in zip(f.rms_norm_exact(xs, weights, 1e-6), want):
            _same_bits(got, w)
        for got, w in zip(f.rms_norm_exact(xs, weights, 1e-6, floats=True), want):
            _same_bits(got, w.float())
        _same_bits(f.rms_norm_exact(xs[1:], weights[1:], 1e-6)[0], want[1])
        a, b = (torch.randn((1, 1, K), generator=g, device=DEV).half() for _ in range(2))
        y = torch.randn((B, L, K), generator=g, device=DEV) * 10
        y[0, 0, :3] = torch.tensor([1e6, float("nan"), 1e-7], device=DEV)
        assert f.modulate_supported(y, a, b) and not f.modulate_supported(y.half(), a, b)
        _same_bits(f.modulate(y, a, b), y.half() * (1 + a) + b)


def _small_model():
    from dataclasses import replace

    from dsaquant_amd import wan_harness as W

    args = replace(W.WAN21_1P3B, num_layers=1, num_heads=2, ffn_dim=512, text_dim=128)
    return W.build_quantized(args, DEV, seed=12), args


@pytest.mark.parametrize("kind", ["function", "dispatch"])
def test_operation_modes_see_the_norms_and_the_modulation(monkeypatch, kind):
    """What no switch turns on is not there for who watches the tensor operations: every one of the norms and the head's reaches a mode."""
    from collections import Counter

    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from dsaquant_amd import fused_ops

    model, args = _small_model()
    g = torch.Generator(device=DEV).manual_seed(13)
    latent = torch.randn((1, 16, 1, 6, 10), generator=g, device=DEV).half()
    ctx, t = torch.randn((1, 77, args.text_dim), generator=g, device=DEV).half(), torch.tensor([500.0], device=DEV)

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen[getattr(func, "__name__", str(func))] += 1
            return func(*args, **(kwargs or {}))

    class Dispatched(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen[str(func)] += 1
            return func(*args, **(kwargs or {}))

    def under_mode():
        with (Functions if kind == "function" else Dispatched)():
            return model(latent, t, ctx)

    with torch.no_grad():
        want = model(latent, t, ctx)
        seen = Counter()
        got, first = under_mode(), seen
        monkeypatch.setattr(fused_ops, "rms_norm_exact_supported", lambda *a: False)
        monkeypatch.setattr(fused_ops, "modulate_supported", lambda *a: False)
        seen = Counter()
        under_mode()
    assert torch.equal(got, want)
    for name in ("rsqrt", "pow", "mean") if kind == "function" else ("aten.rsqrt.default", "aten.pow.Tensor_Scalar", "aten.mean.dim", "aten.mul.Tensor", "aten.add.Tensor"):
        assert first[name] == seen[name] > 0


def test_tangents_pass_the_norms_and_the_head():
    """Forward-mode differentiation through the residual stream does not end, unnoticed, at a norm or at the head."""
    import torch.autograd.forward_ad as fwad

    model, args = _small_model()
    attn = model.blocks[0].attn1
    g = torch.Generator(device=DEV).manual_seed(14)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device=DEV).half()  # noqa: E731
    x, t, scale, shift = rnd(1, 40, args.dim), rnd(1, 40, args.dim), rnd(1, 1, args.dim), rnd(1, 1, args.dim)
    with torch.no_grad():
        attn.to_q(x)  # (loads the library)
        plain = attn._normed(x, attn.norm_q), model._head_norm(x, scale, shift)
        with fwad.dual_level():
            dual = fwad.make_dual(x, t)
            for out, want in zip((attn._normed(dual, attn.norm_q), model._head_norm(dual, scale, shift)), plain):
                primal, tangent = fwad.unpack_dual(out)
                assert tangent is not None and torch.isfinite(tangent).all() and torch.equal(primal, want)
            out = model._head_norm(x, scale, fwad.make_dual(shift, scale))
            assert fwad.unpack_dual(out).tangent is not None


def test_norm_kernels_leave_subclasses_alone():
    from dsaquant_amd import fused_ops as f

    class Sub(torch.Tensor):
        pass

    model, args = _small_model()
    x = torch.ones((1, 8, args.dim), device=DEV).half()
    w = [torch.ones(args.dim, device=DEV).half()]
    model.blocks[0].attn1.to_q(x)
    assert f.rms_norm_exact_supported([x], w, 2) and not f.rms_norm_exact_supported([x.as_subclass(Sub)], w, 2)
    assert isinstance(model._head_norm(x.as_subclass(Sub), x[:, :1], x[:, :1]), Sub)


@pytest.mark.parametrize("frames,h,w", [(1, 6, 10), (2, 10, 14), (3, 34, 50)])
def test_harness_forward_keeps_its_bits_on_the_norm_kernels(monkeypatch, frames, h, w):
    from dataclasses import replace

    from dsaquant_amd import fused_ops
    from dsaquant_amd import wan_harness as W

    args = replace(W.WAN21_1P3B, num_layers=2, num_heads=2, ffn_dim=512, text_dim=128)
    model = W.build_quantized(args, DEV, seed=12)
    g = torch.Generator(device=DEV).manual_seed(13)
    latent = torch.randn((1, 16, frames, h, w), generator=g, device=DEV).half()
    ctx, t = torch.randn((1, 77, args.text_dim), generator=g, device=DEV).half(), torch.tensor([500.0], device=DEV)
    calls = []
    for name in ("rms_norm_exact", "modulate"):
        kernel = getattr(fused_ops, name)
        monkeypatch.setattr(fused_ops, name, lambda *a, kernel=kernel, name=name, **k: (calls.append(name), kernel(*a, **k))[1])
    with torch.no_grad():
        got = model(latent, t, ctx)
        assert calls == ["rms_norm_exact"] * 6 + ["modulate"]  # per block: q and k, then q, then k of the context
        monkeypatch.setattr(fused_ops, "rms_norm_rope_supported", lambda *a: False)
        monkeypatch.setattr(fused_ops, "modulate_supported", lambda *a: False)
        want = model(latent, t, ctx)
    assert len(calls) == 7 and torch.equal(got, want)
