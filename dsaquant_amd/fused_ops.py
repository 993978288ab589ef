"""Producer fusions around the W4A4 linear that the reference runs as separate
kernels.  They are additions next to the drop-in API (the reference's
``QuantLinear.forward`` has no hook for them), for callers that own the module
code between two linears.

``linear_gelu_vdm_w4a4(x, ...)`` computes ``linear_vdm_w4a4(gelu_tanh(x), ...)``:
the second FFN linear of a Wan block applied to the *pre-activation* output of
the first (FeedForward with activation_fn="gelu-approximate",
vdm_infer/models/wan_vdm/modules/dit_block.py:56 of the reference).  The GELU is
evaluated inside the activation quantizer, so the GELU kernel, its [M, ffn]
fp16 write and the quantizer's re-read of it disappear.

``LnInput`` + ``linear_ln_vdm_w4a4`` / ``qkv_projections_ln`` do the same for
the block's ``norm(x) * (1 + scale) + shift`` (dit_block.py:100, :110) and for
the affine ``norm2`` (:105): the LayerNorm, the modulation and the quantizer
become one pass over ``x``.  ``linear_fused`` adds the consumer side: the gated
residual update ``hidden_states + y * gate`` (:102, :107, :112) in the GEMM epilogue.
"""
from __future__ import annotations

import ctypes
from typing import Optional

import torch

from . import _lib
from .kernels import vdm_w4a4 as _k


def gelu_tanh(x: torch.Tensor) -> torch.Tensor:
    """fp16 GELU (tanh approximation) with the arithmetic of the fused quantizer:
    fp32 evaluation, one rounding to fp16."""
    lib = _k._load_ext()
    xh = x.half().contiguous()
    _k._check_device_tensor(xh, "input", torch.float16)
    n = xh.numel()
    if n % 2:
        raise ValueError("gelu_tanh needs an even number of elements")
    out = torch.empty_like(xh)
    if n:
        with torch.cuda.device(xh.device):
            _lib.check(lib.vdmq_gelu_tanh_f16(xh.data_ptr(), out.data_ptr(), n, _k._stream(xh.device)))
    return out


def linear_gelu_vdm_w4a4(
    x: torch.Tensor,
    qweight: torch.Tensor,
    wscales: torch.Tensor,
    bias: Optional[torch.Tensor] = None,
    clip_ratio: float = 1.0,
    bias_half: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """``linear_vdm_w4a4(gelu_tanh(x), qweight, wscales, bias, clip_ratio, bias_half)``
    in two kernels instead of three; same argument conventions and errors as
    ``linear_vdm_w4a4`` (vdm_w4a4.py:222-244 of the reference)."""
    return linear_fused(x, qweight, wscales, bias, clip_ratio, bias_half, act="gelu_tanh")


class LnInput:
    """A linear's input that is still to be produced: ``LayerNorm(x)`` followed by
    the modulation ``* (1 + a) + b`` (``mode="modulate"``, a = scale, b = shift,
    fp16 arithmetic on the fp16 LayerNorm output) or by the affine ``* a + b``
    (``mode="affine"``, a = weight, b = bias, fp32 arithmetic, one rounding).

    ``x`` is ``[B, L, K]`` (or ``[L, K]``); ``a`` and ``b`` hold one vector per batch
    element (``[B, K]``, ``[B, 1, K]`` or ``[K]``) or one per token (``[B, L, K]``).
    """

    def __init__(self, x: torch.Tensor, a: torch.Tensor, b: torch.Tensor, eps: float, mode: str = "modulate"):
        if mode not in ("modulate", "affine"):
            raise ValueError(f"unknown LayerNorm mode {mode!r}")
        self.shape = tuple(x.shape)
        K = x.shape[-1]
        self._rows = None
        if all(t.dtype is torch.float16 and t.is_contiguous() for t in (x, a, b)) and a.shape == b.shape and K > 0 and a.dim() and a.shape[-1] == K:
            M, nvec = x.numel() // K, a.numel() // K
        else:
            self._rows = tuple(_k._half_rows(t, K) for t in (x, a, b))
            if self._rows[1].shape != self._rows[2].shape:
                raise ValueError("the two LayerNorm vectors must have the same shape")
            M, nvec = self._rows[0].shape[0], self._rows[1].shape[0]
        if nvec == 0 or M % nvec != 0:
            raise ValueError(f"{nvec} vectors do not divide {M} rows")
        self._given = x, a, b
        self.rows_per_vec = M // nvec
        self.eps, self.mode = float(eps), mode
        self.code = _lib.VDMQ_LN_MODULATE if mode == "modulate" else _lib.VDMQ_LN_AFFINE

    def _two_d(self, i: int) -> torch.Tensor:
        # rows of K, made when they are asked for: a call that takes the tensors as they were given (3 us less on the host) never does
        if self._rows is None:
            self._rows = tuple(_k._half_rows(t, self.shape[-1]) for t in self._given)
        return self._rows[i]

    def _replace(self, i: int, rows: torch.Tensor) -> None:
        kept = [self._two_d(j) for j in range(3)]
        kept[i] = rows
        self._rows = tuple(kept)

    x, a, b = (property(lambda self, i=i: self._two_d(i), lambda self, rows, i=i: self._replace(i, rows)) for i in range(3))

    def _args(self):
        M, K = self.x.shape
        return (self.x.data_ptr(), M, K, self.x.stride(0), self.eps, self.code, self.a.data_ptr(), self.b.data_ptr(), self.a.stride(0),
                self.rows_per_vec)

    def materialize(self) -> torch.Tensor:
        """The fp16 tensor the fused quantizer sees (same kernel arithmetic), shaped like ``x``."""
        lib = _k._load_ext()
        _k._check_device_tensor(self.x, "input", torch.float16)
        h = torch.empty_like(self.x)
        if h.numel():
            with torch.cuda.device(h.device):
                _lib.check(lib.vdmq_ln_f16(*self._args(), h.data_ptr(), h.stride(0), _k._stream(h.device)))
        return h.view(self.shape)

    def quantize(self, clip_ratio: float = 1.0, bf6: bool = False):
        """``(qact native, scales)`` of the produced input, as ``quantize_activation_native`` returns them
        (``bf6=True``: as ``quantize_activation_bf6`` does)."""
        lib = _k._load_ext()
        _k._check_device_tensor(self.x, "input", torch.float16)
        M, K = self.x.shape
        dev = self.x.device
        if bf6:
            with torch.cuda.device(dev):
                return _k._quantize_for_gemm(self.x, clip_ratio, 0, True, self._args())
        with torch.cuda.device(dev):
            native = torch.empty((M, _k.k_padded(K) // 2), dtype=torch.uint8, device=dev)
            scales = torch.empty((M,), dtype=torch.float16, device=dev)
            if M:
                _lib.check(lib.vdmq_quantize_act_ln(*self._args(), float(clip_ratio), native.data_ptr(), scales.data_ptr(), _k._stream(dev)))
        return native, scales


def linear_ln_vdm_w4a4(
    pre: LnInput,
    qweight: torch.Tensor,
    wscales: torch.Tensor,
    bias: Optional[torch.Tensor] = None,
    clip_ratio: float = 1.0,
    bias_half: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """``linear_vdm_w4a4(pre.materialize(), ...)`` without materializing: LayerNorm,
    modulation and activation quantizer are one kernel and the GEMM the second, or, for many
    short rows, all of it is one (``vdmq_linear_bf6_ex``)."""
    return linear_fused(pre, qweight, wscales, bias, clip_ratio, bias_half)


class QuantizedInput:
    """A linear's input that is already quantized per token (fp16 scales and the operand form
    of the matrix path its row length takes: 6-bit blocks or native int4 rows): one quantizer
    launch serves every linear that reads the same tensor with the same clip ratio.  The
    cross-attention context is such a tensor -- every block's ``attn2`` K/V projection reads
    ``encoder_hidden_states`` (dit_block.py:109 of the reference), which the reference
    quantizes again in each of them."""

    def __init__(self, x: torch.Tensor, clip_ratio: float = 1.0):
        self.shape = tuple(x.shape)
        self.clip_ratio = float(clip_ratio)
        x_2d, _ = _k._as_2d_half_contiguous(x)
        _k._require(x_2d.is_cuda, "input must be a CUDA tensor")
        self.M, self.K = x_2d.shape
        self.device = x_2d.device
        # (the path of a linear depends on its row length alone, so it is known before any weight is)
        self.bf6 = _k._use_bf6(self.M, 128, self.K)
        if self.M:
            self.qact, self.scales = _k._quantize_for_gemm(x_2d, self.clip_ratio, _lib.VDMQ_ACT_NONE, self.bf6, None)
        else:
            self.qact = self.scales = None


def linear_fused(
    x,
    qweight,
    wscales: Optional[torch.Tensor],
    bias: Optional[torch.Tensor] = None,
    clip_ratio: float = 1.0,
    bias_half: Optional[torch.Tensor] = None,
    *,
    act: Optional[str] = None,
    residual: Optional[torch.Tensor] = None,
    gate: Optional[torch.Tensor] = None,
    split_cols: Optional[int] = None,
) -> torch.Tensor:
    """``residual + linear_vdm_w4a4(act(x), ...) * gate`` in two kernels, or in one where the
    rows are short (``vdmq_linear_bf6_ex``).

    ``x`` is a tensor (optionally with ``act="gelu_tanh"`` applied to it inside the
    quantizer), an ``LnInput`` or a ``QuantizedInput`` (whose clip ratio must be the
    layer's; the GEMM then runs on the matrix path the input was quantized for).  ``gate`` (fp16, one ``[N]`` vector per batch element
    or per token) and ``residual`` (fp16, shaped like the output) are folded into the
    GEMM epilogue as the two fp16 tensor operations of the reference's
    ``hidden_states + attn_output * gate`` (dit_block.py:102, :107, :112); either may
    be omitted.  ``qweight`` may be a ``PreparedWeight`` (then ``wscales`` is ignored): the concatenated weight of a
    fused projection.  ``split_cols``: the output columns as N / split_cols contiguous tensors, stacked in front
    (``[N / split_cols, ..., split_cols]``; without gate and residual).  Returns a new tensor; nothing is updated in place."""
    _k._load_ext()  # raises when the library is missing
    if not isinstance(x, QuantizedInput) and (act is None or act == "gelu_tanh") and (split_cols is None or split_cols):
        out = _native_fused(x, qweight, wscales, bias_half if bias_half is not None else bias, clip_ratio, act, residual, gate, split_cols or 0)
        if out is not None:
            return out
    if isinstance(x, LnInput):
        if act is not None:
            raise ValueError("an activation cannot be combined with a LayerNorm input")
        pre, x_2d, lead = x, x.x, x.shape[:-1]
    elif isinstance(x, QuantizedInput):
        if act is not None:
            raise ValueError("an activation cannot be applied to an input that is already quantized")
        if x.clip_ratio != float(clip_ratio):
            raise ValueError(f"input quantized with clip ratio {x.clip_ratio}, the layer wants {float(clip_ratio)}")
        pre, x_2d, lead = x, None, x.shape[:-1]
    else:
        pre = None
        x_2d, lead = _k._as_2d_half_contiguous(x)
    prepared = isinstance(qweight, _k.PreparedWeight)
    if x_2d is not None:
        _k._require(x_2d.is_cuda, "input must be a CUDA tensor")
        M, K = x_2d.shape
        dev = x_2d.device
    else:
        M, K, dev = pre.M, pre.K, pre.device
    if prepared:
        if qweight.K != K:
            raise ValueError("qweight shape must be [N, K/2]")
    else:
        _k._check_packed_weight(qweight, wscales, K)
    act_code = _k._act_code(act)
    weight = qweight if prepared else _k._prepared_weight(qweight, wscales)
    N = weight.N
    b = bias_half if bias_half is not None else bias
    if b is not None:
        b = _k._half_vector(b)
        _k._check_device_tensor(b, "bias", torch.float16)
        _k._require(b.numel() == N, "bias length must equal N")
    g2 = r2 = None
    rows_per_gate = 1
    if gate is not None:
        if gate.shape[-1] != N:
            raise ValueError(f"gate must have {N} channels")
        g2 = _k._half_rows(gate, N)
        _k._check_device_tensor(g2, "gate", torch.float16)
        if g2.shape[0] == 0 or (M and M % g2.shape[0] != 0):
            raise ValueError(f"{g2.shape[0]} gate vectors do not divide {M} rows")
        rows_per_gate = max(1, M // g2.shape[0])
    if residual is not None:
        if tuple(residual.shape) != tuple(lead) + (N,):
            raise ValueError(f"residual must have shape {tuple(lead) + (N,)}, got {tuple(residual.shape)}")
        r2 = _k._half_rows(residual, N)
        _k._check_device_tensor(r2, "residual", torch.float16)
    if split_cols is not None:
        if gate is not None or residual is not None:
            raise ValueError("a split output takes neither gate nor residual")
        if split_cols <= 0 or split_cols % 64 != 0 or N % split_cols != 0:
            raise ValueError(f"split_cols must be a positive multiple of 64 that divides N={N} (got {split_cols})")
    with _k._on(dev):
        out = torch.empty((M, N) if split_cols is None else (N // split_cols, M, split_cols), dtype=torch.float16, device=dev)
        if M and isinstance(pre, QuantizedInput):
            _k._gemm_dispatch(pre.qact, pre.scales, pre.bf6, weight, b, out, K, gate=g2, rows_per_gate=rows_per_gate, residual=r2)
        elif M:
            bf6 = _k._use_bf6(M, N, K)
            ln_args = None if pre is None else pre._args()
            if bf6 and K <= 16384 and _k.matrix_path() != "bf6":
                _k._linear_bf6_ex(x_2d, clip_ratio, act_code, ln_args, weight, b, out, gate=g2, rows_per_gate=rows_per_gate, residual=r2)
            else:
                operand, scales = _k._quantize_for_gemm(x_2d, clip_ratio, act_code, bf6, ln_args)
                _k._gemm_dispatch(operand, scales, bf6, weight, b, out, K, gate=g2, rows_per_gate=rows_per_gate, residual=r2)
    return out.view(*lead, N) if split_cols is None else out.view(N // split_cols, *lead, split_cols)


def _native_fused(x, qweight, wscales, bias, clip_ratio, act, residual, gate, split_cols):
    weight = qweight if type(qweight) is _k.PreparedWeight else (qweight, wscales)
    if type(x) is LnInput:
        if act is not None:
            return None
        rows, a, b = x._given if x._rows is None else x._rows
        return _k._native_linear(rows, weight, bias, clip_ratio, shape=None if x._rows is None else x.shape, ln=(x.code, x.eps, a, b, x.rows_per_vec),
                                 residual=residual, gate=gate, split_cols=split_cols)
    return _k._native_linear(x, weight, bias, clip_ratio, act=_lib.VDMQ_ACT_NONE if act is None else _lib.VDMQ_ACT_GELU_TANH,
                             residual=residual, gate=gate, split_cols=split_cols)


def qkv_projections_ln(attn, pre: LnInput):
    """Self-attention Q, K, V of ``pre`` through the cached concatenation Wq|Wk|Wv
    (the fused branch of ``get_qkv_projections``, attention.py:41-68 of the
    reference) with the LayerNorm fused into the one activation quantization."""
    from .fused_qkv import _cat_prepared

    w, b = _cat_prepared(attn, ["to_q", "to_k", "to_v"], "qkv")
    n = attn.to_q.vdm_weight_packed.shape[0]
    if getattr(attn, "qkv_contiguous_outputs", False):
        return linear_fused(pre, w, None, None, attn.to_q.kernel_clip_ratio, bias_half=b, split_cols=n).unbind(0)
    return linear_ln_vdm_w4a4(pre, w, None, None, attn.to_q.kernel_clip_ratio, bias_half=b).split(n, dim=-1)


def kv_projections(attn, encoder_hidden_states):
    """Cross-attention K, V through the cached concatenation Wk|Wv (attention.py:70-107 of the reference);
    ``encoder_hidden_states`` is the tensor or a ``QuantizedInput`` of it shared between blocks."""
    from .fused_qkv import _cat_prepared

    w, b = _cat_prepared(attn, ["to_k", "to_v"], "kv")
    n = attn.to_k.vdm_weight_packed.shape[0]
    if getattr(attn, "qkv_contiguous_outputs", False):
        return linear_fused(encoder_hidden_states, w, None, None, attn.to_k.kernel_clip_ratio, bias_half=b, split_cols=n).unbind(0)
    return linear_fused(encoder_hidden_states, w, None, None, attn.to_k.kernel_clip_ratio, bias_half=b).split(n, dim=-1)


# ------------------------------------------------------------------ between the linears

def _strides3(t: torch.Tensor):
    # [B, L, H, D] -> (row, head, batch) for the C interface
    return (ctypes.c_int64 * 3)(t.stride(1), t.stride(2), t.stride(0))


def attention_supported(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> bool:
    """Whether ``attention`` takes these [B, L, heads, head_dim] operands (else: the framework's own attention)."""
    tensors = (q, k, v)
    return (all(t.is_cuda and t.dtype == torch.float16 and t.dim() == 4 and t.stride(3) == 1 and t.data_ptr() % 16 == 0
                and t.device == q.device and not (t.requires_grad and torch.is_grad_enabled())
                and all(st % 8 == 0 for st in t.stride()[:3]) and t.stride(1) <= 1 << 22 for t in tensors)
            and q.shape[3] == k.shape[3] == v.shape[3] == 128 and k.shape == v.shape and q.shape[2] == k.shape[2] and q.shape[0] == k.shape[0]
            and k.shape[1] > 0 and q.shape[0] <= 65535 and q.shape[2] <= 65535)


def attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
    """softmax(q k^T / sqrt(head_dim)) v without a mask: operands [B, L, heads, 128] fp16 (any row, head and batch
    strides that are multiples of 8), result [B, Lq, heads, 128], contiguous."""
    lib = _k._load_ext()
    B, lq, heads, d = q.shape
    with torch.cuda.device(q.device):
        out = torch.empty((B, lq, heads, d), dtype=torch.float16, device=q.device)
        _lib.check(lib.vdmq_attention_f16(q.data_ptr(), _strides3(q), k.data_ptr(), _strides3(k), v.data_ptr(), _strides3(v), out.data_ptr(),
                                          _strides3(out), B, heads, lq, k.shape[1], d, d ** -0.5, _k._stream(q.device)))
    return out


def rms_norm_rope_supported(xs, weights, freqs: Optional[torch.Tensor], heads: int) -> bool:
    """Whether ``rms_norm_rope`` takes these operands."""
    x = xs[0]
    grad = torch.is_grad_enabled()
    if not all(t.is_cuda and t.dtype == torch.float16 and t.dim() == 3 and t.shape == x.shape and t.device == x.device and t.stride(2) == 1
               and t.stride(1) % 8 == 0 and t.stride(1) >= t.shape[2] and (t.shape[0] == 1 or t.stride(0) == t.shape[1] * t.stride(1))
               and t.data_ptr() % 16 == 0 and not (grad and t.requires_grad) for t in xs):
        return False
    _, L, K = x.shape
    if not all(w.is_cuda and w.dtype == torch.float16 and w.device == x.device and w.shape == (K,) and w.is_contiguous()
               and w.data_ptr() % 16 == 0 and not (grad and w.requires_grad) for w in weights):
        return False
    if K % 8 != 0 or K > 8192 or x.numel() == 0:
        return False
    if freqs is None:
        return True
    d = K // heads
    return (d % 8 == 0 and freqs.dtype == torch.complex64 and freqs.device == x.device and tuple(freqs.shape) == (L, 1, d // 2)
            and freqs.is_contiguous() and freqs.data_ptr() % 16 == 0 and not freqs.is_conj() and not (grad and freqs.requires_grad))


def rms_norm_rope(xs, weights, eps: float, freqs: Optional[torch.Tensor], heads: int):
    """RMS-norm of one or two [B, L, K] fp16 tensors (q and k) over K, followed with ``freqs`` (complex64 [L, 1, K / heads
    / 2]) by the rotary embedding of consecutive pairs, in one launch; contiguous results."""
    lib = _k._load_ext()
    B, L, K = xs[0].shape
    dev = xs[0].device
    with torch.cuda.device(dev):
        outs = [torch.empty((B, L, K), dtype=torch.float16, device=dev) for _ in xs]
        args = [a for x, w, o in zip(xs, weights, outs) for a in (x.data_ptr(), x.stride(1), w.data_ptr(), o.data_ptr())]
        if len(xs) == 1:
            args += [None, 0, None, None]
        _lib.check(lib.vdmq_rms_norm_rope_f16(*args, B * L, K, float(eps), None if freqs is None else freqs.data_ptr(), K // heads, L, _k._stream(dev)))
    return outs


def rms_norm_exact(xs, weights, eps: float, floats: bool = False):
    """The RMS-norm of one or two [B, L, K] fp16 tensors with the bits of ``(xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) +
    eps)).half() * weight``, xf = x.float(): the row means stay torch's, whose order of summation they have, and the passes
    around them are two kernels.  ``floats``: the same values as fp32, what a rotary embedding converts them to."""
    lib = _k._load_ext()
    B, L, K = xs[0].shape
    dev = xs[0].device
    with _k._on(dev):
        stream, two = _k._stream(dev), len(xs) == 2
        squares = [torch.empty((B, L, K), dtype=torch.float32, device=dev) for _ in xs]
        args = [a for x, s in zip(xs, squares) for a in (x.data_ptr(), x.stride(1), s.data_ptr())]
        _lib.check(lib.vdmq_row_squares_f32(*args, *(() if two else (None, 0, None)), B * L, K, stream))
        r = [torch.rsqrt(s.mean(dim=-1, keepdim=True) + eps) for s in squares]
        outs = squares if floats else [torch.empty((B, L, K), dtype=torch.float16, device=dev) for _ in xs]  # (the squares have been read)
        args = [a for x, t, w, o in zip(xs, r, weights, outs) for a in (x.data_ptr(), x.stride(1), t.data_ptr(), w.data_ptr(), o.data_ptr())]
        _lib.check(lib.vdmq_scale_rows(*args, *(() if two else (None, 0, None, None, None)), int(floats), B * L, K, stream))
    return outs


def _unseen(*tensors: torch.Tensor) -> bool:
    # Whether nobody sees a difference between tensor operations on these and a kernel with their bits: no mode, transform, trace or
    # tangent.  Without the extension module, which knows (a linear in front has loaded it): not.
    return _lib.host is not None and not torch.compiler.is_compiling() and _lib.host.plain(*tensors)


def rms_norm_exact_supported(xs, weights, heads: int) -> bool:
    """Whether ``rms_norm_exact`` may stand in for the tensor operations on these operands."""
    return _unseen(*xs, *weights) and rms_norm_rope_supported(xs, weights, None, heads)


def modulate_supported(y: torch.Tensor, a: torch.Tensor, b: torch.Tensor) -> bool:
    """Whether ``modulate`` may stand in for the tensor operations on these operands."""
    grad = torch.is_grad_enabled()
    return (_unseen(y, a, b) and y.is_cuda and y.dtype == torch.float32 and y.is_contiguous() and y.dim() == 3 and y.shape[2] % 8 == 0 and y.numel() > 0 and y.data_ptr() % 16 == 0
            and not (grad and y.requires_grad)
            and all(t.dtype == torch.float16 and t.device == y.device and t.numel() == y.shape[2] and t.is_contiguous() and t.data_ptr() % 16 == 0
                    and not (grad and t.requires_grad) for t in (a, b)))


def modulate(y: torch.Tensor, a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """``y.half() * (1 + a) + b`` for an fp32 [B, L, K] and one fp16 vector of K each, the same bits in one pass."""
    lib = _k._load_ext()
    with _k._on(y.device):
        out = torch.empty(y.shape, dtype=torch.float16, device=y.device)
        _lib.check(lib.vdmq_modulate_rows_f16(y.data_ptr(), a.data_ptr(), b.data_ptr(), out.data_ptr(), y.shape[0] * y.shape[1], y.shape[2], _k._stream(y.device)))
    return out


def rope_table(head_dim: int, f: int, h: int, w: int, device) -> torch.Tensor:
    """The complex64 [f * h * w, 1, head_dim / 2] table of rotations, computed on the GPU in double precision."""
    lib = _k._load_ext()
    third = head_dim // 3
    pairs = (head_dim - 2 * third) // 2 + 2 * (third // 2)
    table = torch.empty((f * h * w, 1, pairs), dtype=torch.complex64, device=device)
    with torch.cuda.device(table.device):
        _lib.check(lib.vdmq_rope_table(table.data_ptr(), head_dim, f, h, w, _k._stream(table.device)))
    return table


def timestep_embedding(freq_dim: int, timestep: torch.Tensor) -> torch.Tensor:
    """[B] -> fp16 [B, 2 * (freq_dim // 2)]: cosines, then sines, of the angles, computed in double precision."""
    lib = _k._load_ext()
    t = timestep.double().contiguous()
    out = torch.empty((t.shape[0], freq_dim // 2 * 2), dtype=torch.float16, device=t.device)
    with torch.cuda.device(t.device):
        _lib.check(lib.vdmq_timestep_embedding_f16(t.data_ptr(), out.data_ptr(), t.shape[0], freq_dim // 2, _k._stream(t.device)))
    return out
