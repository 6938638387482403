"""Host-side operator interface of the fused normalization path.

Exposes the names HunyuanVideo blocks import from the reference's
teletron/models/dit/dit_fusedlayers.py -- AdaLNModelFunction (:59),
AdaLNCustom (:139), FusedAdaLayerNormZero (:155), FusedAdaLayerNormZeroSingle
(:226), RMSNormModelFunction (:274), Get_RMSNorm (:350), FP32LayerNorm (:48) --
with the same call signatures, argument meaning, returned gradients and
ValueErrors, backed by the gfx950 kernels.

What differs from the reference, on purpose:
  * the autograd functions keep the INPUT and per-row statistics for backward
    (the reference keeps a second full-size tensor), so forward writes one
    tensor and backward is a single pass plus a fixed-order reducer;
  * scale/shift may carry one row per sample ([B, C]) and their gradients come
    back per sample, which is what the eager formula at :223 computes; the
    reference kernels only handle a single modulation row;
  * both operators accept any row of whole 16-byte pieces (up to 8192 two-byte or
    4096 four-byte columns) in bf16, fp16 or fp32; 128 and 3072 columns
    run the tuned kernels; strided views are read in place at every width, the
    gated and residual forms exist for every supported row, the rotary form
    for 128 columns;
  * gated_residual_layer_norm fuses the residual update in front of a modulated
    LayerNorm (dit_layerspec.py:152-163) into the norm, forward and backward;
  * nothing here falls back silently: with FUSED_KERNELS on, a missing
    extension or a non-GPU tensor raises.  The eager branches below exist only
    because the reference modules select eager math when FUSED_KERNELS is off.
"""
from __future__ import annotations

import functools
import logging
import os
from typing import Optional, Tuple

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd import Function
from torch.overrides import has_torch_function_variadic

log = logging.getLogger(__name__)
log.addHandler(logging.NullHandler())

try:  # same guard as dit_fusedlayers.py:35-45, but the reason is kept for the error message
    from teletron_amd.ext import fused_adaln, fused_rmsnorm
    _IMPORT_ERROR: Optional[BaseException] = None
except ImportError as exc:  # pragma: no cover - exercised only on an unbuilt tree
    fused_adaln = None
    fused_rmsnorm = None
    _IMPORT_ERROR = exc
    log.warning("fused_adaln / fused_rmsnorm extensions not importable (%s); "
                "build them with `python -m teletron_amd.build`.", exc)

TUNED_COLS = (128, 3072)  # the reference's two shapes (the tuned kernels)
_ELEM_BYTES = {torch.bfloat16: 2, torch.float16: 2, torch.float32: 4}
_MAX_PIECES = 1024  # 16-byte pieces per row the kernels are built for
_MAX_JOINT_HEAD_BYTES = 1024  # a head's row the joint q / k / v kernels take: 64 16-byte pieces
_PLAIN = frozenset((torch.Tensor, nn.Parameter, int, float, bool, type(None)))  # what a native node takes for itself
_MAX_JOINT_ROWS = 2 ** 31 - 1  # rows of q (or k) whose groups their 32-bit unit numbers are sure to hold


def cols_supported(cols: int, dtype: torch.dtype) -> bool:
    """Whether the fused kernels take rows of `cols` elements of `dtype`: whole 16-byte pieces,
    at most 8192 two-byte or 4096 four-byte columns, bf16 / fp16 / fp32."""
    size = _ELEM_BYTES.get(dtype)
    if size is None or cols <= 0:
        return False
    vec = 16 // size
    return cols % vec == 0 and cols // vec <= _MAX_PIECES


def wide_forms_supported(cols: int, dtype: torch.dtype) -> bool:
    """Whether the gated residual + AdaLN and the stream-keeping AdaLN take rows of `cols` elements."""
    return cols_supported(cols, dtype)   # every supported row: tuned, any-width and wide-row kernels all have the forms


def _unsupported(cols: int, dtype: torch.dtype) -> str:
    return (f"unsupported cols {cols} for {dtype}: rows must be whole 16-byte pieces, at most 8192 two-byte "
            f"or 4096 four-byte columns, dtype bfloat16, float16 or float32")


def fused_kernels_available() -> bool:
    return fused_adaln is not None and fused_rmsnorm is not None


def fused_kernels_requested() -> bool:
    """The reference's switch: env FUSED_KERNELS parsed as an int (dit_fusedlayers.py:364-365)."""
    flag = os.environ.get("FUSED_KERNELS")
    return bool(int(flag)) if flag else False


def eager_fallback_enabled() -> bool:
    """TELETRON_AMD_FALLBACK=eager restores the reference's silent gating (dit_fusedlayers.py:194-204, 364-370):
    where the fused path cannot run -- extension not importable, tensor not on a GPU, a row the kernels do
    not take, a weight whose dtype differs from the input's -- the modules compute the eager formula
    instead of raising.  Off by default: a training run that asked for fused kernels and silently did not
    get them is the failure this package would rather report."""
    return os.environ.get("TELETRON_AMD_FALLBACK", "").strip().lower() == "eager"


def _require_extension(mod, name: str):
    if mod is None:
        raise RuntimeError(f"{name} extension is not built/importable ({_IMPORT_ERROR}); "
                           "run `python -m teletron_amd.build`")
    return mod


def _require_gpu(t: torch.Tensor, what: str):
    if not t.is_cuda:
        raise ValueError(f"{what}: fused kernels need a GPU tensor, got device {t.device}")


def _aligned_contiguous(t: torch.Tensor) -> torch.Tensor:
    """Contiguous and 16-byte aligned (a contiguous slice may start at any element)."""
    t = t.contiguous()
    return t.clone() if t.data_ptr() % 16 else t


def _native(site, *args):
    """The call as an autograd node of the host runtime (torch_glue.h: forward, graph and backward without Python frames),
    or None where it does not apply as it is -- operands that need preparation, transforms, dispatch modes, a compiler
    tracing this frame -- and the autograd functions below take it.  So they do with a tensor subclass: an input handed
    back as an output keeps its class there, a node's view of it is a plain tensor.  A function mode alone changes
    nothing (has_torch_function_variadic is true for it too, hence the second look)."""
    if torch.compiler.is_compiling() or (has_torch_function_variadic(*args) and not _PLAIN.issuperset(map(type, args))):
        return None
    return site(*args)


class _FirstOrderOnly(Function):
    @staticmethod
    def forward(ctx, grad, *computed_from):
        return grad.data

    @staticmethod
    def backward(ctx, grad):
        raise RuntimeError("the fused norms have no second derivative: a gradient of theirs taken with create_graph=True "
                           "cannot be differentiated again")


def _first_order(backward):
    """A backward whose gradients refuse a second differentiation.  Under create_graph autograd takes gradients that carry
    no graph for constants, and a second derivative would lose their part without a word.  A gradient handed on as it
    came stays differentiable."""
    @functools.wraps(backward)
    def guarded(ctx, *grads):
        result = backward(ctx, *grads)
        if not torch.is_grad_enabled():
            return result
        computed_from = (*ctx.saved_tensors, *grads)   # asking for a derivative by any of it meets the refusal
        return tuple(r if r is None or any(r is g for g in grads) else
                     _FirstOrderOnly.apply(r.detach().requires_grad_(True), *computed_from) for r in result)
    return guarded


class FP32LayerNorm(nn.LayerNorm):
    """LayerNorm evaluated in fp32 and cast back (dit_fusedlayers.py:48-57)."""

    def forward(self, inputs: torch.Tensor) -> torch.Tensor:
        w = None if self.weight is None else self.weight.float()
        b = None if self.bias is None else self.bias.float()
        return F.layer_norm(inputs.float(), self.normalized_shape, w, b, self.eps).to(inputs.dtype)


def _like_modulation(ctx, *grads):
    """Gradients of scale and shift in the shapes and dtypes the caller passed; ctx.mod_meta is None where the rows
    were used as they came, both in one shape."""
    if ctx.mod_meta is None:
        return grads
    return tuple(g.reshape(shape).to(dtype) for g, (shape, dtype) in zip(grads, ctx.mod_meta))


class AdaLNModelFunction(Function):
    """out = LayerNorm(x) * (1 + scale) + shift, no LayerNorm affine.

    apply(x, scale, shift, epsilon, cols) -> out, with gradients for x, scale
    and shift (dit_fusedlayers.py:66,108).  x is [..., cols]; scale and shift are
    [cols] or [B, cols] with B == x.shape[0] (one modulation row per sample).
    A sixth argument True says x is sequence-first, [S, B, cols] with B == x.shape[1]
    (the layout the output norm sees, dit_layerspec.py:72-78): it is normalised in place,
    without regrouping the rows by sample.
    """

    @staticmethod
    def forward(ctx, x, scale, shift, epsilon, cols, *seq_first):
        ext = _require_extension(fused_adaln, "fused_adaln")
        ctx.n_extra = len(seq_first)
        seq_first = bool(seq_first[0]) if seq_first else False
        done = ext.adaln_forward(x, scale, shift, cols, float(epsilon), seq_first)
        if done is not None:   # every operand was ready as it is; anything else is prepared, or refused, below
            out, mean, invvar = done
            ctx.save_for_backward(x, scale, mean, invvar)
            ctx.rows, ctx.cols, ctx.seq_first = invvar.shape[0], cols, seq_first
            ctx.mod_meta = None if scale.shape == shift.shape else [(t.shape, t.dtype) for t in (scale, shift)]
            return out
        _require_gpu(x, "AdaLNModelFunction")
        x = _aligned_contiguous(x)
        scale_c = scale.contiguous()
        shift_c = shift.contiguous()
        if x.numel() % cols != 0:
            raise ValueError(f"Input tensor size {x.numel()} not divisible by cols {cols}")
        if not cols_supported(cols, x.dtype):
            raise ValueError(_unsupported(cols, x.dtype))
        rows = x.numel() // cols
        if scale_c.numel() % cols != 0 or shift_c.numel() != scale_c.numel():
            raise ValueError(f"scale/shift sizes {scale_c.numel()}/{shift_c.numel()} do not match cols {cols}")
        batch = scale_c.numel() // cols
        if seq_first:
            if x.dim() != 3 or x.shape[1] != batch:
                raise ValueError(f"sequence-first input must be [S, {batch}, {cols}], got {tuple(x.shape)}")
        elif batch > 1 and (x.dim() < 2 or x.shape[0] != batch):
            raise ValueError(f"{batch} modulation rows need x.shape[0] == {batch}, got {tuple(x.shape)}")
        if scale_c.dtype != x.dtype or shift_c.dtype != x.dtype:
            scale_c, shift_c = scale_c.to(x.dtype), shift_c.to(x.dtype)

        out = torch.empty_like(x)
        mean = torch.empty(rows, device=x.device, dtype=torch.float32)
        invvar = torch.empty(rows, device=x.device, dtype=torch.float32)
        launch = ext.torch_launch_adaln_forward_stats_seq_first if seq_first else ext.torch_launch_adaln_forward_stats
        launch(out, x, scale_c, shift_c, rows, cols, float(epsilon), mean, invvar)
        ctx.save_for_backward(x, scale_c, mean, invvar)
        ctx.rows, ctx.cols, ctx.seq_first = rows, cols, seq_first
        ctx.mod_meta = [(t.shape, t.dtype) for t in (scale, shift)]
        return out

    @staticmethod
    @_first_order
    def backward(ctx, grad_output):
        x, scale_c, mean, invvar = ctx.saved_tensors
        done = fused_adaln.adaln_backward(grad_output, None, x, scale_c, mean, invvar, ctx.cols, ctx.seq_first)
        if done is not None:
            grad_input, grad_scale, grad_shift = done
            return (grad_input, *_like_modulation(ctx, grad_scale, grad_shift), None, None) + (None,) * ctx.n_extra
        grad_output = _aligned_contiguous(grad_output)
        if grad_output.dtype != x.dtype:
            grad_output = grad_output.to(x.dtype)
        grad_input = torch.empty_like(x)
        grad_scale = torch.empty_like(scale_c)
        grad_shift = torch.empty_like(scale_c)
        launch = (fused_adaln.torch_launch_adaln_backward_x_seq_first if ctx.seq_first
                  else fused_adaln.torch_launch_adaln_backward_x)
        launch(grad_input, grad_scale, grad_shift, grad_output, x, scale_c, mean, invvar, ctx.rows, ctx.cols)
        return (grad_input, *_like_modulation(ctx, grad_scale, grad_shift), None, None) + (None,) * ctx.n_extra


def _adaln(x, scale, shift, eps, cols, *seq_first):
    if fused_adaln is not None:
        done = _native(fused_adaln.adaln_site, x, scale, shift, cols, float(eps), bool(seq_first))
        if done is not None:
            return done
    return AdaLNModelFunction.apply(x, scale, shift, eps, cols, *seq_first)


class AdaLNResidualFunction(Function):
    """(x_same, out) = apply(x, scale, shift, epsilon): out is AdaLNModelFunction's result and x_same is x
    itself, handed back as an output for the caller to continue the residual stream with
    (dit_layerspec.py:126-131 then :152).  Routing the stream through the Function lets backward add the
    gradient it collected downstream to the norm's dx inside the kernel, in place of the separate
    accumulation pass autograd runs when a tensor has two consumers.  Any supported row."""

    @staticmethod
    def forward(ctx, x, scale, shift, epsilon):
        ext = _require_extension(fused_adaln, "fused_adaln")
        ctx.set_materialize_grads(False)
        done = ext.adaln_forward(x, scale, shift, x.shape[-1], float(epsilon), False) if x.dim() else None
        if done is not None:
            out, mean, invvar = done
            ctx.save_for_backward(x, scale, mean, invvar)
            ctx.rows, ctx.cols = invvar.shape[0], x.shape[-1]
            ctx.mod_meta = None if scale.shape == shift.shape else [(t.shape, t.dtype) for t in (scale, shift)]
            return x, out
        _require_gpu(x, "AdaLNResidualFunction")
        cols = x.shape[-1]
        if x.dtype not in _ELEM_BYTES or not wide_forms_supported(cols, x.dtype):
            raise ValueError(f"AdaLNResidualFunction: {_unsupported(cols, x.dtype)}")
        x_c = _aligned_contiguous(x)
        scale_c, shift_c = scale.contiguous().to(x.dtype), shift.contiguous().to(x.dtype)
        if scale_c.numel() % cols or shift_c.numel() != scale_c.numel():
            raise ValueError("scale and shift must each hold [B, cols] elements")
        batch = scale_c.numel() // cols
        if batch > 1 and (x.dim() < 2 or x.shape[0] != batch):
            raise ValueError(f"{batch} modulation rows need x.shape[0] == {batch}, got {tuple(x.shape)}")
        rows = x_c.numel() // cols
        out = torch.empty_like(x_c)
        mean = torch.empty(rows, device=x.device, dtype=torch.float32)
        invvar = torch.empty(rows, device=x.device, dtype=torch.float32)
        ext.torch_launch_adaln_forward_stats(out, x_c, scale_c, shift_c, rows, cols, float(epsilon), mean, invvar)
        ctx.save_for_backward(x_c, scale_c, mean, invvar)
        ctx.rows, ctx.cols = rows, cols
        ctx.mod_meta = [(t.shape, t.dtype) for t in (scale, shift)]
        return x, out

    @staticmethod
    @_first_order
    def backward(ctx, grad_x_same, grad_out):
        x, scale_c, mean, invvar = ctx.saved_tensors
        if grad_out is None:   # only the stream was used: the Function was an identity
            return grad_x_same, None, None, None
        done = fused_adaln.adaln_backward(grad_out, grad_x_same, x, scale_c, mean, invvar, ctx.cols, False)
        if done is not None:
            return (done[0], *_like_modulation(ctx, done[1], done[2]), None)
        grad_out = _aligned_contiguous(grad_out.to(x.dtype))
        grad_input = torch.empty_like(x)
        grad_scale, grad_shift = torch.empty_like(scale_c), torch.empty_like(scale_c)
        if grad_x_same is None:
            fused_adaln.torch_launch_adaln_backward_x(grad_input, grad_scale, grad_shift, grad_out, x, scale_c, mean,
                                                      invvar, ctx.rows, ctx.cols)
        else:
            fused_adaln.torch_launch_adaln_backward_residual(grad_input, grad_scale, grad_shift, grad_out,
                                                             _aligned_contiguous(grad_x_same.to(x.dtype)), x, scale_c,
                                                             mean, invvar, ctx.rows, ctx.cols)
        return (grad_input, *_like_modulation(ctx, grad_scale, grad_shift), None)


def modulated_layer_norm_keeping_stream(x, scale, shift, eps: float = 1e-6):
    """Returns (x, LayerNorm(x) * (1 + scale[:, None]) + shift[:, None]); use the returned x for the residual
    connection so that its gradient is added inside the norm's backward kernel."""
    if fused_adaln is not None:
        done = _native(fused_adaln.adaln_residual_site, x, scale, shift, float(eps))
        if done is not None:
            return done
    return AdaLNResidualFunction.apply(x, scale, shift, eps)


class AdaLNCustom(nn.Module):
    """Module form of AdaLNModelFunction (dit_fusedlayers.py:139-153)."""

    def __init__(self, hidden_size, eps=1e-6):
        super().__init__()
        self.hidden_size = hidden_size
        self.eps = eps

    def forward(self, x, scale, shift):
        cols = self.hidden_size
        for name, t in (("input x", x), ("scale", scale), ("shift", shift)):
            if t.shape[-1] != cols:
                raise ValueError(f"Last dim of {name} must be hidden_size {cols}, got {t.shape[-1]}")
        return _adaln(x, scale, shift, self.eps, cols)


def modulated_layer_norm(x: torch.Tensor, scale: torch.Tensor, shift: torch.Tensor, eps: float = 1e-6,
                         seq_first: bool = False):
    """LayerNorm(x) * (1 + scale[:, None]) + shift[:, None] through the fused kernel.

    The same math as the adaLN-Zero input norm; also what the reference leaves
    un-fused after attention (`norm2` + modulate, dit_layerspec.py:158-167) and
    in the output head (AdaLNContinuous, dit_layerspec.py:55-78).  seq_first: x is [S, B, C]
    and the result is LayerNorm(x) * (1 + scale) + shift broadcast over S, in place."""
    return _adaln(x, scale, shift, eps, x.shape[-1], *((True,) if seq_first else ()))


class GatedResidualAdaLNFunction(Function):
    """(h2, out) = apply(h, attn, gate, scale, shift, epsilon):
    h2 = h + attn * gate[:, None];  out = LayerNorm(h2) * (1 + scale[:, None]) + shift[:, None].

    The residual update and the norm that follows it in the transformer blocks
    (dit_layerspec.py:152-167, :351-352), which the reference runs as separate
    elementwise kernels around the norm.  h, attn [B, S, C]; gate, scale, shift [B, C].
    h2 is the new residual stream; its gradient from later uses is folded into the
    same backward pass.  C: any supported row."""

    @staticmethod
    def forward(ctx, h, attn, gate, scale, shift, epsilon):
        ext = _require_extension(fused_adaln, "fused_adaln")
        ctx.set_materialize_grads(False)  # an unused h2 costs no zero tensor and no read
        done = ext.gated_forward(h, attn, gate, scale, shift, float(epsilon))
        if done is not None:
            h2, out, mean, invvar = done
            ctx.save_for_backward(h2, attn, gate, scale, mean, invvar)
            ctx.rows, ctx.cols, ctx.mod_meta = invvar.shape[0], h.shape[-1], None
            ctx.attn_dtype = attn.dtype
            return h2, out
        _require_gpu(h, "GatedResidualAdaLNFunction")
        cols = h.shape[-1]
        if h.dtype not in _ELEM_BYTES or not wide_forms_supported(cols, h.dtype):
            raise ValueError(f"GatedResidualAdaLNFunction: {_unsupported(cols, h.dtype)}")
        if attn.shape != h.shape:
            raise ValueError(f"attn {tuple(attn.shape)} must have the shape of h {tuple(h.shape)}")
        mods = [t.contiguous().to(h.dtype) for t in (gate, scale, shift)]
        if any(m.numel() != mods[0].numel() or m.numel() % cols for m in mods):
            raise ValueError("gate, scale and shift must each hold [B, cols] elements")
        batch = mods[0].numel() // cols
        if batch > 1 and (h.dim() < 2 or h.shape[0] != batch):
            raise ValueError(f"{batch} modulation rows need h.shape[0] == {batch}, got {tuple(h.shape)}")
        h_c = _aligned_contiguous(h)
        attn_c = _aligned_contiguous(attn.to(h.dtype))
        rows = h_c.numel() // cols
        h2 = torch.empty_like(h_c)
        out = torch.empty_like(h_c)
        mean = torch.empty(rows, device=h.device, dtype=torch.float32)
        invvar = torch.empty(rows, device=h.device, dtype=torch.float32)
        ext.torch_launch_gated_adaln_forward(h2, out, h_c, attn_c, mods[0], mods[1], mods[2], rows, cols,
                                             float(epsilon), mean, invvar)
        ctx.save_for_backward(h2, attn_c, mods[0], mods[1], mean, invvar)
        ctx.rows, ctx.cols = rows, cols
        ctx.mod_meta = [(t.shape, t.dtype) for t in (gate, scale, shift)]
        ctx.attn_dtype = attn.dtype
        return h2, out

    @staticmethod
    @_first_order
    def backward(ctx, grad_h2, grad_out):
        h2, attn_c, gate_c, scale_c, mean, invvar = ctx.saved_tensors
        if grad_out is None:
            grad_out = torch.zeros_like(h2)
        if ctx.mod_meta is None:
            done = fused_adaln.gated_backward(grad_out, grad_h2, h2, attn_c, gate_c, scale_c, mean, invvar, ctx.cols)
            if done is not None:
                return (*done, None)
        grad_out = _aligned_contiguous(grad_out.to(h2.dtype))
        if grad_h2 is not None:
            grad_h2 = _aligned_contiguous(grad_h2.to(h2.dtype))
        dh = torch.empty_like(h2)
        dattn = torch.empty_like(h2)
        dgate, dscale, dshift = (torch.empty_like(m) for m in (gate_c, scale_c, scale_c))
        fused_adaln.torch_launch_gated_adaln_backward(dh, dattn, dgate, dscale, dshift, grad_out, grad_h2, h2,
                                                      attn_c, gate_c, scale_c, mean, invvar, ctx.rows, ctx.cols)
        if ctx.mod_meta is not None:
            dgate, dscale, dshift = (g.reshape(shape).to(dtype)
                                     for g, (shape, dtype) in zip((dgate, dscale, dshift), ctx.mod_meta))
        return dh, dattn.to(ctx.attn_dtype), dgate, dscale, dshift, None


def gated_residual_layer_norm(h, attn, gate, scale, shift, eps: float = 1e-6):
    """Returns (h + attn * gate[:, None], modulated LayerNorm of that sum) from one fused pass."""
    if fused_adaln is not None:
        done = _native(fused_adaln.gated_residual_site, h, attn, gate, scale, shift, float(eps))
        if done is not None:
            return done
    return GatedResidualAdaLNFunction.apply(h, attn, gate, scale, shift, eps)


def _make_modulation_linear(embedding_dim: int, n_chunks: int, bias: bool, linear_parallel: bool, config):
    if not linear_parallel:
        return nn.Linear(embedding_dim, n_chunks * embedding_dim, bias=bias)
    # The reference builds a Megatron/TransformerEngine column-parallel linear here
    # (dit_fusedlayers.py:184-192); that stack is a dependency of the caller, not of this package.
    assert config is not None
    try:
        from megatron.core.transformer.custom_layers.transformer_engine import TEColumnParallelLinear
    except ImportError as exc:
        raise ImportError("linear_parallel=True needs megatron.core's TEColumnParallelLinear; "
                          "pass linear_parallel=False to use nn.Linear") from exc
    return TEColumnParallelLinear(input_size=embedding_dim, output_size=n_chunks * embedding_dim, config=config,
                                  gather_output=False, init_method=config.init_method, bias=bias,
                                  skip_bias_add=False, is_expert=False)


def _gather_modulation(emb, linear_parallel: bool):
    if not linear_parallel:
        return emb
    from megatron.core.tensor_parallel.mappings import gather_from_tensor_model_parallel_region
    return gather_from_tensor_model_parallel_region(emb[0])


class _AdaLNZeroBase(nn.Module):
    """Shared part of the two adaLN-Zero modules: SiLU -> linear -> chunks, then
    the modulated LayerNorm, fused or eager as the constructor flag says."""

    n_chunks = 0

    def __init__(self, embedding_dim: int, norm_type: str, bias: bool, fused_kernels: bool,
                 linear_parallel: bool, config, fused_eps: Optional[float] = None):
        super().__init__()
        self.silu = nn.SiLU()
        self.linear_parallel = linear_parallel
        self.linear = _make_modulation_linear(embedding_dim, self.n_chunks, bias, linear_parallel, config)
        self.fused_kernels = bool(fused_kernels)
        self.embedding_dim = embedding_dim
        self.norm_eps = 1e-5 if norm_type == "fp32_layer_norm" else 1e-6   # of the eager norm built below
        if self.fused_kernels and eager_fallback_enabled() and (
                fused_adaln is None or not cols_supported(embedding_dim, torch.float32)):
            self.fused_kernels = False      # the reference's constructor gate: fall through to the eager norm
        if self.fused_kernels:
            if not cols_supported(embedding_dim, torch.float32):  # the strictest element size
                raise ValueError(f"fused_kernels=True: {_unsupported(embedding_dim, torch.float32)}")
            _require_extension(fused_adaln, "fused_adaln")
            # As in the reference, the fused branch normalises with eps 1e-6 whatever norm_type says
            # (dit_fusedlayers.py:194-195, 249-250), so a checkpoint trained through the reference's fused branch
            # sees the same function here.  The eager branch of norm_type="fp32_layer_norm" builds FP32LayerNorm
            # with nn.LayerNorm's default 1e-5: pass fused_eps=1e-5 to have the fused branch match THAT instead
            # (the two differ visibly only on rows whose variance is not far above 1e-5).
            self.adaLN = AdaLNCustom(embedding_dim, eps=1e-6 if fused_eps is None else float(fused_eps))
        elif norm_type == "layer_norm":
            self.norm = nn.LayerNorm(embedding_dim, elementwise_affine=False, eps=1e-6)
        elif norm_type == "fp32_layer_norm":
            self.norm = FP32LayerNorm(embedding_dim, elementwise_affine=False, bias=False)
        else:
            raise ValueError(f"Unsupported `norm_type` ({norm_type}) provided. "
                             "Supported ones are: 'layer_norm', 'fp32_layer_norm'.")

    def _modulate(self, x, scale, shift):
        if self.fused_kernels:
            if eager_fallback_enabled() and not (x.is_cuda and x.dtype in _ELEM_BYTES):
                xn = F.layer_norm(x, (self.embedding_dim,), None, None, self.adaLN.eps)
                return xn * (1 + scale[:, None]) + shift[:, None]
            return self.adaLN(x, scale, shift)
        return self.norm(x) * (1 + scale[:, None]) + shift[:, None]


class FusedAdaLayerNormZero(_AdaLNZeroBase):
    """adaLN-Zero for the double-stream blocks (dit_fusedlayers.py:155-224):
    returns (x_mod, gate_msa, shift_mlp, scale_mlp, gate_mlp)."""

    n_chunks = 6

    def __init__(self, embedding_dim: int, num_embeddings: Optional[int] = None, norm_type="layer_norm",
                 bias=True, fused_kernels=False, linear_parallel=True, config=None, fused_eps: Optional[float] = None):
        super().__init__(embedding_dim, norm_type, bias, fused_kernels, linear_parallel, config, fused_eps)
        self.emb = None
        if num_embeddings is not None:
            try:
                from diffusers.models.embeddings import CombinedTimestepLabelEmbeddings
            except ImportError as exc:
                raise ImportError("num_embeddings needs diffusers' CombinedTimestepLabelEmbeddings") from exc
            self.emb = CombinedTimestepLabelEmbeddings(num_embeddings, embedding_dim)

    def forward(self, x, timestep=None, class_labels=None, hidden_dtype=None, emb=None):
        if self.emb is not None:
            emb = self.emb(timestep, class_labels, hidden_dtype=hidden_dtype)
        emb = _gather_modulation(self.linear(self.silu(emb)), self.linear_parallel)
        shift_msa, scale_msa, gate_msa, shift_mlp, scale_mlp, gate_mlp = emb.chunk(6, dim=1)
        return self._modulate(x, scale_msa, shift_msa), gate_msa, shift_mlp, scale_mlp, gate_mlp


class FusedAdaLayerNormZeroSingle(_AdaLNZeroBase):
    """adaLN-Zero for the single-stream blocks (dit_fusedlayers.py:226-272):
    returns (x_mod, gate_msa)."""

    n_chunks = 3

    def __init__(self, embedding_dim: int, norm_type="layer_norm", bias=True, fused_kernels=False,
                 linear_parallel=True, config=None, fused_eps: Optional[float] = None):
        super().__init__(embedding_dim, norm_type, bias, fused_kernels, linear_parallel, config, fused_eps)

    def forward(self, x, emb=None):
        emb = _gather_modulation(self.linear(self.silu(emb)), self.linear_parallel)
        shift_msa, scale_msa, gate_msa = emb.chunk(3, dim=1)
        return self._modulate(x, scale_msa, shift_msa), gate_msa


def _strided_rows_ok(x: torch.Tensor) -> bool:
    """True if x can be normalised in place as a strided view: at most 4-D, last
    dimension contiguous, every other stride a non-negative multiple of 16 bytes."""
    if x.is_contiguous() or x.dim() > 4 or x.dim() < 2 or x.stride(-1) != 1:
        return False
    vec = 16 // x.element_size()
    return all(st >= 0 and st % vec == 0 for st in x.stride()[:-1]) and x.data_ptr() % 16 == 0


def _dense_like_layout(x: torch.Tensor) -> torch.Tensor:
    """Uninitialised tensor of x's shape laid out in x's dimension order but without its gaps."""
    order = sorted(range(x.dim()), key=lambda d: (-x.stride(d), d))
    buf = torch.empty([x.shape[d] for d in order], dtype=x.dtype, device=x.device)
    return buf.permute([order.index(d) for d in range(x.dim())])


class RMSNormModelFunction(Function):
    """out = (x * rsqrt(mean(x^2) + eps)) * weight over the last `cols` elements.

    apply(x, weight, epsilon, cols) -> out, with gradients for x and weight
    (dit_fusedlayers.py:281,317).  A non-contiguous view with a contiguous last
    dimension -- the attention caller passes query.transpose(1, 2),
    dit_attention.py:201-212 -- is read in place; the reference copies it first
    (dit_fusedlayers.py:296).  The output is contiguous either way."""

    @staticmethod
    def forward(ctx, x, weight, epsilon, cols):
        ext = _require_extension(fused_rmsnorm, "fused_rmsnorm")
        done = ext.rms_forward(x, weight, cols, float(epsilon))
        if done is not None:
            out, invvar = done
            ctx.save_for_backward(x, weight, invvar)
            ctx.rows, ctx.cols, ctx.strided = invvar.shape[0], cols, False
            ctx.w_shape, ctx.w_dtype = weight.shape, weight.dtype
            return out
        _require_gpu(x, "RMSNormModelFunction")
        if x.numel() % cols != 0:
            raise ValueError(f"Input size {x.numel()} not divisible by cols {cols}")
        if not cols_supported(cols, x.dtype):
            raise ValueError(_unsupported(cols, x.dtype))
        if weight.numel() != cols:
            raise ValueError(f"weight has {weight.numel()} elements, expected cols {cols}")
        strided = x.shape[-1] == cols and _strided_rows_ok(x)
        if not strided:
            x = _aligned_contiguous(x)
        w = weight.contiguous()
        if w.dtype != x.dtype:
            w = w.to(x.dtype)
        rows = x.numel() // cols
        out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        invvar = torch.empty(rows, device=x.device, dtype=torch.float32)
        if strided:
            ext.torch_launch_rms_forward_strided(out, x, w, float(epsilon), invvar)
        else:
            ext.torch_launch_rms_forward(out, x, w, rows, cols, float(epsilon), invvar)
        ctx.save_for_backward(x, w, invvar)
        ctx.rows, ctx.cols, ctx.strided = rows, cols, strided
        ctx.w_shape, ctx.w_dtype = weight.shape, weight.dtype
        return out

    @staticmethod
    @_first_order
    def backward(ctx, grad_output):
        x, w, invvar = ctx.saved_tensors
        done = fused_rmsnorm.rms_backward(grad_output, x, w, invvar, ctx.cols, ctx.strided)
        if done is not None:
            grad_input, grad_weight = done
            return grad_input, grad_weight.reshape(ctx.w_shape).to(ctx.w_dtype), None, None
        grad_output = _aligned_contiguous(grad_output)
        if grad_output.dtype != x.dtype:
            grad_output = grad_output.to(x.dtype)
        grad_weight = torch.empty_like(w)
        if ctx.strided:
            grad_input = _dense_like_layout(x)   # x's dimension order, so the transposed view's grad is cheap to undo
            fused_rmsnorm.torch_launch_rms_backward_strided(grad_input, grad_weight, grad_output, x, w, invvar)
        else:
            grad_input = torch.empty_like(x)
            fused_rmsnorm.torch_launch_rms_backward_x(grad_input, grad_weight, grad_output, x, w, invvar,
                                                      ctx.rows, ctx.cols)
        return grad_input, grad_weight.reshape(ctx.w_shape).to(ctx.w_dtype), None, None


class RMSNorm(nn.Module):
    """RMSNorm with a learnable scale (dit_fusedlayers.py:353-370).  Uses the fused
    kernel when FUSED_KERNELS is on and hidden_size is one the kernels are built
    for; otherwise the reference's eager formula."""

    def __init__(self, hidden_size: int, config=None, eps: float = 1e-6):
        super().__init__()
        self.eps = eps
        self.weight = nn.Parameter(torch.ones(hidden_size))
        self.hidden_size = hidden_size

    def _norm(self, x):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + self.eps)

    def forward(self, x):
        if fused_kernels_requested() and cols_supported(self.hidden_size, x.dtype):
            if not (eager_fallback_enabled() and (fused_rmsnorm is None or not x.is_cuda
                                                  or self.weight.dtype != x.dtype)):
                if fused_rmsnorm is not None:
                    done = _native(fused_rmsnorm.rms_site, x, self.weight, self.hidden_size, float(self.eps))
                    if done is not None:
                        return done
                return RMSNormModelFunction.apply(x, self.weight, self.eps, self.hidden_size)
        return self._norm(x.float()).type_as(x) * self.weight


class QKVSplitNormFunction(Function):
    """(q, k, v) = apply(mixed_qkv, weight_q, weight_k, epsilon)

    mixed_qkv is the fused QKV projection as the attention module views it, [B, S, H, 3*D] with q, k, v
    of one head side by side (dit_attention.py:149-190 with one query head per group).  q and k come
    back RMS-normalised over D as contiguous [B, H, S, D] tensors, v as the transposed view of its
    slice -- what torch.split, .transpose(1, 2), q_layernorm and k_layernorm produce together
    (dit_attention.py:191-214) -- read straight out of mixed_qkv, both in one kernel.
    Backward writes the whole [B, S, H, 3*D] gradient tensor in one kernel (the norms' gradients and the
    copy of v's), so the concatenation that torch.split's backward would run over three separate gradients
    never happens.
    D: any supported row (the rotary form needs 128); rows of more than 1 KiB run one strided norm per tensor."""

    @staticmethod
    def forward(ctx, mixed_qkv, weight_q, weight_k, epsilon, *rotary):
        """rotary: nothing, or (freqs_cos, freqs_sin) as the attention forward receives them
        (dit_attention.py:244-245): float32 [S_img, D].  q and k are then also rotated the way
        apply_rotary_emb does behind q_layernorm / k_layernorm (dit_attention.py:266-273), for the first
        S_img tokens (all of them in the double-stream block, the image part in the single-stream block,
        :435-443), inside the same kernels."""
        ext = _require_extension(fused_rmsnorm, "fused_rmsnorm")
        if len(rotary) not in (0, 2):
            raise ValueError("pass freqs_cos and freqs_sin together, or neither")
        done = ext.qkv_forward(mixed_qkv, weight_q, weight_k, float(epsilon), *(rotary or (None, None)))
        if done is not None:
            ctx.epsilon, ctx.n_rotary, ctx.joint = float(epsilon), len(rotary), True
            ctx.w_meta = [(w.shape, w.dtype) for w in (weight_q, weight_k)]
            ctx.set_materialize_grads(False)
            ctx.save_for_backward(mixed_qkv, weight_q, weight_k, *rotary)
            return tuple(done)
        _require_gpu(mixed_qkv, "QKVSplitNormFunction")
        if mixed_qkv.dim() != 4 or mixed_qkv.shape[-1] % 3:
            raise ValueError(f"mixed_qkv must be [B, S, H, 3*D], got {tuple(mixed_qkv.shape)}")
        cols = mixed_qkv.shape[-1] // 3
        if mixed_qkv.dtype not in _ELEM_BYTES or not cols_supported(cols, mixed_qkv.dtype):
            raise ValueError(f"QKVSplitNormFunction: {_unsupported(cols, mixed_qkv.dtype)}")
        tables = None
        if rotary:
            if cols != 128:
                raise ValueError(f"the fused rotary embedding is built for head dimension 128, got {cols}")
            tables = tuple(_aligned_contiguous(t.to(device=mixed_qkv.device, dtype=torch.float32)) for t in rotary)
            if tables[0].dim() != 2 or tables[0].shape != tables[1].shape or tables[0].shape[1] != cols \
                    or tables[0].shape[0] > mixed_qkv.shape[1]:
                raise ValueError(f"freqs_cos/freqs_sin must both be [S_img <= {mixed_qkv.shape[1]}, {cols}], got "
                                 f"{tuple(tables[0].shape)} and {tuple(tables[1].shape)}")
        if weight_q.numel() != cols or weight_k.numel() != cols:
            raise ValueError(f"weights must have {cols} elements")
        mixed = mixed_qkv if mixed_qkv.is_contiguous() and mixed_qkv.data_ptr() % 16 == 0 else \
            _aligned_contiguous(mixed_qkv)
        q_in, k_in, v_in = (mixed[..., i * cols:(i + 1) * cols].transpose(1, 2) for i in range(3))
        ws = [w.contiguous().to(mixed.dtype) for w in (weight_q, weight_k)]
        B, H, S, _ = q_in.shape
        ctx.cols = cols
        ctx.epsilon = float(epsilon)
        ctx.n_rotary = len(rotary)
        ctx.w_meta = [(w.shape, w.dtype) for w in (weight_q, weight_k)]
        ctx.set_materialize_grads(False)
        # v leaves as a copy-free view only when mixed_qkv itself was usable in place
        v_out = v_in if mixed is mixed_qkv else v_in.clone()
        ctx.joint = cols * mixed.element_size() <= _MAX_JOINT_HEAD_BYTES and (bool(rotary) or B * H * S <= _MAX_JOINT_ROWS)
        if ctx.joint:
            q, k = (torch.empty((B, H, S, cols), dtype=mixed.dtype, device=mixed.device) for _ in range(2))
            ext.torch_launch_qkv_rms_forward(q, k, mixed, ws[0], ws[1], ctx.epsilon, *(tables or (None, None)))
            ctx.save_for_backward(mixed, ws[0], ws[1], *(tables or ()))
            return q, k, v_out
        outs, stats = [], []   # wider heads, more rows: one strided norm per tensor
        for x, w in ((q_in, ws[0]), (k_in, ws[1])):
            out = torch.empty((B, H, S, cols), dtype=mixed.dtype, device=mixed.device)
            invvar = torch.empty(B * H * S, device=mixed.device, dtype=torch.float32)
            ext.torch_launch_rms_forward_strided(out, x, w, ctx.epsilon, invvar)
            outs.append(out)
            stats.append(invvar)
        ctx.save_for_backward(mixed, ws[0], ws[1], stats[0], stats[1])
        return outs[0], outs[1], v_out

    @staticmethod
    @_first_order
    def backward(ctx, grad_q, grad_k, grad_v):
        if ctx.joint:
            mixed, wq, wk, *tables = ctx.saved_tensors
            done = fused_rmsnorm.qkv_backward(grad_q, grad_k, grad_v, mixed, wq, wk, ctx.epsilon, *(tables or (None, None)))
            if done is not None:
                d_mixed, *grads_w = done
                grads_w = [dw.reshape(shape).to(dtype) for dw, (shape, dtype) in zip(grads_w, ctx.w_meta)]
                return (d_mixed, grads_w[0], grads_w[1], None) + (None,) * ctx.n_rotary
            d_mixed = torch.empty_like(mixed)
            grads = [None if g is None else _aligned_contiguous(g.to(mixed.dtype)) for g in (grad_q, grad_k, grad_v)]
            grads_w = [torch.empty_like(w) for w in (wq, wk)]
            fused_rmsnorm.torch_launch_qkv_rms_backward(d_mixed, *grads_w, *grads, mixed, wq, wk, ctx.epsilon,
                                                        *(tables or (None, None)))
            grads_w = [dw.reshape(shape).to(dtype) for dw, (shape, dtype) in zip(grads_w, ctx.w_meta)]
            return (d_mixed, grads_w[0], grads_w[1], None) + (None,) * ctx.n_rotary
        mixed, wq, wk, rstd_q, rstd_k = ctx.saved_tensors
        d_mixed = torch.empty_like(mixed)
        cols = ctx.cols
        slices = [d_mixed[..., i * cols:(i + 1) * cols].transpose(1, 2) for i in range(3)]
        grads_w = []
        for i, (g, w, rstd) in enumerate(((grad_q, wq, rstd_q), (grad_k, wk, rstd_k))):
            dw = torch.empty_like(w)
            if g is None:
                slices[i].zero_()
                dw.zero_()
            else:
                g = _aligned_contiguous(g.to(mixed.dtype))
                x = mixed[..., i * cols:(i + 1) * cols].transpose(1, 2)
                fused_rmsnorm.torch_launch_rms_backward_strided(slices[i], dw, g, x, w, rstd)
            shape, dtype = ctx.w_meta[i]
            grads_w.append(dw.reshape(shape).to(dtype))
        if grad_v is None:
            slices[2].zero_()
        else:
            fused_rmsnorm.torch_launch_copy_rows_strided(slices[2], _aligned_contiguous(grad_v.to(mixed.dtype)))
        return d_mixed, grads_w[0], grads_w[1], None


def rotate_pairs_eager(x: torch.Tensor, freqs_cos: torch.Tensor, freqs_sin: torch.Tensor) -> torch.Tensor:
    """What the reference's callers get from diffusers' apply_rotary_emb(x, (freqs_cos, freqs_sin)) with its
    defaults (real tables, pairs unbound along the last dimension): x [B, H, S, D], tables [S, D]."""
    cos, sin = freqs_cos[None, None].to(x.device), freqs_sin[None, None].to(x.device)
    x_real, x_imag = x.reshape(*x.shape[:-1], -1, 2).unbind(-1)
    x_rotated = torch.stack([-x_imag, x_real], dim=-1).flatten(3)
    return (x.float() * cos + x_rotated.float() * sin).to(x.dtype)


def split_qkv_and_norm(mixed_qkv: torch.Tensor, q_norm: "RMSNorm", k_norm: "RMSNorm", rotary=None):
    """query, key, value as `[B, H, S, D]` from the fused projection `[B, S, H, 3*D]`: the split, the
    transposes and the two per-head RMSNorms of dit_attention.py:149-214 in one call, and with
    rotary=(freqs_cos, freqs_sin) also the rotary embedding of query and key that follows them
    (dit_attention.py:266-273; tables of S_img <= S rows rotate the first S_img tokens, :435-443).
    Fused when FUSED_KERNELS is on and the kernels take the head dimension; the rotation itself is fused at
    head dimension 128 and applied as PyTorch ops to the fused norm's output at any other one.  The
    reference's own sequence of operations otherwise."""
    D = mixed_qkv.shape[-1] // 3
    fusable = (fused_kernels_requested() and mixed_qkv.dtype in _ELEM_BYTES and cols_supported(D, mixed_qkv.dtype)
               and q_norm.eps == k_norm.eps)
    if fusable and (rotary is None or D == 128):
        tables = () if rotary is None else tuple(rotary)
        if fused_rmsnorm is not None and len(tables) in (0, 2):
            done = _native(fused_rmsnorm.qkv_site, mixed_qkv, q_norm.weight, k_norm.weight, float(q_norm.eps),
                           *(tables or (None, None)))
            if done is not None:
                return done
        return QKVSplitNormFunction.apply(mixed_qkv, q_norm.weight, k_norm.weight, q_norm.eps, *tables)
    if fusable:   # the strided-norm fusion is kept; only the rotation runs as separate ops
        query, key, value = QKVSplitNormFunction.apply(mixed_qkv, q_norm.weight, k_norm.weight, q_norm.eps)
    else:
        query, key, value = torch.split(mixed_qkv, [D, D, D], dim=3)
        query, key, value = q_norm(query.transpose(1, 2)), k_norm(key.transpose(1, 2)), value.transpose(1, 2)
    if rotary is not None:
        n = rotary[0].shape[0]
        query = torch.cat([rotate_pairs_eager(query[:, :, :n], *rotary), query[:, :, n:]], dim=2)
        key = torch.cat([rotate_pairs_eager(key[:, :, :n], *rotary), key[:, :, n:]], dim=2)
    return query, key, value


def Get_RMSNorm():
    """Returns the RMSNorm class (the reference hands the class out through a
    factory, dit_fusedlayers.py:350-375)."""
    return RMSNorm


class AdaLNContinuous(nn.Module):
    """The model's output norm (dit_layerspec.py:50-78): SiLU -> Linear -> (scale, shift), then
    norm(x) * (1 + scale) + shift with scale, shift [B, C] broadcast as written there, i.e. along
    x's second-to-last dimension: x is [S, B, C] (the sequence-first layout of the caller) or [B, C].
    Same constructor arguments (config needs .hidden_size only) plus fused_kernels: with it, and
    norm_type "layer_norm", norm and modulation run as the fused AdaLN kernel."""

    def __init__(self, config, conditioning_embedding_dim: int, modulation_bias: bool = True,
                 norm_type: str = "layer_norm", fused_kernels: bool = False):
        super().__init__()
        hidden = config.hidden_size
        self.hidden_size = hidden
        self.adaLN_modulation = nn.Sequential(nn.SiLU(), nn.Linear(conditioning_embedding_dim, hidden * 2,
                                                                   bias=modulation_bias))
        self.fused_kernels = bool(fused_kernels) and norm_type == "layer_norm"
        if norm_type == "layer_norm":
            self.norm = nn.LayerNorm(hidden, elementwise_affine=False, eps=1e-6)
        elif norm_type == "rms_norm":
            # the reference calls RMSNorm(hidden, eps=1e-6), which its own RMSNorm signature rejects
            # (config is a required argument, dit_fusedlayers.py:354); built here as evidently meant
            self.norm = RMSNorm(hidden, config, eps=1e-6)
        else:
            raise ValueError("Unknown normalization type {}".format(norm_type))
        if self.fused_kernels:
            if not cols_supported(hidden, torch.float32):
                raise ValueError(f"fused_kernels=True: {_unsupported(hidden, torch.float32)}")
            _require_extension(fused_adaln, "fused_adaln")

    def forward(self, x: torch.Tensor, conditioning_embedding: torch.Tensor) -> torch.Tensor:
        emb = self.adaLN_modulation(conditioning_embedding)
        scale, shift = torch.chunk(emb, 2, dim=1)
        if not self.fused_kernels:
            return self.norm(x) * (1 + scale) + shift
        if x.dim() == 3:    # [S, B, C]: normalised where it lies, sample b owning rows b, b + B, ...
            return modulated_layer_norm(x, scale, shift, eps=1e-6, seq_first=True)
        if x.dim() == 2:    # [B, C]: one row per sample
            return modulated_layer_norm(x.unsqueeze(1), scale, shift, eps=1e-6).squeeze(1)
        raise ValueError(f"AdaLNContinuous expects x of [S, B, C] or [B, C], got {tuple(x.shape)}")


def install_as_teletron_op() -> None:
    """Registers the extension modules under the reference's top-level names so
    that `import fused_adaln` / `import fused_rmsnorm` in unmodified reference
    code (dit_fusedlayers.py:35-45) picks up this build."""
    import sys
    sys.modules.setdefault("fused_adaln", _require_extension(fused_adaln, "fused_adaln"))
    sys.modules.setdefault("fused_rmsnorm", _require_extension(fused_rmsnorm, "fused_rmsnorm"))
