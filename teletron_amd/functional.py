"""``torch.autograd.Function`` / ``nn.Module`` surface of the fused ops.

``AdaLNModelFunction`` and ``RMSNormModelFunction`` keep the call signatures and
return orders documented for TeleTron's ops (``teletron_op/README.md:20-92`` and
``:104-172``): ``apply(x, scale, shift, epsilon, cols)`` / ``apply(x, weight,
epsilon, cols)``, backward returning ``(dx, dscale, dshift, None, None)`` /
``(dx, dweight, None, None)``.  Differences, all widening:

* any ``cols`` that is a multiple of 8 (the reference: 3072 / 128 only);
* ``scale`` / ``shift`` may be per-sample ``[B, 1, C]`` as produced by
  ``(modulation + t_mod).chunk(...)`` in ``teletron/models/wan/wan_model.py:234-235``;
* backward saves ``x`` (not ``x_norm`` / the forward output) and recomputes the
  row statistics; parameter gradients are reduced in fp32 and cast once to the
  parameter's dtype.

``FusedRMSNorm`` has the constructor and ``weight`` state-dict key of the Wan
``RMSNorm`` (``wan_model.py:113-124``); ``FusedAdaLN`` replaces
``modulate(nn.LayerNorm(dim, eps, elementwise_affine=False)(x), shift, scale)``
(``wan_model.py:77-78,222-223,236``).
"""
from __future__ import annotations

import torch
import torch.nn as nn
from torch.autograd import Function

from . import ops


def _check_row_groups(x, *params):
    """The ops read a parameter as one vector per consecutive group of rows of the flattened input.
    A parameter with the input's rank is shaped for broadcasting, and must then mean the same thing
    ([B, 1, C] for x [B, S, C] does; [1, S, C] with B > 1 does not): refused rather than misread."""
    for p in params:
        if p is not None and p.dim() == 3 == x.dim() and p.shape == (x.shape[0], 1, x.shape[2]):
            continue
        if p is not None and x.dim() >= 3 and p.dim() == x.dim() and ops.row_groups(x, p) is None:
            raise ValueError(f"a parameter of shape {tuple(p.shape)} does not broadcast over consecutive groups of rows "
                             f"of an input of shape {tuple(x.shape)}")


def _adaln_forward(ctx, x, scale, shift, epsilon, cols):
    if x.numel() % cols != 0 or x.shape[-1] != cols:
        raise ValueError(f"Input tensor size {x.numel()} not divisible by cols {cols}")
    _check_row_groups(x, scale, shift)
    ctx.eps = float(epsilon)
    ctx.scale_meta = (scale.shape, scale.dtype)
    ctx.shift_meta = (shift.shape, shift.dtype)
    x = x.contiguous()
    save = any(ctx.needs_input_grad)
    native = ops.native(x)
    y, scale_c = (native and native.adaln_forward(x, scale, shift, ctx.eps, save)) or \
        ops.adaln_forward_saving(x, scale.detach(), shift.detach(), ctx.eps, save)
    if save:
        ctx.save_for_backward(x, scale_c)
    return y


def _adaln_backward(ctx, grad_output, grad_reduce=None):
    x, scale_c = ctx.saved_tensors
    (sc_shape, sc_dtype), (sh_shape, sh_dtype) = ctx.scale_meta, ctx.shift_meta
    # one rounding to the parameters' dtype in the kernel, unless an exchange in fp32 comes first
    dtype = ops._grad_dtype(sc_dtype) if grad_reduce is None and sc_dtype == sh_dtype else torch.float32
    grad_output = grad_output.contiguous()
    native = ops.native(x)
    if native and grad_reduce is None and sc_dtype == sh_dtype:
        done = native.adaln_backward(grad_output, x, scale_c, ctx.eps, dtype == torch.bfloat16, sc_shape, sh_shape)
        if done:
            dx, dscale, dshift = done
            need = ctx.needs_input_grad
            return dx if need[0] else None, dscale.to(sc_dtype) if need[1] else None, dshift.to(sh_dtype) if need[2] else None
    dx, grads = ops.adaln_backward_packed(grad_output, x, scale_c, ctx.eps, dtype)
    if grad_reduce is not None:
        grad_reduce(grads)                  # fp32 [2, n_batches, C]: dscale and dshift in ONE exchange, before the cast
    if sc_dtype == sh_dtype:
        grads = grads.to(sc_dtype)          # both parameter gradients in one cast
    dx = dx if ctx.needs_input_grad[0] else None
    dscale = grads[0].to(sc_dtype).reshape(sc_shape) if ctx.needs_input_grad[1] else None
    dshift = grads[1].to(sh_dtype).reshape(sh_shape) if ctx.needs_input_grad[2] else None
    return dx, dscale, dshift


_python_apply = Function.apply.__func__    # torch.compile follows this call, but not super() of a Function


class NativeFirst(Function):
    """A Function whose ``apply`` is one native call (csrc/torch_ext/native_ops.cpp) where its arguments are what a model
    passes in earnest: forward and graph node there, backward on the engine's thread without the interpreter.  What
    that declines, and whatever has to see the Python class (a compiler, functorch's transforms, other tensor
    classes), takes ``forward`` and ``backward`` below, which do the same.

    A short pass is host time.  us of one through the Python classes -> through native nodes, of which the engine's
    hand-over to its thread and back takes about 25: RMSNorm 512 x 5120 78 -> 56, 2 x 4096 x 1536 80 -> 60, AdaLN
    3 x 5000 x 1000 87 -> 67, gate 512 x 5120 80 -> 60, gated residual + norm 512 x 5120 119 -> 90; AdaLN 256 x 3072
    without gradients 10.6 -> 6.7."""

    _native = None      # name of the native function, of the class that names it and not of its subclasses

    @classmethod
    def apply(cls, *args):
        if torch.compiler.is_compiling():
            return _python_apply(cls, *args)
        name = cls.__dict__.get("_native")
        if name and args and not torch._C._are_functorch_transforms_active():
            native = ops.native(args[0])
            if native:
                out = getattr(native, name)(*args)
                if out is not None:
                    return out
        return _python_apply(cls, *args)


class AdaLNModelFunction(NativeFirst):
    _native = "adaln"

    @staticmethod
    def forward(ctx, x, scale, shift, epsilon, cols):
        return _adaln_forward(ctx, x, scale, shift, epsilon, cols)

    @staticmethod
    def backward(ctx, grad_output):
        return (*_adaln_backward(ctx, grad_output), None, None)


class AdaLNGradReduceFunction(Function):
    """``AdaLNModelFunction`` for a sequence-sharded (context-parallel) model: every rank holds a slice
    of the rows, so the gradients of ``scale`` / ``shift`` must be summed over the ranks, which is what
    ``ModulateWithCPGradReduce`` does with two all-reduces of bf16 ``[B, 1, C]`` tensors
    (``teletron/core/context_parallel/layers.py:39-53``).  ``grad_reduce`` is any callable that sums an
    fp32 tensor over the group in place (``lambda t: torch.distributed.all_reduce(t, group=cp_group)``);
    it is called once per backward, on the fp32 ``[2, B, C]`` tensor holding both gradients, before
    the cast to the parameters' dtype.  ``apply(x, scale, shift, epsilon, cols, grad_reduce)``."""

    @staticmethod
    def forward(ctx, x, scale, shift, epsilon, cols, grad_reduce):
        ctx.grad_reduce = grad_reduce
        return _adaln_forward(ctx, x, scale, shift, epsilon, cols)

    @staticmethod
    def backward(ctx, grad_output):
        return (*_adaln_backward(ctx, grad_output, ctx.grad_reduce), None, None, None)


def _rmsnorm_backward(grad_output, x, weight, freqs, eps, head_dim, heads, w_shape, w_dtype):
    native = ops.native(x)
    return native and native.rmsnorm_backward(grad_output, x, weight, freqs, eps, head_dim, heads,
                                              w_dtype == torch.bfloat16, w_shape)


class RMSNormModelFunction(NativeFirst):
    _native = "rmsnorm"

    @staticmethod
    def forward(ctx, x, weight, epsilon, cols):
        if x.numel() % cols != 0 or x.shape[-1] != cols:
            raise ValueError(f"Input size {x.numel()} not divisible by cols {cols}")
        ctx.eps = float(epsilon)
        ctx.weight_meta = (weight.shape, weight.dtype)
        if ops.memory_order_view(x)[0] is None:      # dense permuted views are handled without a copy
            x = x.contiguous()
        save = any(ctx.needs_input_grad)
        native = ops.native(x)               # (not for permuted views: it takes dense ones)
        y, weight_c = (native and native.rmsnorm_forward(x, weight, ctx.eps, save)) or \
            ops.rmsnorm_forward_saving(x, weight.detach(), ctx.eps, save)
        if save:
            ctx.save_for_backward(x, weight_c)
        return y

    @staticmethod
    def backward(ctx, grad_output):
        x, weight_c = ctx.saved_tensors
        if x.is_contiguous():
            grad_output = grad_output.contiguous()
        w_shape, w_dtype = ctx.weight_meta
        dx, dweight = _rmsnorm_backward(grad_output, x, weight_c, None, ctx.eps, 0, 0, w_shape, w_dtype) or \
            ops.rmsnorm_backward(grad_output, x, weight_c, ctx.eps, ops._grad_dtype(w_dtype))
        dx = dx if ctx.needs_input_grad[0] else None
        dweight = dweight.to(w_dtype).reshape(w_shape) if ctx.needs_input_grad[1] else None
        return dx, dweight, None, None


class RMSNormRopeFunction(NativeFirst):
    """``rope_apply(RMSNorm(x), freqs, num_heads)`` (``teletron/models/wan/wan_model.py:105-110,154-158``)
    as one op.  ``freqs`` is the model's complex ``[S, 1, head_dim/2]`` table (or real
    ``[S, head_dim/2, 2]`` cos/sin); it gets no gradient."""

    _native = "rope"

    @staticmethod
    def forward(ctx, x, weight, freqs, epsilon, num_heads):
        cols = x.shape[-1]
        if cols % num_heads != 0:
            raise ValueError(f"hidden size {cols} not divisible by num_heads {num_heads}")
        ctx.eps, ctx.head_dim = float(epsilon), cols // num_heads
        ctx.weight_meta = (weight.shape, weight.dtype)
        x = x.contiguous()
        weight_c = weight.detach().to(torch.bfloat16).contiguous()
        freqs_c = ops._check_freqs(freqs.detach(), x, ctx.head_dim)
        ctx.save_for_backward(x, weight_c, freqs_c)
        native = ops.native(x)
        y = native.rope_forward(x, weight_c, freqs_c, ctx.eps, ctx.head_dim, 0) if native else None
        return ops.rmsnorm_rope_forward(x, weight_c, freqs_c, ctx.eps, ctx.head_dim) if y is None else y

    @staticmethod
    def backward(ctx, grad_output):
        x, weight_c, freqs_c = ctx.saved_tensors
        w_shape, w_dtype = ctx.weight_meta
        grad_output = grad_output.contiguous()
        dx, dweight = _rmsnorm_backward(grad_output, x, weight_c, freqs_c, ctx.eps, ctx.head_dim, 0, w_shape, w_dtype) or \
            ops.rmsnorm_rope_backward(grad_output, x, weight_c, freqs_c, ctx.eps, ctx.head_dim, ops._grad_dtype(w_dtype))
        return (dx if ctx.needs_input_grad[0] else None,
                dweight.to(w_dtype).reshape(w_shape) if ctx.needs_input_grad[1] else None, None, None, None)


class RMSNormRopeHeadsFunction(NativeFirst):
    """HunyuanVideo's ``apply_rotary_emb(attn.norm_q(query), image_rotary_emb)``
    (``teletron/models/hunyuan/model.py:92-125``) as one op: ``apply(query, weight, freqs, epsilon)``
    with ``query`` ``[B, H, S, D]`` as the model holds it (the transposed view of a ``[B, S, H, D]``
    buffer; processed in memory order without a copy) or ``[B, S, H, D]`` contiguous, ``weight``
    ``[D]`` and ``freqs`` real ``[S, D/2, 2]`` (cos, sin) or complex ``[S, 1, D/2]`` (no gradient).
    ``rope_table_from_cos_sin`` converts the model's ``(cos, sin)`` pair."""

    _native = "rope_heads"

    @staticmethod
    def forward(ctx, x, weight, freqs, epsilon):
        ctx.eps = float(epsilon)
        ctx.weight_meta = (weight.shape, weight.dtype)
        weight_c = weight.detach().to(torch.bfloat16).contiguous()
        freqs_c = ops._check_freqs(freqs.detach(), x, x.shape[-1])
        ctx.save_for_backward(x, weight_c, freqs_c)
        return ops.rmsnorm_rope_heads_forward(x, weight_c, freqs_c, ctx.eps)

    @staticmethod
    def backward(ctx, grad_output):
        x, weight_c, freqs_c = ctx.saved_tensors
        w_shape, w_dtype = ctx.weight_meta
        dx, dweight = ops.rmsnorm_rope_heads_backward(grad_output, x, weight_c, freqs_c, ctx.eps, ops._grad_dtype(w_dtype))
        return (dx if ctx.needs_input_grad[0] else None,
                dweight.to(w_dtype).reshape(w_shape) if ctx.needs_input_grad[1] else None, None, None)


def rope_table_from_cos_sin(cos: torch.Tensor, sin: torch.Tensor, extra_tokens: int = 0) -> torch.Tensor:
    """``(cos, sin)`` tables ``[S, D]`` in which every value appears twice in a row (the
    ``image_rotary_emb`` pair of HunyuanVideo) -> fp32 ``[S + extra_tokens, D/2, 2]``; the extra
    tokens (text tokens appended after the latent ones, which take no rotation) get (1, 0)."""
    table = torch.stack([cos[:, 0::2].float(), sin[:, 0::2].float()], dim=-1)
    if extra_tokens:
        ident = torch.zeros(extra_tokens, table.shape[1], 2, dtype=table.dtype, device=table.device)
        ident[..., 0] = 1.0
        table = torch.cat([table, ident], dim=0)
    return table.contiguous()


def _gate_forward(ctx, x, gate, residual):
    _check_row_groups(x, gate)
    ctx.gate_meta = (gate.shape, gate.dtype)
    residual = residual.contiguous()
    save = any(ctx.needs_input_grad)
    x = x.contiguous()
    native = ops.native(x)
    out, gate_c = (native and native.gate_forward(x, gate, residual, save)) or \
        ops.gate_residual_forward_saving(x, gate.detach(), residual, save)
    if save:
        ctx.save_for_backward(gate_c, residual)
    return out


def _gate_backward(ctx, grad_output, grad_reduce=None):
    gate_c, residual = ctx.saved_tensors
    g_shape, g_dtype = ctx.gate_meta
    if not (ctx.needs_input_grad[1] or ctx.needs_input_grad[2]):
        return grad_output, None, None
    dtype = ops._grad_dtype(g_dtype) if grad_reduce is None else torch.float32
    dout = grad_output.contiguous()
    native = ops.native(dout)
    vectors = (gate_c.numel() // gate_c.shape[-1], gate_c.shape[-1])
    dres, dgate = (native and native.gate_backward(dout, gate_c, residual, dtype == torch.bfloat16, vectors)) or \
        ops.gate_residual_backward(dout, gate_c, residual, dtype)
    if grad_reduce is not None and ctx.needs_input_grad[1]:
        grad_reduce(dgate)                  # fp32 [n_batches, C], before the cast
    return (grad_output if ctx.needs_input_grad[0] else None,
            dgate.to(g_dtype).reshape(g_shape) if ctx.needs_input_grad[1] else None,
            dres if ctx.needs_input_grad[2] else None)


class GateResidualFunction(NativeFirst):
    """``x + gate * residual`` with the hand-written backward of ``GateWithGradReduce``
    (``teletron/core/context_parallel/layers.py:24-36``) on one GPU: returns
    ``(dout, sum_rows(dout * residual), dout * gate)``, dgate reduced in fp32."""

    _native = "gate_residual"

    @staticmethod
    def forward(ctx, x, gate, residual):
        return _gate_forward(ctx, x, gate, residual)

    @staticmethod
    def backward(ctx, grad_output):
        return _gate_backward(ctx, grad_output)


class GateResidualGradReduceFunction(Function):
    """``GateResidualFunction`` whose gate gradient is summed over the ranks of a sequence-sharded
    model, as ``GateWithGradReduce`` does (``context_parallel/layers.py:31-36``): ``grad_reduce`` is
    called on the fp32 ``[B, C]`` gradient before the cast.  ``apply(x, gate, residual, grad_reduce)``."""

    @staticmethod
    def forward(ctx, x, gate, residual, grad_reduce):
        ctx.grad_reduce = grad_reduce
        return _gate_forward(ctx, x, gate, residual)

    @staticmethod
    def backward(ctx, grad_output):
        return (*_gate_backward(ctx, grad_output, ctx.grad_reduce), None)


class ResidualNormFunction(NativeFirst):
    """``apply(x, residual, gate, scale, shift, epsilon, affine, grad_reduce=None) -> (s, y)``: the residual update of
    a DiT block and the normalisation that reads it, one kernel each way
    (``teletron/models/wan/wan_model.py:239-241``).  ``s = x + gate * residual`` (``gate`` None:
    ``x + residual``); ``y = LayerNorm(s) * (1 + scale) + shift``, or ``LayerNorm(s) * scale + shift``
    with ``affine`` (scale / shift = weight / bias of ``nn.LayerNorm``).  Backward adds the gradients
    arriving at ``s`` and at ``y`` in fp32 and rounds once.  ``grad_reduce`` (sequence-sharded models,
    see ``AdaLNGradReduceFunction``) is called once, on one fp32 tensor holding the gradients of the
    modulation inputs: gate, and scale / shift unless ``affine`` (the weight and bias of an
    ``nn.LayerNorm`` are module parameters, reduced by the model's own parameter hooks)."""

    _native = "residual_norm"

    @staticmethod
    def forward(ctx, x, residual, gate, scale, shift, epsilon, affine, grad_reduce=None):
        ctx.eps, ctx.affine, ctx.grad_reduce = float(epsilon), bool(affine), grad_reduce
        _check_row_groups(x, gate, scale, shift)
        ctx.set_materialize_grads(False)
        ctx.metas = [None if t is None else (t.shape, t.dtype) for t in (gate, scale, shift)]
        save = any(ctx.needs_input_grad)
        residual = residual.contiguous()
        x = x.contiguous()
        native = ops.native(x)
        s, y, gate_c, scale_c = \
            (native and native.residual_norm_forward(x, residual, gate, scale, shift, ctx.eps, ctx.affine, save)) or \
            ops.residual_norm_forward_saving(x, residual, None if gate is None else gate.detach(), scale.detach(),
                                             shift.detach(), ctx.eps, ctx.affine, save)
        if save:
            ctx.save_for_backward(s, residual if gate is not None else None, gate_c, scale_c)
        return s, y

    @staticmethod
    def backward(ctx, grad_s, grad_y):
        s, residual, gate_c, scale_c = ctx.saved_tensors
        if grad_y is None:
            grad_y = torch.zeros_like(s)
        # one rounding in the kernel where every gradient leaves as it is: bf16, one vector per batch
        n = max(c.numel() for c in (gate_c, scale_c) if c is not None)
        direct = ctx.grad_reduce is None and all(
            m is None or (m[1] == torch.bfloat16 and m[0].numel() == n) for m in ctx.metas)
        grad_y, grad_s = grad_y.contiguous(), None if grad_s is None else grad_s.contiguous()
        native = ops.native(s)
        dx, dr, dscale, dshift, dgate = \
            (native and native.residual_norm_backward(grad_y, grad_s, s, residual, gate_c, scale_c, ctx.eps, ctx.affine, direct)) or \
            ops.residual_norm_backward(grad_y, grad_s, s, residual, gate_c, scale_c, ctx.eps, ctx.affine,
                                       torch.bfloat16 if direct else torch.float32)
        if ctx.grad_reduce is not None:
            parts = [g for g in ((dgate,) if ctx.affine else (dscale, dshift, dgate)) if g is not None]
            if parts:
                packed = torch.stack(parts)              # fp32 [k, n_batches, C]: one exchange
                ctx.grad_reduce(packed)
                parts = list(packed.unbind(0))
                if not ctx.affine:
                    dscale, dshift = parts[0], parts[1]
                if dgate is not None:
                    dgate = parts[-1]

        def param_grad(g, meta, needed):
            if not needed or g is None:
                return None
            shape, dtype = meta
            n = 1
            for d in shape:
                n *= d
            if g.numel() != n:            # one parameter vector shared by several batches
                g = g.sum(dim=0)
            return g.to(dtype).reshape(shape)

        need = ctx.needs_input_grad
        return (dx if need[0] else None, dr if need[1] else None, param_grad(dgate, ctx.metas[0], need[2]),
                param_grad(dscale, ctx.metas[1], need[3]), param_grad(dshift, ctx.metas[2], need[4]), None, None, None)


def gate_residual(x, gate, residual, grad_reduce=None):
    """``x + gate * residual``; ``grad_reduce`` as in ``GateResidualGradReduceFunction``."""
    if grad_reduce is not None:
        return GateResidualGradReduceFunction.apply(x, gate, residual, grad_reduce)
    return GateResidualFunction.apply(x, gate, residual)


def residual_adaln(x, residual, gate, shift, scale, eps: float = 1e-6, grad_reduce=None):
    """``s = x + gate * residual`` (gate None: ``x + residual``) and
    ``modulate(layer_norm(s), shift, scale)``; returns ``(s, y)``.  Argument order of ``modulate``.
    Shapes without a fused kernel (rows of at most 256 elements) run the two fused halves.
    ``grad_reduce``: see ``ResidualNormFunction``."""
    if ops.residual_norm_supported(x):
        return ResidualNormFunction.apply(x, residual, gate, scale, shift, eps, False, grad_reduce)
    s = gate_residual(x, gate, residual, grad_reduce) if gate is not None else x + residual
    return s, adaln_modulate(s, shift, scale, eps, grad_reduce)


def residual_layer_norm(x, residual, gate, weight, bias, eps: float = 1e-5, grad_reduce=None):
    """``s = x + gate * residual`` (gate None: ``x + residual``) and
    ``F.layer_norm(s, weight, bias)``; returns ``(s, y)``.  ``grad_reduce``: see ``ResidualNormFunction``
    (it reaches the gate gradient only)."""
    if ops.residual_norm_supported(x):
        return ResidualNormFunction.apply(x, residual, gate, weight, bias, eps, True, grad_reduce)
    s = gate_residual(x, gate, residual, grad_reduce) if gate is not None else x + residual
    return s, torch.nn.functional.layer_norm(s, (s.shape[-1],), weight, bias, eps)


class FusedGate(nn.Module):
    """Drop-in for ``GateModule`` (``teletron/models/wan/wan_model.py:205-210``): ``forward(x, gate, residual)``."""

    def forward(self, x: torch.Tensor, gate: torch.Tensor, residual: torch.Tensor) -> torch.Tensor:
        return GateResidualFunction.apply(x, gate, residual)


def adaln_modulate(x, shift, scale, eps: float = 1e-6, grad_reduce=None):
    """``modulate(layer_norm(x), shift, scale)`` in one kernel (argument order of ``modulate``);
    ``grad_reduce`` as in ``AdaLNGradReduceFunction``."""
    if grad_reduce is not None:
        return AdaLNGradReduceFunction.apply(x, scale, shift, eps, x.shape[-1], grad_reduce)
    return AdaLNModelFunction.apply(x, scale, shift, eps, x.shape[-1])


def rms_norm(x, weight, eps: float = 1e-5):
    return RMSNormModelFunction.apply(x, weight, eps, x.shape[-1])


class FusedRMSNorm(nn.Module):
    """Drop-in for the Wan ``RMSNorm(dim, eps)`` module: same constructor, same ``weight`` key."""

    def __init__(self, dim: int, eps: float = 1e-5):
        super().__init__()
        self.dim = dim
        self.eps = eps
        self.weight = nn.Parameter(torch.ones(dim))

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return RMSNormModelFunction.apply(x, self.weight, self.eps, self.dim)

    def extra_repr(self) -> str:
        return f"{self.dim}, eps={self.eps}"


class FusedAdaLN(nn.Module):
    """LayerNorm without affine parameters fused with ``x * (1 + scale) + shift``; parameter-free."""

    def __init__(self, dim: int, eps: float = 1e-6):
        super().__init__()
        self.dim = dim
        self.eps = eps

    def forward(self, x: torch.Tensor, shift: torch.Tensor, scale: torch.Tensor) -> torch.Tensor:
        return AdaLNModelFunction.apply(x, scale, shift, self.eps, self.dim)

    def extra_repr(self) -> str:
        return f"{self.dim}, eps={self.eps}"
