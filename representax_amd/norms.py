"""The normalisations between a layer's quantized linears, through the fused
HIP kernels where those apply: LayerNorm and RMSNorm with float32 statistics
(src/representax/models/components.py:110-150), the residual addition before
them, and the per-head RMSNorm of queries and keys with the rotary rotation
after it (src/representax/models/qwen3_vl/text.py:30-61).

The kernels take bf16 device values with frozen weights; everything else
(float32, trainable norm weights, autocast, function transforms, tracing,
other widths and layouts) runs the torch expressions, which also define the
values: both round to bf16 at the same places. The frozen weights are saved for
the backward as they are, so they do not change between a call and its backward.
"""

from __future__ import annotations

import torch
import torch.nn.functional as F

from . import _native as nat
from .ops import (BF16, F32, _aligned, _dtype_code, _on_device, _ptr, _stream, eager_calls,
                  on_current_device, plain_tensor)

_MAX_SIZE = 4096  # elements of a row that the kernels keep in registers


def rms_norm(value: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    """The torch expression of ``RMSNorm``."""

    v = value.float()
    v = v * torch.rsqrt(v.square().mean(-1, keepdim=True) + eps)
    return (v * weight.float()).to(value.dtype)


def layer_norm(value, weight, bias, eps: float) -> torch.Tensor:
    """The torch expression of ``LayerNorm``: reduced-precision layer_norm
    keeps float32 statistics and rounds the normalized, affine-transformed
    value once."""

    return F.layer_norm(value, value.shape[-1:], weight.to(value.dtype), bias.to(value.dtype), eps)


def _rotate_half(value: torch.Tensor) -> torch.Tensor:
    first, second = value.chunk(2, dim=-1)
    return torch.cat((-second, first), dim=-1)


def rotate(value: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
           dtype: torch.dtype | None = None) -> torch.Tensor:
    """The rotary rotation of ``[B, S, H, D]`` by ``[1, S, D]`` angles, in float32."""

    cos, sin = cos[:, :, None], sin[:, :, None]
    value, dtype = value.float(), dtype or value.dtype
    return (value * cos + _rotate_half(value) * sin).to(dtype)


# ---------------------------------------------------------------------------
# where the kernels apply
# ---------------------------------------------------------------------------
def _dense(t: torch.Tensor) -> bool:
    return t.is_contiguous() and t.data_ptr() % 16 == 0


def _frozen(size: int, device, *weights: torch.Tensor) -> bool:
    """Weights that the kernels take: dense float32 or bf16 rows of one
    dtype, none of which wants a gradient."""

    grad = torch.is_grad_enabled()
    return all(plain_tensor(w) and w.device == device and w.shape == (size,)
               and w.dtype in (F32, BF16) and w.dtype == weights[0].dtype and _dense(w)
               and not (grad and w.requires_grad) for w in weights)


def _rows_fit(value: torch.Tensor, *weights: torch.Tensor) -> bool:
    size = value.shape[-1] if value.dim() else 0
    return (plain_tensor(value) and on_current_device(value) and value.dtype == BF16
            and 8 <= size <= _MAX_SIZE and size % 8 == 0
            and 0 < value.numel() and value.numel() // size <= 1 << 31
            and _dense(value) and _frozen(size, value.device, *weights)
            and not torch.is_autocast_enabled("cuda"))


def _row_kernel(value: torch.Tensor, *weights: torch.Tensor) -> bool:
    return eager_calls() and _rows_fit(value, *weights)


def _unhooked(module: torch.nn.Module, cls: type) -> bool:
    """Calling ``module`` is calling ``cls.forward``: no subclass, hook or
    replaced forward would see (or miss) a fused call."""

    return (type(module) is cls and "forward" not in module.__dict__
            and not (module._forward_hooks or module._forward_pre_hooks or module._backward_hooks
                     or module._backward_pre_hooks)
            and not torch.nn.modules.module._has_any_global_hook())


# ---------------------------------------------------------------------------
# the fused calls
# ---------------------------------------------------------------------------
def _forward(x, residual, weight, bias, kind: int, eps: float, keep: bool = False):
    """``(t, norm(t))``, t = x + residual, or a copy of x with ``keep`` (else None)."""

    device = _on_device(x, residual, weight, bias)
    size = x.shape[-1]
    y = torch.empty_like(x)
    total = torch.empty_like(x) if keep or residual is not None else None
    nat.call("rpx_norm_forward", _ptr(x), _ptr(residual), _ptr(weight), _ptr(bias),
             _dtype_code(weight.dtype), x.numel() // size, size, float(eps), kind, _ptr(total),
             _ptr(y), _stream(device))
    return total, y


def _expression(kind: int, value, weight, bias, eps):
    if kind == nat.NORM_RMS:
        return rms_norm(value, weight, eps)
    return layer_norm(value, weight, bias, eps)


def _kernel_gradients(*grads) -> bool:
    """The backward kernels take these gradients. Not where the gradient is
    itself differentiated (create_graph), batched (is_grads_batched) or traced:
    there the expressions are differentiated instead."""

    return (not torch.is_grad_enabled() and eager_calls()
            and all(g is None or plain_tensor(g) for g in grads))


def _gradient(ctx, dy, d_total):
    """The gradient of the normalised row for the gradients of the norm and
    (or None) of the row's other use."""

    value, weight, bias = ctx.saved_tensors
    if dy is None:
        return d_total
    if not _kernel_gradients(dy, d_total):
        again = torch.is_grad_enabled()
        with torch.enable_grad():
            y = _expression(ctx.kind, value, weight, bias, ctx.eps)
        dx, = torch.autograd.grad(y, value, dy, create_graph=again)
        return dx if d_total is None else dx + d_total
    device = _on_device(value, dy)
    size = value.shape[-1]
    dy, d_total = _aligned(dy), _aligned(d_total)
    dx = torch.empty_like(value)
    nat.call("rpx_norm_backward", _ptr(dy), _ptr(d_total), _ptr(value), _ptr(weight),
             _dtype_code(weight.dtype), value.numel() // size, size, float(ctx.eps), ctx.kind,
             _ptr(dx), _stream(device))
    return dx


class NormFn(torch.autograd.Function):
    """A LayerNorm or RMSNorm with frozen weights."""

    @staticmethod
    def forward(ctx, x, weight, bias, kind, eps):
        ctx.set_materialize_grads(False)
        ctx.save_for_backward(x, weight, bias)
        ctx.kind, ctx.eps = kind, eps
        return _forward(x, None, weight, bias, kind, eps)[1]

    @staticmethod
    def backward(ctx, dy):
        return _gradient(ctx, dy, None), None, None, None, None


class AddNormFn(torch.autograd.Function):
    """``t = x + residual`` (or, without a residual, a copy of x) and its norm,
    with frozen weights: ``(t, norm(t))``. The backward reads t."""

    @staticmethod
    def forward(ctx, x, residual, weight, bias, kind, eps):
        ctx.set_materialize_grads(False)
        total, y = _forward(x, residual, weight, bias, kind, eps, keep=True)
        ctx.save_for_backward(total, weight, bias)
        ctx.kind, ctx.eps, ctx.added = kind, eps, residual is not None
        return total, y

    @staticmethod
    def backward(ctx, d_total, dy):
        dx = _gradient(ctx, dy, d_total)
        return dx, dx if ctx.added else None, None, None, None, None


class HeadNormFn(torch.autograd.Function):
    """A layer's queries, keys and values in one launch: per-head RMSNorm with
    a frozen weight and the rotary rotation (where there is a weight), each
    head repeated: ``[B, S, H, D] -> [B, S, H * repeat, D]``.

    Arguments: cos, sin, a tuple of (eps, repeat) per part, then per part x
    and its weight or None.
    """

    @staticmethod
    def forward(ctx, cos, sin, cfg, *operands):
        xs, weights = operands[::2], operands[1::2]
        b, s, _, d = xs[0].shape
        ctx.cfg = cfg
        # a part that is only repeated: its gradient does not depend on it
        kept = [t for x, w in zip(xs, weights) if w is not None for t in (x, w)]
        ctx.normed = [w is not None for w in weights]
        ctx.heads = [x.shape[2] for x in xs]
        ctx.save_for_backward(cos, sin, *kept)
        outs = [torch.empty((b, s, x.shape[2] * repeat, d), dtype=BF16, device=x.device)
                for x, (_, repeat) in zip(xs, cfg)]
        _head_norm(cos, sin, cfg, xs, weights, None, outs)
        return tuple(outs)

    @staticmethod
    def backward(ctx, *grads):
        cos, sin, *kept = ctx.saved_tensors
        saved = iter(kept)
        pairs = [(next(saved), next(saved)) if normed else (None, None) for normed in ctx.normed]
        if not _kernel_gradients(*grads):
            again = torch.is_grad_enabled()
            found = []
            for (x, w), g, heads, (eps, repeat) in zip(pairs, grads, ctx.heads, ctx.cfg):
                dx = None
                if w is None:
                    dx = g.reshape(*g.shape[:2], heads, repeat, g.shape[3]).sum(3)
                elif x.requires_grad:
                    with torch.enable_grad():
                        y = rotate(rms_norm(x, w, eps), cos, sin).repeat_interleave(repeat, dim=2)
                    dx, = torch.autograd.grad(y, x, g, create_graph=again)
                found += [dx, None]
            return (None, None, None, *found)
        grads = [g if g.stride(3) == 1 and not any(n % 8 for n in g.stride()[:3])
                 and g.data_ptr() % 16 == 0 else _aligned(g) for g in grads]
        outs = [torch.empty((*g.shape[:2], heads, g.shape[3]), dtype=BF16, device=g.device)
                for g, heads in zip(grads, ctx.heads)]
        # where there is no norm to go back through, no row is read
        xs = [dx if x is None else x for (x, _), dx in zip(pairs, outs)]
        _head_norm(cos, sin, ctx.cfg, xs, [w for _, w in pairs], grads, outs)
        return (None, None, None, *(t for dx in outs for t in (dx, None)))


def _head_norm(cos, sin, cfg, xs, weights, grads, outs) -> None:
    b, s, _, d = xs[0].shape
    if any(x.shape != (b, s, x.shape[2], d) for x in xs):
        raise ValueError(f"parts of one launch have the same tokens and head width, got "
                         f"{[tuple(x.shape) for x in xs]}")
    device = _on_device(cos, sin, *xs, *weights)
    parts = (nat.HeadPart * len(xs))()
    for i, (x, w, (eps, repeat)) in enumerate(zip(xs, weights, cfg)):
        part = parts[i]
        part.x, part.out = x.data_ptr(), outs[i].data_ptr()
        part.heads, part.repeat, part.eps = x.shape[2], repeat, eps
        if w is not None:
            part.weight, part.weight_dtype = w.data_ptr(), _dtype_code(w.dtype)
        if grads is not None:
            part.g = grads[i].data_ptr()
            part.stride_b, part.stride_s, part.stride_h, _ = grads[i].stride()
    nat.call("rpx_head_norm", parts, len(xs), _ptr(cos), _ptr(sin), b * s, s, d,
             int(grads is not None), _stream(device))


class LayerNorm(torch.nn.Module):
    """Last-axis LayerNorm with float32 statistics, output in the input dtype."""

    def __init__(self, size: int, eps: float, device=None) -> None:
        super().__init__()
        self.weight = torch.nn.Parameter(torch.ones(size, device=device))
        self.bias = torch.nn.Parameter(torch.zeros(size, device=device))
        self.eps = eps

    def forward(self, value: torch.Tensor) -> torch.Tensor:
        if _row_kernel(value, self.weight, self.bias):
            return NormFn.apply(value, self.weight, self.bias, nat.NORM_LAYER, self.eps)
        return layer_norm(value, self.weight, self.bias, self.eps)


class RMSNorm(torch.nn.Module):
    """Last-axis RMS normalisation with float32 statistics
    (src/representax/models/components.py:134-150)."""

    def __init__(self, size: int, eps: float, device=None) -> None:
        super().__init__()
        self.weight = torch.nn.Parameter(torch.ones(size, device=device))
        self.eps = eps

    def forward(self, value: torch.Tensor) -> torch.Tensor:
        if _row_kernel(value, self.weight):
            if torch.is_grad_enabled() and value.requires_grad:
                # the expression keeps a float32 copy, so its argument may
                # change in place before the backward: keep a copy here too
                return AddNormFn.apply(value, None, self.weight, None, nat.NORM_RMS, self.eps)[1]
            return NormFn.apply(value, self.weight, None, nat.NORM_RMS, self.eps)
        return rms_norm(value, self.weight, self.eps)


def add_norm(norm: torch.nn.Module, value: torch.Tensor, update: torch.Tensor):
    """``t = value + update`` and ``norm(t)``: ``(t, norm(t))``, in one pass
    where the kernels apply. The backward reads t: it must not change in place."""

    kind = {LayerNorm: nat.NORM_LAYER, RMSNorm: nat.NORM_RMS}.get(type(norm))
    if kind is not None and eager_calls() and _unhooked(norm, type(norm)):
        bias = norm.bias if kind == nat.NORM_LAYER else None
        weights = (norm.weight,) if bias is None else (norm.weight, bias)
        if (_rows_fit(value, *weights) and plain_tensor(update) and update.dtype == BF16
                and update.shape == value.shape and update.device == value.device
                and _dense(update)):
            return AddNormFn.apply(value, update, norm.weight, bias, kind, norm.eps)
    total = value + update
    return total, norm(total)


def attention_heads(query_norm: torch.nn.Module, key_norm: torch.nn.Module, q: torch.Tensor,
                    k: torch.Tensor, v: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                    dtype: torch.dtype):
    """The operands of grouped-query attention from ``[B, S, H, D]`` projections:
    queries and keys through their norms, rotated by ``[1, S, D]`` float32
    angles and rounded to ``dtype``, key and value heads repeated to the
    queries' count. One launch where the kernels apply; its backward reads q and
    k, which must not change in place."""

    b, s, h, d = q.shape
    repeat = h // k.shape[2]
    if (eager_calls() and _unhooked(query_norm, RMSNorm) and _unhooked(key_norm, RMSNorm)
            and d in (64, 128)
            and dtype == BF16 and h <= 65536 and repeat * k.shape[2] == h
            and k.shape == v.shape == (b, s, k.shape[2], d)  # the launch reads b * s tokens of each
            and _rows_fit(q, query_norm.weight) and _rows_fit(k, key_norm.weight)
            and plain_tensor(v) and v.dtype == BF16 and _dense(v)
            and k.device == q.device == v.device
            and all(plain_tensor(t) and t.dtype == F32 and t.device == q.device
                    and t.shape == (1, s, d) and _dense(t) and not t.requires_grad
                    for t in (cos, sin))):
        cfg = ((query_norm.eps, 1), (key_norm.eps, repeat))
        operands = (q, query_norm.weight, k, key_norm.weight)
        if repeat == 1:
            return (*HeadNormFn.apply(cos, sin, cfg, *operands), v)
        return HeadNormFn.apply(cos, sin, (*cfg, (0.0, repeat)), *operands, v, None)
    q, k = (rotate(norm(t), cos, sin, dtype) for norm, t in ((query_norm, q), (key_norm, k)))
    if repeat > 1:
        k, v = (t.repeat_interleave(repeat, dim=2) for t in (k, v))
    return q, k, v


__all__ = ["LayerNorm", "RMSNorm", "add_norm", "attention_heads"]
