"""The row work of a training step: residual additions with the norm that
follows, attention from the fused projection on, the gated activation.

Each op has a general form in torch's own ops, which every device, type and
transform gets, and a form on train_rows.hip's kernels for what a bf16 step on
the GPU calls. Both give gradients that can be differentiated again: where a
graph of the gradients is asked for, or a transform runs, the backward is the
general form's.
"""

from __future__ import annotations

from typing import Callable, Optional, Sequence

import torch
import torch.nn.functional as F

from . import _flash_bwd, _flash_fwd, _load_ext, flash_attn_train, \
    flash_attn_train_available, plain_tensors


def _again(form: Callable, inputs: Sequence, dy: torch.Tensor) -> list:
    """Gradients of form(*inputs) as a part of the graph."""
    with torch.enable_grad():
        # gradients are taken at places of their own: an input may also have
        # led to another one
        at = [t if t is None else t.view_as(t) for t in inputs]
        wanted = [t for t in at if t is not None and t.requires_grad]
        got = iter(torch.autograd.grad(form(*at), wanted, dy,
                                       create_graph=True))
        return [next(got) if t is not None and t.requires_grad else None
                for t in at]


def _values_only(*grads: Optional[torch.Tensor]) -> bool:
    """Whether a backward may take its kernels for these."""
    return not torch.is_grad_enabled() and plain_tensors(*grads)


def _whole(*tensors: Optional[torch.Tensor]) -> bool:
    """Contiguous bf16 on one GPU and 16-byte boundaries, as the kernels read
    them."""
    given = [t for t in tensors if t is not None]
    return all(t.is_cuda and t.device == given[0].device
               and t.dtype == torch.bfloat16 and t.is_contiguous()
               and t.numel() > 0 and t.data_ptr() % 16 == 0 for t in given)


# -------------------------------------------------------------------- lookup

class _Lookup(torch.autograd.Function):
    @staticmethod
    def forward(ctx, tokens, weight):
        tokens = tokens.contiguous()
        ctx.save_for_backward(tokens, weight)
        return F.embedding(tokens, weight)

    @staticmethod
    def backward(ctx, dy):
        tokens, weight = ctx.saved_tensors
        if not _values_only(dy):
            return None, _again(lambda w: F.embedding(tokens, w), (weight,),
                                dy)[0]
        dw = torch.zeros_like(weight)
        _load_ext().lookup_bwd(dw, _aligned(dy), tokens)
        return None, dw


def lookup(tokens: torch.Tensor, table: torch.nn.Embedding) -> torch.Tensor:
    """table(tokens). Up to 8192 of them on the GPU get their gradients from a
    kernel of their own."""
    w = table.weight
    if (type(table) is torch.nn.Embedding and table.padding_idx is None
            and table.max_norm is None and not table.sparse
            and not table.scale_grad_by_freq
            and not torch.nn.modules.module._has_any_global_hook()
            and not any((table._forward_hooks, table._forward_pre_hooks,
                         table._backward_hooks, table._backward_pre_hooks))
            and w.requires_grad and torch.is_grad_enabled() and _whole(w)
            and tokens.dtype == torch.int64 and tokens.device == w.device
            and 0 < tokens.numel() <= 8192
            and plain_tensors(tokens, w) and _load_ext() is not None
            and _load_ext().train_norm_takes(w.shape[1])):
        return _Lookup.apply(tokens, w)
    return table(tokens)


# --------------------------------------------------------------------- norms

def _add(h: torch.Tensor, deltas: Sequence[torch.Tensor]) -> torch.Tensor:
    for d in deltas:
        h = h + d
    return h


def _norm(h: torch.Tensor, weight: torch.Tensor,
          bias: Optional[torch.Tensor], eps: float) -> torch.Tensor:
    if bias is None:
        y = F.rms_norm(h.float(), weight.shape, weight.float(), eps)
    else:
        y = F.layer_norm(h.float(), weight.shape, weight.float(),
                         bias.float(), eps)
    return y.to(h.dtype)


class _AddNorm(torch.autograd.Function):
    """norm(h + deltas), and the sum where there are deltas."""

    @staticmethod
    def forward(ctx, eps, weight, bias, h, *deltas):
        ctx.set_materialize_grads(False)
        y = torch.empty_like(h)
        stats = torch.empty(h.numel() // h.shape[-1], 2, dtype=torch.float32,
                            device=h.device)
        d1, d2 = (*deltas, None, None)[:2]
        total = None if d1 is None else torch.empty_like(h)
        _load_ext().add_norm_fwd(y, total, stats, h, d1, d2, weight, bias,
                                 eps)
        ctx.eps, ctx.n = eps, len(deltas)
        ctx.save_for_backward(h if total is None else total, stats, weight,
                              bias)
        return y if total is None else (y, total)

    @staticmethod
    def backward(ctx, dy, dsum=None):
        x, stats, weight, bias = ctx.saved_tensors
        if dy is None:
            return None, None, None, *[dsum] * (1 + ctx.n)
        if not _values_only(dy, dsum):
            dw, db, dh = _again(
                lambda w, b, x: _norm(x, w, b, ctx.eps), (weight, bias, x),
                dy)
            if dsum is not None:
                dh = dsum if dh is None else dh + dsum
            return None, dw, db, *[dh] * (1 + ctx.n)
        dy = _aligned(dy)
        dsum = None if dsum is None else _aligned(dsum)
        dh, dw = torch.empty_like(x), torch.empty_like(weight)
        db = None if bias is None else torch.empty_like(bias)
        _load_ext().add_norm_bwd(dh, dw, db, dy, dsum, x, stats, weight)
        return None, dw, db, *[dh] * (1 + ctx.n)


def _aligned(t: torch.Tensor) -> torch.Tensor:
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def fused_add_norm(h: torch.Tensor, deltas: Sequence[torch.Tensor],
                   weight: torch.Tensor, bias: Optional[torch.Tensor],
                   eps: float) -> Optional[tuple]:
    """add_norm where train_rows.hip takes it, or None."""
    if (len(deltas) <= 2 and _whole(h, weight, bias, *deltas)
            and h.shape[-1:] == weight.shape
            and (bias is None or bias.shape == weight.shape)
            and all(d.shape == h.shape for d in deltas)
            and plain_tensors(h, weight, bias, *deltas)
            and _load_ext() is not None
            and _load_ext().train_norm_takes(weight.numel())):
        out = _AddNorm.apply(eps, weight, bias, h, *deltas)
        return out if deltas else (out, h)
    return None


def add_norm(h: torch.Tensor, deltas: Sequence[torch.Tensor],
             weight: torch.Tensor, bias: Optional[torch.Tensor],
             eps: float) -> tuple[torch.Tensor, torch.Tensor]:
    """(norm(h + deltas), h + deltas): LayerNorm, without bias RMSNorm, over
    the last dimension, in 32 bits."""
    got = fused_add_norm(h, deltas, weight, bias, eps)
    if got is None:
        h = _add(h, deltas)
        got = _norm(h, weight, bias, eps), h
    return got


# ----------------------------------------------------------------- attention

def rope(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
         bshd: bool = False) -> torch.Tensor:
    """x: [B, H, S, D] (or [B, S, H, D] when bshd); cos/sin: [S, D/2]."""
    d = x.shape[-1]
    x1, x2 = x[..., : d // 2], x[..., d // 2:]
    if bshd:
        c = cos[None, :, None, :]
        s = sin[None, :, None, :]
    else:
        c = cos[None, None, :, :]
        s = sin[None, None, :, :]
    return torch.cat([x1 * c - x2 * s, x2 * c + x1 * s], dim=-1).to(x.dtype)


def _attend(qkv, cos, sin, hq: int, hkv: int, scale: float) -> torch.Tensor:
    b, s, width = qkv.shape
    d = width // (hq + 2 * hkv)
    q, k, v = qkv.split([hq * d, hkv * d, hkv * d], dim=-1)
    if (qkv.is_cuda and qkv.dtype == torch.bfloat16
            and flash_attn_train_available(d)):
        # BSHD layout end-to-end — no transposes, no GQA head materialization
        q, k, v = (t.view(b, s, -1, d) for t in (q, k, v))
        if cos is not None:
            q, k = rope(q, cos, sin, bshd=True), rope(k, cos, sin, bshd=True)
        return flash_attn_train(q, k, v, scale).reshape(b, s, hq * d)
    q, k, v = (t.view(b, s, -1, d).transpose(1, 2) for t in (q, k, v))
    if cos is not None:
        q, k = rope(q, cos, sin), rope(k, cos, sin)
    if hkv != hq:
        k, v = (t.repeat_interleave(hq // hkv, dim=1) for t in (k, v))
    a = F.scaled_dot_product_attention(q, k, v, is_causal=True)
    return a.transpose(1, 2).reshape(b, s, hq * d)


def _attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, s: int,
               scale: float) -> torch.Tensor:
    """Causal attention of sequences of s rows, rows of heads to rows of
    heads, in 32-bit steps that can be differentiated any number of times."""
    hq, d = q.shape[1:]
    q32, k32, v32 = (
        t.view(-1, s, *t.shape[1:]).transpose(1, 2).float()
        .repeat_interleave(hq // t.shape[1], dim=1) for t in (q, k, v))
    scores = q32 @ k32.transpose(2, 3).contiguous() * scale
    later = torch.ones(s, s, dtype=torch.bool, device=q.device).triu(1)
    a = scores.masked_fill(later, -torch.inf).softmax(-1) @ v32
    return a.transpose(1, 2).reshape(-1, hq, d).to(q.dtype)


def attention_again(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                    dout: torch.Tensor, s: int, scale: float) -> list:
    """Gradients of attention as a part of the graph."""
    return _again(lambda *t: _attention(*t, s, scale), (q, k, v),
                  dout.reshape(q.shape))


class _Attend(torch.autograd.Function):
    """From rows of a fused projection to rows of heads: split and rotation in
    one kernel either way around the attention's own. Split rows are outputs as
    well, which nobody else sees: so they are kept as a part of the graph."""

    @staticmethod
    def forward(ctx, qkv, cos, sin, hq, hkv, scale):
        ctx.set_materialize_grads(False)
        b, s, width = qkv.shape
        d = width // (hq + 2 * hkv)
        q = qkv.new_empty(b * s, hq, d)
        k, v = (qkv.new_empty(b * s, hkv, d) for _ in range(2))
        _load_ext().rope_split(q, k, v, qkv, cos, sin, s)
        seq_start = torch.arange(0, (b + 1) * s, s, dtype=torch.int32,
                                 device=qkv.device)
        out, lse = _flash_fwd(q, k, v, seq_start, s, scale)
        ctx.save_for_backward(q, k, v, out, lse, seq_start, cos, sin)
        ctx.scale, ctx.shape = scale, qkv.shape
        return out.view(b, s, hq * d), q, k, v

    @staticmethod
    def backward(ctx, dout, *dsplit):
        q, k, v, out, lse, seq_start, cos, sin = ctx.saved_tensors
        b, s, width = ctx.shape
        if dout is not None and _values_only(dout) and not any(
                t is not None for t in dsplit):
            dq, dk, dv = _flash_bwd(q, k, v, out, _aligned(dout).view_as(out),
                                    lse, seq_start, s, ctx.scale)
            dqkv = q.new_empty(ctx.shape)
            _load_ext().rope_join(dqkv, dq, dk, dv, cos, sin, s)
            return dqkv, None, None, None, None, None
        parts = [torch.zeros_like(t) for t in (q, k, v)] if dout is None \
            else attention_again(q, k, v, dout, s, ctx.scale)
        parts = [(t if g is None else t + g).view(b, s, -1, q.shape[2])
                 for t, g in zip(parts, dsplit)]
        if cos is not None:         # turned back
            parts[:2] = (rope(t, cos, -sin, bshd=True) for t in parts[:2])
        return torch.cat([t.reshape(b, s, -1) for t in parts], -1), \
            None, None, None, None, None


def _angles(t: Optional[torch.Tensor], s: int, d: int,
            device: torch.device) -> bool:
    return t is None or (t.device == device and t.dtype == torch.float32
                         and t.shape == (s, d // 2) and t.is_contiguous()
                         and t.data_ptr() % 16 == 0 and not t.requires_grad)


def attend(qkv: torch.Tensor, cos: Optional[torch.Tensor],
           sin: Optional[torch.Tensor], hq: int, hkv: int,
           scale: float) -> torch.Tensor:
    """Causal attention of every sequence: qkv [B, S, (hq + 2 hkv) D], angles
    [S, D/2] or None -> [B, S, hq D]."""
    d = qkv.shape[-1] // (hq + 2 * hkv)
    if (qkv.dim() == 3 and qkv.shape[2] == (hq + 2 * hkv) * d and _whole(qkv)
            and all(_angles(t, qkv.shape[1], d, qkv.device)
                    for t in (cos, sin))
            and plain_tensors(qkv, cos, sin)
            and flash_attn_train_available(d)):
        return _Attend.apply(qkv, cos, sin, hq, hkv, scale)[0]
    return _attend(qkv, cos, sin, hq, hkv, scale)


# ---------------------------------------------------------------- activation

def _silu_mul(gu: torch.Tensor) -> torch.Tensor:
    g, u = gu.chunk(2, dim=-1)
    return F.silu(g) * u


class _SiluMul(torch.autograd.Function):
    @staticmethod
    def forward(ctx, gu):
        out = gu.new_empty(*gu.shape[:-1], gu.shape[-1] // 2)
        _load_ext().silu_mul(out, gu)
        ctx.save_for_backward(gu)
        return out

    @staticmethod
    def backward(ctx, dy):
        gu, = ctx.saved_tensors
        if not _values_only(dy):
            return _again(_silu_mul, (gu,), dy)[0]
        dx = torch.empty_like(gu)
        _load_ext().silu_mul_bwd(dx, _aligned(dy), gu)
        return dx


def silu_mul(gu: torch.Tensor) -> torch.Tensor:
    """silu(first half) * second half of the last dimension."""
    if (_whole(gu) and gu.shape[-1] % 16 == 0 and plain_tensors(gu)
            and _load_ext() is not None):
        return _SiluMul.apply(gu)
    return _silu_mul(gu)
