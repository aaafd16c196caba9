"""Unified decoder-only transformer for the llama / falcon / opt families.

One implementation serves all model configs the reference's examples name:
llama2-7b/13b/70b (RMSNorm + RoPE + GQA + SwiGLU),
falcon-7b-instruct (LayerNorm + RoPE + MQA + parallel attn/MLP + GELU),
facebook/opt-125m (LayerNorm + learned positions + GELU).

Three execution paths:
  * forward_prefill — varlen packed prompt ingestion writing the paged KV cache
  * forward_decode  — one token per sequence over the paged KV cache (the serve
    hot loop; every op here is a hand-written HIP kernel on GPU)
  * forward_train   — dense differentiable forward (trainer; autograd +
    torch SDPA; loss/gradients via the fused cross-entropy kernel)

Tensor-parallel: heads are sharded column-parallel for QKV, row-parallel for
the output/down projections (2 RCCL all-reduces per layer).
"""

from __future__ import annotations

import math
from typing import Optional

import torch
import torch.nn as nn
import torch.nn.functional as F

from .. import ops
from ..ops import train as train_ops
from ..parallel.comm import state
from ..parallel.tp import (ColumnParallelLinear, Linear, RowParallelLinear,
                           bare)
from .config import ModelConfig


def _norm(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor],
          eps: float, rms: bool) -> torch.Tensor:
    if rms:
        return ops.rms_norm(x, weight, eps)
    return ops.layer_norm(x, weight, bias, eps)


def fused_norm_residual(deltas: tuple, h: torch.Tensor, norm: "NormParams",
                        eps: float) -> tuple[torch.Tensor, torch.Tensor]:
    """y = norm(h + deltas), h = h + deltas — fused so the hidden state makes
    one HBM round trip per norm (profiles/serve_decode_r01_baseline.txt:
    unfused residual adds were ~2.2 ms of a 10.3 ms decode step). RMSNorm of
    one delta works in place on h."""
    if isinstance(deltas, ops.Normed):
        return deltas.rows, h
    got = None
    if bare(norm, NormParams):
        if norm.rms and len(deltas) == 1:
            return ops.rms_norm_residual(deltas[0], h, norm.weight, eps)
        got = train_ops.fused_add_norm(h, deltas, norm.weight, norm.bias, eps)
    if got is None:
        for d in deltas:
            h = h + d
        got = norm(h, eps), h
    return got


# Products with what follows them in one kernel: by methods of the module's own
# class, since any module may stand where a projection was.

def normed_product(lin: nn.Module, deltas: tuple, h: torch.Tensor,
                   norm: "NormParams", eps: float, **how):
    """(lin of norm(h + deltas), h + deltas) in one kernel, or None."""
    normed = getattr(type(lin), "normed", None)
    if normed is None or len(deltas) != 1 or not bare(norm, NormParams) \
            or not norm.rms:
        return None
    return normed(lin, deltas[0], h, norm.weight, eps, **how)


def added_product(lin: nn.Module, x: torch.Tensor, h: torch.Tensor,
                  norm: Optional["NormParams"], eps: float) -> tuple:
    """(h + lin(x), what of norm's rows is there already), or h and what is
    still to be added to it."""
    if norm is not None and bare(norm, NormParams) and norm.rms:
        for name, more in ("added", ()), ("added_norm", (eps,)):
            how = getattr(type(lin), name, None)
            got = None if how is None else how(lin, x, h, norm.weight, *more)
            if got is not None:
                return got
    return h, (lin(x),)


def scaled_product(lin: nn.Module, deltas: tuple, h: torch.Tensor,
                   norm: "NormParams", eps: float, **how):
    """(lin of norm(h + deltas), h + deltas) in one kernel, or None, and what
    is still to be added to h."""
    if isinstance(deltas, ops.Normed):
        return None, deltas
    if not isinstance(deltas, ops.Undivided):
        return normed_product(lin, deltas, h, norm, eps, **how), deltas
    scaled = getattr(type(lin), "scaled", None)
    y = None if scaled is None else scaled(lin, deltas, eps, **how)
    return None if y is None else (y, h), ()


def heads_product(lin: nn.Module, y: torch.Tensor, cache: ops.Cache):
    """ops.rope_kv_append of lin(y) in one kernel, or None."""
    heads = getattr(type(lin), "heads", None)
    return None if heads is None else heads(lin, y, cache)


def gated_product(lin: nn.Module, y: torch.Tensor) -> torch.Tensor:
    """ops.silu_mul(lin(y))"""
    gated = getattr(type(lin), "gated", None)
    return ops.silu_mul(lin(y)) if gated is None else gated(lin, y)


def gelu_product(lin: nn.Module, y: torch.Tensor) -> torch.Tensor:
    """ops.gelu(lin(y))"""
    gelu = getattr(type(lin), "gelu", None)
    return ops.gelu(lin(y)) if gelu is None else gelu(lin, y)


class NormParams(nn.Module):
    def __init__(self, size: int, rms: bool, device=None, dtype=None):
        super().__init__()
        self.rms = rms
        self.weight = nn.Parameter(torch.ones(size, device=device, dtype=dtype))
        self.bias = None if rms else nn.Parameter(
            torch.zeros(size, device=device, dtype=dtype))

    def forward(self, x: torch.Tensor, eps: float) -> torch.Tensor:
        return _norm(x, self.weight, self.bias, eps, self.rms)


class Block(nn.Module):
    def __init__(self, cfg: ModelConfig, device=None, dtype=None):
        super().__init__()
        st = state()
        tp = st.tp_size
        self.cfg = cfg
        self.tp = tp
        assert cfg.num_heads % tp == 0, "num_heads must divide TP world size"
        self.n_heads = cfg.num_heads // tp
        # KV heads: shard when possible, replicate when fewer than TP ranks
        # (falcon MQA, llama2-70b GQA at high TP).
        if cfg.num_kv_heads >= tp:
            assert cfg.num_kv_heads % tp == 0
            self.n_kv_heads = cfg.num_kv_heads // tp
            self.kv_replicated = False
        else:
            self.n_kv_heads = 1
            self.kv_replicated = True
        d = cfg.head_dim
        rms = cfg.family == "llama"
        bias = cfg.family == "opt"
        eps = cfg.rms_norm_eps if rms else cfg.layer_norm_eps
        self.eps = eps
        self.norm1 = NormParams(cfg.hidden_size, rms, device, dtype)
        # Fused QKV, column-parallel by construction: this rank's slice is
        # (n_heads + 2*n_kv_heads) * head_dim output features.
        self.wqkv = Linear(cfg.hidden_size,
                           (self.n_heads + 2 * self.n_kv_heads) * d,
                           bias=bias, device=device, dtype=dtype)
        self.wo = RowParallelLinear(cfg.num_heads * d, cfg.hidden_size,
                                    bias=bias, device=device, dtype=dtype)
        self.parallel_attn = cfg.parallel_attn
        self.parallel_norms = cfg.parallel_norms
        # norm2 is the post-attention norm (sequential blocks) OR falcon-40b's
        # ln_mlp (parallel blocks with parallel_norms: norm1 = ln_attn feeds
        # attention, norm2 = ln_mlp feeds the MLP, both of the same residual)
        if not cfg.parallel_attn or cfg.parallel_norms:
            self.norm2 = NormParams(cfg.hidden_size, rms, device, dtype)
        if cfg.activation == "silu":
            self.w_gateup = ColumnParallelLinear(
                cfg.hidden_size, 2 * cfg.intermediate_size, bias=bias,
                device=device, dtype=dtype)
        else:
            self.w_up = ColumnParallelLinear(
                cfg.hidden_size, cfg.intermediate_size, bias=bias,
                device=device, dtype=dtype)
        self.w_down = RowParallelLinear(cfg.intermediate_size, cfg.hidden_size,
                                        bias=bias, device=device, dtype=dtype)
        self.scale = 1.0 / math.sqrt(d)
        self.rope_theta = cfg.rope_theta if cfg.family in ("llama", "falcon") else 0.0

    # -- shared pieces ------------------------------------------------------
    def _split_qkv(self, qkv: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
        d = self.cfg.head_dim
        n = qkv.shape[0]
        q, k, v = qkv.split([self.n_heads * d, self.n_kv_heads * d,
                             self.n_kv_heads * d], dim=-1)
        return (q.view(n, self.n_heads, d), k.view(n, self.n_kv_heads, d),
                v.view(n, self.n_kv_heads, d))

    def _mlp_up(self, y: torch.Tensor) -> torch.Tensor:
        if self.cfg.activation == "silu":
            return gated_product(self.w_gateup, y)
        return gelu_product(self.w_up, y)

    def _mlp(self, y: torch.Tensor) -> torch.Tensor:
        return self.w_down(self._mlp_up(y))

    # -- decode -------------------------------------------------------------
    def decode_ops(self, h: torch.Tensor, deltas: tuple,
                   positions: torch.Tensor,
                   k_cache: torch.Tensor, v_cache: torch.Tensor,
                   slots: torch.Tensor, block_table: torch.Tensor,
                   seq_lens: torch.Tensor,
                   after: Optional[NormParams] = None):
        """Generator form of the decode block: yields after each op group
        (norm + qkv GEMM | rope+attention | o GEMM | up GEMM | down GEMM) so
        the dual-stream runner (serve/graph_runner.py) can interleave two
        half-batches op-by-op — the trailing half's GEMMs re-read weights
        the leading half just streamed (LLC-hot) while its attention
        overlaps the leader's compute. forward_decode drives this
        generator to completion, so single-stream numerics are by
        construction identical.

        h: the residual stream, deltas: what is still to be added to it, which
        this block's first norm does, or ops.Undivided or ops.Normed, what is
        there of that norm already; the same is returned, of the norm after."""
        cache = ops.Cache(positions, k_cache, v_cache, slots, self.rope_theta)
        got = None
        if not self.parallel_attn:
            got, deltas = scaled_product(self.wqkv, deltas, h, self.norm1,
                                         self.eps, cache=cache)
        if got is not None:
            q, h = got
        else:
            y, h = fused_norm_residual(deltas, h, self.norm1, self.eps)
            q = heads_product(self.wqkv, y, cache)
            qkv = self.wqkv(y) if q is None else None
        yield
        if q is None:
            q, k, v = self._split_qkv(qkv)
            q = ops.rope_kv_append(q, k, v, *cache)
        a = ops.paged_attn_decode(q, k_cache, v_cache, block_table, seq_lens,
                                  self.scale)
        yield
        a = a.reshape(a.shape[0], -1)
        if self.parallel_attn:
            attn_out = self.wo(a)
            yield
            if self.parallel_norms:
                y = self.norm2(h, self.eps)
            up = self._mlp_up(y)
            yield
            return h, (attn_out, self.w_down(up))
        silu = self.cfg.activation == "silu"
        h, deltas = added_product(self.wo, a, h,
                                  self.norm2 if silu else None, self.eps)
        yield
        got = None
        if silu:
            got, deltas = scaled_product(self.w_gateup, deltas, h, self.norm2,
                                         self.eps, gated=True)
        if got is not None:
            up, h = got
        else:
            y, h = fused_norm_residual(deltas, h, self.norm2, self.eps)
            up = self._mlp_up(y)
        yield
        return added_product(self.w_down, up, h, after, self.eps)

    # -- prefill ------------------------------------------------------------
    def forward_prefill(self, h: torch.Tensor, deltas: tuple,
                        positions: torch.Tensor, seq_start: torch.Tensor,
                        k_cache: torch.Tensor, v_cache: torch.Tensor,
                        slots: torch.Tensor,
                        max_len: Optional[int]) -> tuple:
        """(h, deltas): the residual stream and what is still to be added to
        it, which the next norm does; the same is returned."""
        y, h = fused_norm_residual(deltas, h, self.norm1, self.eps)
        q, k, v = ops.rope_split_append(
            self.wqkv(y), self.n_heads, self.n_kv_heads,
            ops.Cache(positions, k_cache, v_cache, slots, self.rope_theta))
        a = ops.attn_prefill(q, k, v, seq_start, self.scale, max_len)
        attn_out = self.wo(a.reshape(a.shape[0], -1))
        if self.parallel_attn:
            if self.parallel_norms:
                y = self.norm2(h, self.eps)
            return h, (attn_out, self._mlp(y))
        y, h = fused_norm_residual((attn_out,), h, self.norm2, self.eps)
        return h, (self._mlp(y),)

    # -- train (dense, differentiable) --------------------------------------
    def forward_train(self, h: torch.Tensor, deltas: tuple,
                      cos: Optional[torch.Tensor],
                      sin: Optional[torch.Tensor]) -> tuple:
        """(h, deltas): the residual stream and what is still to be added to
        it, which the next norm does; the same is returned."""
        y, h = train_ops.add_norm(h, deltas, self.norm1.weight,
                                  self.norm1.bias, self.eps)
        if self.rope_theta <= 0:
            cos = sin = None
        attn_out = self.wo(train_ops.attend(
            self.wqkv(y), cos, sin, self.n_heads, self.n_kv_heads,
            self.scale))
        if self.parallel_attn:
            if self.parallel_norms:
                y, _ = train_ops.add_norm(h, (), self.norm2.weight,
                                          self.norm2.bias, self.eps)
            return h, (attn_out, self._mlp_train(y))
        y, h = train_ops.add_norm(h, (attn_out,), self.norm2.weight,
                                  self.norm2.bias, self.eps)
        return h, (self._mlp_train(y),)

    def whole_train(self, h: torch.Tensor, cos: Optional[torch.Tensor],
                    sin: Optional[torch.Tensor]) -> torch.Tensor:
        """forward_train with its additions done, so that one tensor is kept
        between recomputed blocks."""
        h, deltas = self.forward_train(h, (), cos, sin)
        for d in deltas:
            h = h + d
        return h

    def _mlp_train(self, y: torch.Tensor) -> torch.Tensor:
        if self.cfg.activation == "silu":
            return self.w_down(train_ops.silu_mul(self.w_gateup(y)))
        return self.w_down(F.gelu(self.w_up(y), approximate="tanh"))


class CausalLM(nn.Module):
    def __init__(self, cfg: ModelConfig, device=None, dtype=torch.bfloat16):
        super().__init__()
        if cfg.layers:
            raise ValueError(f"{cfg.name}: models of unlike layers are built "
                             "by models.build_model, and served only")
        self.cfg = cfg
        st = state()
        self.embed_tokens = nn.Embedding(cfg.vocab_size, cfg.hidden_size,
                                         device=device, dtype=dtype)
        if cfg.learned_pos_emb:
            self.embed_positions = nn.Embedding(
                cfg.max_position_embeddings, cfg.hidden_size, device=device,
                dtype=dtype)
        self.blocks = nn.ModuleList(
            Block(cfg, device=device, dtype=dtype) for _ in range(cfg.num_layers))
        rms = cfg.family == "llama"
        self.eps = cfg.rms_norm_eps if rms else cfg.layer_norm_eps
        self.final_norm = NormParams(cfg.hidden_size, rms, device, dtype)
        if cfg.tie_word_embeddings:
            self.lm_head = None
        else:
            self.lm_head = Linear(cfg.hidden_size, cfg.vocab_size, bias=False,
                                  device=device, dtype=dtype)
        self.n_kv_heads = self.blocks[0].n_kv_heads  # per-rank
        self.gradient_checkpointing = False

    def _logits(self, y: torch.Tensor) -> torch.Tensor:
        if self.lm_head is None:
            return ops.linear(y, self.embed_tokens.weight)
        return self.lm_head(y)  # module call: works for Linear AND QuantLinear

    @torch.no_grad()
    def init_random(self, seed: int = 0) -> None:
        """Initialize EVERY parameter (models are built on meta + to_empty,
        so nothing may be left untouched): matrices ~ N(0, 0.02), norm
        weights = 1, biases = 0."""
        dev = next(self.parameters()).device
        g = torch.Generator(device=dev).manual_seed(seed)
        for name, p in self.named_parameters():
            if p.dim() >= 2:
                p.normal_(0.0, 0.02, generator=g)
            elif name.endswith("bias"):
                p.zero_()
            else:  # norm weights
                p.fill_(1.0)

    # -- decode --------------------------------------------------------------
    def decode_ops(self, tokens: torch.Tensor, positions: torch.Tensor,
                   kv_caches: list[tuple[torch.Tensor, torch.Tensor]],
                   slots: torch.Tensor, block_table: torch.Tensor,
                   seq_lens: torch.Tensor):
        """Whole-model decode as an op-group generator (see
        TransformerBlock.decode_ops); returns the logits."""
        h = self.embed_tokens(tokens)
        if self.cfg.learned_pos_emb:
            h = h + self.embed_positions(positions.long())
        # each block's outputs are added to the residual stream inside the
        # NEXT norm
        deltas = ()
        for blk, after, (kc, vc) in zip(self.blocks, self._norms_after(),
                                        kv_caches):
            h, deltas = yield from blk.decode_ops(h, deltas, positions, kc,
                                                  vc, slots, block_table,
                                                  seq_lens, *after)
            yield
        if self.lm_head is not None:
            got, deltas = scaled_product(self.lm_head, deltas, h,
                                         self.final_norm, self.eps)
            if got is not None:
                return got[0]
        elif isinstance(deltas, ops.Undivided):
            deltas = ()
        y, _ = fused_norm_residual(deltas, h, self.final_norm, self.eps)
        return self._logits(y)

    def _norms_after(self) -> list[tuple]:
        """For every block (the norm after it,), which its last product may
        begin, or () where that block or the next one has a decode_ops of its
        own, which knows nothing of it, or an eps of its own."""
        def knows(blk):
            return (blk is self or isinstance(blk, Block)
                    and type(blk).decode_ops is Block.decode_ops
                    and "decode_ops" not in blk.__dict__
                    and not blk.parallel_attn)
        blocks = [*self.blocks, self]
        return [(nxt.final_norm if nxt is self else nxt.norm1,)
                if knows(blk) and knows(nxt) and blk.eps == nxt.eps else ()
                for blk, nxt in zip(blocks, blocks[1:])]

    def forward_decode(self, tokens: torch.Tensor, positions: torch.Tensor,
                       kv_caches: list[tuple[torch.Tensor, torch.Tensor]],
                       slots: torch.Tensor, block_table: torch.Tensor,
                       seq_lens: torch.Tensor) -> torch.Tensor:
        gen = self.decode_ops(tokens, positions, kv_caches, slots,
                              block_table, seq_lens)
        while True:
            try:
                next(gen)
            except StopIteration as e:
                return e.value

    # -- prefill -------------------------------------------------------------
    def forward_prefill(self, tokens: torch.Tensor, positions: torch.Tensor,
                        seq_start: torch.Tensor,
                        kv_caches: list[tuple[torch.Tensor, torch.Tensor]],
                        slots: torch.Tensor) -> torch.Tensor:
        """Returns logits for the LAST token of each sequence: [num_seqs, V]."""
        h = self.embed_tokens(tokens)
        if self.cfg.learned_pos_emb:
            h = h + self.embed_positions(positions.long())
        elif not bare(self.embed_tokens, nn.Embedding):
            h = h.clone()       # added to in place, and a hook may keep it
        max_len = ops.longest(seq_start) if h.is_cuda else None
        deltas = ()
        for blk, (kc, vc) in zip(self.blocks, kv_caches):
            h, deltas = blk.forward_prefill(h, deltas, positions, seq_start,
                                            kc, vc, slots, max_len)
        last = (seq_start[1:] - 1).long()
        y, _ = fused_norm_residual(tuple(d[last] for d in deltas), h[last],
                                   self.final_norm, self.eps)
        return self._logits(y)

    # -- train ---------------------------------------------------------------
    def forward_train(self, tokens: torch.Tensor) -> torch.Tensor:
        """tokens: [B, S] -> logits [B, S, V], differentiable."""
        b, s = tokens.shape
        h = train_ops.lookup(tokens, self.embed_tokens)
        pos = torch.arange(s, device=tokens.device)
        if self.cfg.learned_pos_emb:
            h = h + self.embed_positions(pos)
        if self.cfg.family in ("llama", "falcon"):
            from ..ops.ref import rope_cos_sin
            cos, sin = rope_cos_sin(pos, self.cfg.head_dim, self.cfg.rope_theta)
            cos, sin = cos.to(h.device), sin.to(h.device)
        else:
            cos = sin = None
        deltas = ()
        recompute = self.gradient_checkpointing and torch.is_grad_enabled()
        for blk in self.blocks:
            if recompute:       # what a block left is a part of the one tensor
                for d in deltas:
                    h = h + d
                deltas = ()
            if recompute and h.requires_grad:
                h = torch.utils.checkpoint.checkpoint(
                    blk.whole_train, h, cos, sin, use_reentrant=False)
            else:
                h, deltas = blk.forward_train(h, deltas, cos, sin)
        y, _ = train_ops.add_norm(h, deltas, self.final_norm.weight,
                                  self.final_norm.bias, self.eps)
        return self._logits(y)
