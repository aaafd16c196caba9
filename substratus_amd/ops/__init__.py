"""Op dispatch: hand-written CDNA4 HIP kernels on GPU, reference PyTorch on CPU.

Policy (task contract): on a ROCm GPU the HIP extension is MANDATORY — if a
tensor lives on a CUDA/HIP device and `substratus_amd._C` is not importable the
op raises instead of silently falling back to eager PyTorch. CPU tensors run
the fp32 reference implementations (substratus_amd/ops/ref.py), which are also
the parity oracle for the GPU tests.
"""

from __future__ import annotations

import os
from typing import NamedTuple, Optional

import torch
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from . import ref

_EXT = None
_EXT_ERR: Optional[str] = None


def _load_ext():
    global _EXT, _EXT_ERR
    if _EXT is not None or _EXT_ERR is not None:
        return _EXT
    try:
        from substratus_amd import _C  # built in-tree by setup.py build_ext --inplace
        _EXT = _C
    except ImportError as e:  # pragma: no cover - exercised only without the .so
        _EXT_ERR = str(e)
    return _EXT


def have_ext() -> bool:
    return _load_ext() is not None


def _dispatch(t: torch.Tensor):
    """Return the extension for GPU tensors (raising loudly if absent), None for CPU."""
    if t.is_cuda:
        ext = _load_ext()
        if ext is None:
            raise RuntimeError(
                "substratus_amd HIP extension (substratus_amd/_C*.so) is not built "
                f"but a GPU tensor was passed — no eager fallback on GPU. Build it "
                f"with `python setup.py build_ext --inplace` (PYTORCH_ROCM_ARCH=gfx950). "
                f"Import error: {_EXT_ERR}")
        return ext
    return None


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    ext = _dispatch(x)
    if ext is None:
        return ref.rms_norm(x, weight, eps)
    out = torch.empty_like(x)
    ext.rms_norm(out, x.contiguous(), weight, eps)
    return out


def rms_norm_residual(x: torch.Tensor, residual: torch.Tensor,
                      weight: torch.Tensor, eps: float) -> tuple[torch.Tensor, torch.Tensor]:
    """Fused: residual += x; y = rms_norm(residual). Returns (y, residual).

    The producing kernel fuses the residual add so the hidden state is read
    once from HBM (guide: fuse elementwise work into the producing kernel).
    """
    ext = _dispatch(x)
    if ext is None:
        residual = residual + x
        return ref.rms_norm(residual, weight, eps), residual
    y = torch.empty_like(x)
    ext.rms_norm_residual(y, residual, x.contiguous(), weight, eps)
    return y, residual


def layer_norm(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor,
               eps: float) -> torch.Tensor:
    ext = _dispatch(x)
    if ext is None:
        return ref.layer_norm(x, weight, bias, eps)
    out = torch.empty_like(x)
    ext.layer_norm(out, x.contiguous(), weight, bias, eps)
    return out


def _rows_contiguous(t: torch.Tensor) -> bool:
    """[n, h, d] with contiguous inner rows; the leading (token) stride may
    be larger — a qkv-split view."""
    return t.stride(2) == 1 and t.stride(1) == t.shape[2]


def rope_kv_append(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                   positions: torch.Tensor, k_cache: torch.Tensor,
                   v_cache: torch.Tensor, slots: torch.Tensor,
                   theta: float) -> torch.Tensor:
    ext = _dispatch(q)
    if ext is None:
        return ref.rope_kv_append(q, k, v, positions, k_cache, v_cache, slots, theta)
    # The kernel takes a token-row stride, so qkv-split VIEWS flow straight
    # through (decode saves three elementwise copies per layer; rotation
    # lands in-place inside the fused qkv buffer, which nothing re-reads).
    # Only reshape if the inner [h, d] rows themselves aren't contiguous.
    if not _rows_contiguous(q):
        q = q.contiguous()
    if not _rows_contiguous(k):
        k = k.contiguous()
    if not _rows_contiguous(v):
        v = v.contiguous()
    ext.rope_kv_append(q, k, v, positions, k_cache, v_cache, slots, theta)
    return q


def paged_attn_decode(q: torch.Tensor, k_cache: torch.Tensor,
                      v_cache: torch.Tensor, block_table: torch.Tensor,
                      seq_lens: torch.Tensor, scale: float) -> torch.Tensor:
    ext = _dispatch(q)
    if ext is None:
        return ref.paged_attn_decode(q, k_cache, v_cache, block_table, seq_lens, scale)
    if not _rows_contiguous(q):
        q = q.contiguous()
    out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
    ext.paged_attn_decode(out, q, k_cache, v_cache,
                          block_table, seq_lens, scale)
    return out


def longest(seq_start: torch.Tensor) -> int:
    return int((seq_start[1:] - seq_start[:-1]).max())


def attn_prefill(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                 seq_start: torch.Tensor, scale: float,
                 max_len: Optional[int] = None) -> torch.Tensor:
    """max_len: of the sequences, where the caller knows it; the host waits
    for it otherwise."""
    ext = _dispatch(q)
    if ext is None:
        return ref.attn_prefill(q, k, v, seq_start, scale)
    out = torch.empty_like(q)
    if max_len is None:
        max_len = longest(seq_start)
    if os.environ.get("SUB_ATTN_V5", "1") != "0":
        # scores transposed, softmax in registers: two to three times as fast
        # as the older kernel (scripts/microbench.py --which attnv5)
        ext.attn_v5(out, q.contiguous(), k.contiguous(), v.contiguous(),
                    seq_start, max_len, scale, None)
        return out
    ext.attn_prefill(out, q.contiguous(), k.contiguous(), v.contiguous(),
                     seq_start, max_len, scale)
    return out


def _flash_fwd(q, k, v, seq_start, max_len, scale):
    """(out, log-sums) of training attention; q, k, v contiguous."""
    ext = _dispatch(q)
    assert ext is not None, "flash_attn_train needs the HIP extension"
    out = torch.empty_like(q)
    lse = torch.empty(q.shape[0], q.shape[1], dtype=torch.float32,
                      device=q.device)
    if os.environ.get("SUB_ATTN_V5", "1") != "0":
        ext.attn_v5(out, q, k, v, seq_start, max_len, scale, lse)
    else:
        ext.attn_train_fwd(out, lse, q, k, v, seq_start, max_len, scale)
    return out, lse


def _flash_bwd(q, k, v, out, dout, lse, seq_start, max_len, scale):
    """(dq, dk, dv), the latter two 32-bit sums."""
    ext = _dispatch(q)
    dq = torch.empty_like(q)
    # f32 accumulators: under GQA every q head of a group atomically
    # adds its dK/dV contribution (attention_bwd.hip dkv kernel)
    dk32 = torch.zeros(k.shape, dtype=torch.float32, device=k.device)
    dv32 = torch.zeros(v.shape, dtype=torch.float32, device=v.device)
    delta = torch.empty_like(lse)
    ext.attn_train_bwd(dq, dk32, dv32, q, k, v, out, dout, lse, delta,
                       seq_start, max_len, scale)
    return dq, dk32, dv32


class _FlashAttnTrain(torch.autograd.Function):
    """Training attention on the first-party MFMA kernels: varlen causal
    forward (attention_prefill.hip, LSE saved) + FA2-style backward
    (attention_bwd.hip). GQA native — K/V stay at n_kv_heads; no
    repeat_interleave materialization."""

    @staticmethod
    def forward(ctx, q, k, v, seq_start, max_len, scale):
        q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
        out, lse = _flash_fwd(q, k, v, seq_start, max_len, scale)
        ctx.save_for_backward(q, k, v, out, lse, seq_start)
        ctx.max_len = max_len
        ctx.scale = scale
        return out

    @staticmethod
    def backward(ctx, dout):
        q, k, v, out, lse, seq_start = ctx.saved_tensors
        if torch.is_grad_enabled() or not plain_tensors(dout):
            from .train import attention_again
            return *attention_again(q, k, v, dout, ctx.max_len,
                                    ctx.scale), None, None, None
        dq, dk32, dv32 = _flash_bwd(q, k, v, out, dout.contiguous(), lse,
                                    seq_start, ctx.max_len, ctx.scale)
        return dq, dk32.to(k.dtype), dv32.to(v.dtype), None, None, None


def flash_attn_train(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                     scale: float) -> torch.Tensor:
    """q: [B, S, HQ, D] bf16 cuda; k/v: [B, S, HKV, D]. Returns [B, S, HQ, D].
    Equal-length sequences are packed varlen (seq_start = i*S)."""
    b, s, hq, d = q.shape
    seq_start = torch.arange(0, (b + 1) * s, s, dtype=torch.int32,
                             device=q.device)
    out = _FlashAttnTrain.apply(
        *(t.reshape(b * s, -1, d).contiguous() for t in (q, k, v)),
        seq_start, s, scale)
    return out.view(b, s, hq, d)


def flash_attn_train_available(d: int) -> bool:
    return have_ext() and d in (64, 128)


# decode-projection GEMM (mfma_gemm.hip): split-K fp32 workspaces, cached
# per (splitk, m, n) so hipGraph capture replays into stable buffers
_GEMM_WS: dict = {}


_compiling = torch.compiler.is_compiling


def plain_tensors(*tensors: Optional[torch.Tensor]) -> bool:
    """No transform, trace, autocast, function or dispatch mode that expects
    torch's own ops, no tensor subclass, batch of tensors, dual number or
    sparse layout; and there are kernels to ask for."""
    if _compiling():        # first: a compiler does not know the others
        return False
    ext = _load_ext()
    if ext is None:
        return False
    state = ext.plain_tensors(*tensors)
    # function modes: one that only gives new tensors a device sees nothing
    return state == 2 or state == 1 and all(
        type(m) is DeviceContext for m in _get_current_function_mode_stack())


def inference_only(*tensors: torch.Tensor) -> bool:
    """Nothing but values is asked of an op on these: no gradients in either
    direction, nothing that expects torch's own ops."""
    if torch.is_grad_enabled() and any(t.requires_grad for t in tensors):
        return False
    return plain_tensors(*tensors)


def _rows_gemm_pays(numel: int, n: int, k: int) -> bool:
    """Whether a product of numel / k rows is faster by rows_gemm.hip than by
    the library, wherever the question is asked (the extension knows more of
    them). Up to 16 rows always: it reads the weights once. Then every
    workgroup, 16 columns, reads all rows as well, which costs less than the
    library's few tiles where there is no more than a workgroup per CU. us, the
    library's and ours:
        32 x 4096 x 4096    13.4  10.3     48 x 4096 x 4096    13.7  12.6
        64 x 4096 x 2048    12.2   8.5     64 x 6144 x 2048    13.2  13.7
    """
    return numel <= 16 * k or n <= 4096 and (
        k <= 4096 and numel <= 32 * k or k <= 2048 and numel <= 64 * k)


def _few_rows(x: torch.Tensor, weight: torch.Tensor,
              bias: Optional[torch.Tensor], gated: bool,
              summed: bool = False):
    """(x as rows, extension) where the product goes to rows_gemm.hip, or
    None. summed: only where the norm that follows adds up its shares."""
    if not (x.is_cuda and weight.is_cuda and x.device == weight.device
            and x.dtype == weight.dtype == torch.bfloat16 and x.dim() >= 1
            and weight.dim() == 2 and x.shape[-1] == weight.shape[1]
            and x.numel() > 0):
        return None
    n, k = weight.shape
    if x.numel() >= 256 * k and os.environ.get("SUB_MGEMM") == "1":
        return None
    # more of them, and larger matrices' rows by mid_gemm.hip, in the same call; a
    # compiler would hold the number of rows to a side of 256
    if _rows_gemm_pays(x.numel(), n, k):
        if summed:
            return None
    elif _compiling() or x.numel() > 256 * k or _load_ext() is None or not (
            _load_ext().mid_norm_good(x.numel() // k, n, k) if summed else
            _load_ext().few_rows_good(x.numel() // k, n, k, gated)):
        return None
    if bias is not None and not (bias.dtype == torch.bfloat16
                                 and bias.device == x.device
                                 and bias.is_contiguous()
                                 and bias.shape == weight.shape[:1]):
        return None
    given = (x, weight) if bias is None else (x, weight, bias)
    ext = _load_ext()
    if ext is None or not inference_only(*given):
        return None
    if x.dim() != 2:
        x = x.reshape(-1, k)
    if not ((summed or ext.rows_gemm_ok(x.shape[0], n, k, gated))
            and weight.is_contiguous() and weight.data_ptr() % 16 == 0
            and x.stride(1) == 1 and x.data_ptr() % 16 == 0
            and (x.stride(0) % 8 == 0 and x.stride(0) >= k
                 or x.shape[0] == 1)):
        return None
    return x, ext


def _tile_gemm(a: torch.Tensor, b: torch.Tensor,
               bias: Optional[torch.Tensor] = None, a_flipped: bool = False,
               b_flipped: bool = False,
               gated: bool = False,
               gelu: bool = False) -> Optional[torch.Tensor]:
    """a b^T + bias on tile_gemm.hip, a stored as [k, m] and b as [k, n] where
    flipped, gated as linear_gated's, its gelu, or None where it does not take them or
    does not pay."""
    ext = _load_ext()
    m, k = a.shape[::-1] if a_flipped else a.shape
    n = b.shape[1 if b_flipped else 0]
    if (ext is None or not all(
            t.is_cuda and t.device == a.device and t.dtype == torch.bfloat16
            and t.stride(1) == 1 and t.data_ptr() % 16 == 0 for t in (a, b))
            or not ext.tile_gemm_good(m, n, k, a.stride(0), b.stride(0),
                                      a_flipped, b_flipped, gated)):
        return None
    if bias is not None and not (
            bias.device == a.device and bias.dtype == torch.bfloat16
            and bias.is_contiguous() and bias.shape == (n,)
            and bias.data_ptr() % 16 == 0):
        return None
    return ext.tile_gemm(a, b, bias, a_flipped, b_flipped, gated, gelu)


class _Linear(torch.autograd.Function):
    """F.linear of rows, each product where it is faster."""

    @staticmethod
    def forward(ctx, x, weight, bias):
        # each gradient needs the other operand: a frozen weight's input is
        # not kept
        dx, dw, _ = ctx.needs_input_grad
        ctx.save_for_backward(x if dw else None, weight if dx else None)
        y = _tile_gemm(x, weight, bias)
        return torch.nn.functional.linear(x, weight, bias) if y is None else y

    @staticmethod
    def backward(ctx, dy):
        x, weight = ctx.saved_tensors
        dx = dw = db = None
        # gradients that can be differentiated again are torch's
        own = not torch.is_grad_enabled() and plain_tensors(dy, x, weight)
        if own and ctx.needs_input_grad[0]:
            dx = _tile_gemm(dy, weight, b_flipped=True)
        if own and ctx.needs_input_grad[1]:
            dw = _tile_gemm(dy, x, a_flipped=True, b_flipped=True)
        if dx is None and ctx.needs_input_grad[0]:
            dx = dy @ weight
        if dw is None and ctx.needs_input_grad[1]:
            dw = dy.t() @ x
        if ctx.needs_input_grad[2]:
            db = dy.sum(0)
        return dx, dw, db


def _many_rows(x: torch.Tensor, weight: torch.Tensor,
               bias: Optional[torch.Tensor],
               gated: bool = False,
               gelu: bool = False) -> Optional[torch.Tensor]:
    """F.linear of 256 rows and more, or None where torch's is as good; or what
    linear_gated or linear_gelu makes of it, without gradients."""
    if not (x.is_cuda and weight.dim() == 2 and weight.shape[0] >= 256
            and x.dim() >= 2 and x.shape[-1] == weight.shape[1] > 0
            and x.numel() >= 256 * x.shape[-1] and not _compiling()
            and _load_ext() is not None):
        return None
    # sizes first, which cost a microsecond: a step of a few hundred rows has
    # dozens of products that stay with torch's
    n, k = weight.shape
    m, good = x.numel() // k, _load_ext().tile_gemm_good
    given = [t for t in (x, weight, bias) if t is not None]
    asked = torch.is_grad_enabled() and any(t.requires_grad for t in given)
    if asked and (gated or gelu) or not (
            good(m, n, k, k, k, False, False, gated)
            or asked and (good(m, k, n, n, k, False, True, False)
                          or good(n, k, m, n, k, True, True, False))):
        return None
    if not (all(t.device == x.device and t.dtype == torch.bfloat16
                for t in given) and plain_tensors(*given)):
        return None
    rows = x.reshape(-1, k)
    y = _Linear.apply(rows, weight, bias) if asked else \
        _tile_gemm(rows, weight, bias, gated=gated, gelu=gelu)
    return y if y is None or x.dim() == 2 else \
        y.view(*x.shape[:-1], y.shape[1])


def linear(x: torch.Tensor, weight: torch.Tensor,
           bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """F.linear. Up to 16 rows of bf16 without gradients, or up to 64 with a
    matrix of few rows, take the kernel that streams weights at the memory's
    rate (rows_gemm.hip), up to 256 rows the one for tiles of them where the
    library's are too few (mid_gemm.hip), products of 256 rows and more the one
    for the matrix cores (tile_gemm.hip) where that is the faster one, in a
    backward as well.
    SUB_MGEMM=1 routes decode shapes of 256 rows and more, whatever else would
    take them, to the 256x256 glds GEMM (mfma_gemm.hip).

    The latter is NOT on by default: measurement
    (profiles/mgemm_r02.md) shows hipBLASLt's MT192/MT256 solutions at 1.3-4.1
    TB/s of weight stream on the llama2-7b decode shapes vs our kernel's
    1.0-2.25 — the library's measured rates reach the ceiling measured for a
    deep-pipelined schedule on this chip (~1.33-1.47 PF). The kernel stays for
    measurement and as the base for a future counted-vmcnt schedule."""
    if not isinstance(x, torch.Tensor):         # a symbolic trace's stand-in
        return torch.nn.functional.linear(x, weight, bias)
    few = _few_rows(x, weight, bias, False)
    if few is not None:
        rows, ext = few
        y = rows.new_empty(rows.shape[0], weight.shape[0])
        ext.rows_gemm(y, rows, weight, bias, False)
        return y if x.dim() == 2 else y.view(*x.shape[:-1], weight.shape[0])
    if (os.environ.get("SUB_MGEMM") != "1" or x.dtype != torch.bfloat16
            or torch.is_grad_enabled() and (
                x.requires_grad or weight.requires_grad)):
        y = _many_rows(x, weight, bias)
        return torch.nn.functional.linear(x, weight, bias) if y is None else y
    ext = _dispatch(x)
    if ext is None:
        return torch.nn.functional.linear(x, weight, bias)
    x2 = x.reshape(-1, x.shape[-1])
    m, k = x2.shape
    n = weight.shape[0]
    if not (256 <= m <= 1024):
        return torch.nn.functional.linear(x, weight, bias)
    splitk = int(ext.mfma_gemm_pick_splitk(m, n, k))
    if splitk == 0:   # unsupported shape
        return torch.nn.functional.linear(x, weight, bias)
    y = x.new_empty(*x.shape[:-1], n)
    part = None
    if splitk > 1:
        key = (x.device.index, splitk, m, n)
        part = _GEMM_WS.get(key)
        if part is None:
            part = torch.empty(splitk * m * n, dtype=torch.float32,
                               device=x.device)
            _GEMM_WS[key] = part
    ext.mfma_gemm(y.view(m, n), x2.contiguous(), weight, bias, part, splitk)
    return y


def linear_gated(x: torch.Tensor, weight: torch.Tensor,
                 bias: Optional[torch.Tensor] = None
                 ) -> Optional[torch.Tensor]:
    """silu(first half) * second half of F.linear's columns, in one kernel, or
    None where it is not made for that."""
    few = _few_rows(x, weight, bias, True)
    if few is None:
        return _many_rows(x, weight, bias, True)
    rows, ext = few
    n = weight.shape[0] // 2
    y = rows.new_empty(rows.shape[0], n)
    ext.rows_gemm(y, rows, weight, bias, True)
    return y if x.dim() == 2 else y.view(*x.shape[:-1], n)


def linear_gelu(x: torch.Tensor, weight: torch.Tensor,
                bias: Optional[torch.Tensor] = None
                ) -> Optional[torch.Tensor]:
    """gelu of F.linear, in one kernel and bit by bit the same, or None where
    it is not made for that."""
    few = _few_rows(x, weight, bias, False)
    if few is None and os.environ.get("SUB_MGEMM") != "1":
        return _many_rows(x, weight, bias, gelu=True)
    if few is None or x.numel() // x.shape[-1] * weight.shape[0] % 8:
        return None
    rows, ext = few
    y = rows.new_empty(rows.shape[0], weight.shape[0])
    ext.rows_gemm(y, rows, weight, bias, False, True)
    return y if x.dim() == 2 else y.view(*x.shape[:-1], weight.shape[0])


class Cache(NamedTuple):
    """What rope_kv_append is told besides the heads: where their tokens are
    and go."""
    positions: torch.Tensor
    k: torch.Tensor
    v: torch.Tensor
    slots: torch.Tensor
    theta: float

    def takes(self, x: torch.Tensor, n: int) -> bool:
        """Whether a product of x with n columns may write it: shapes, types
        and places as its kernel reads them. What is not, rope_kv_append
        copies or refuses."""
        hkv, d = self.k.shape[1], self.k.shape[-1]
        return (self.k.dim() == 4 and self.k.shape == self.v.shape
                and self.k.dtype == self.v.dtype
                and self.k.dtype in (torch.bfloat16, torch.float8_e4m3fn)
                and d % 16 == 0 and n % d == 0 and n > 2 * hkv * d
                and all(t.device == x.device and t.is_contiguous()
                        for t in self[:4])
                and all(t.dtype == torch.int32
                        and t.numel() == x.numel() // x.shape[-1]
                        for t in (self.positions, self.slots))
                and plain_tensors(*self[:4]))


def rope_split_append(qkv: torch.Tensor, hq: int, hkv: int, cache: Cache
                      ) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """(q, k, v), each [rows, heads, d], of fused rows; rope_kv_append of
    them."""
    n, d = qkv.shape[0], qkv.shape[1] // (hq + 2 * hkv)
    if (qkv.is_cuda and qkv.dtype == torch.bfloat16 and qkv.is_contiguous()
            and qkv.numel() > 0 and cache.takes(qkv, qkv.shape[1])
            and cache.k.shape[1] == hkv and d in (16, 32, 64, 128)
            and all(t.data_ptr() % 16 == 0 for t in (qkv, cache.k, cache.v))
            and inference_only(qkv)):
        q = qkv.new_empty(n, hq, d)
        k, v = (qkv.new_empty(n, hkv, d) for _ in range(2))
        _dispatch(qkv).rope_split_append(q, k, v, qkv, *cache)
        return q, k, v
    q, k, v = (t.view(n, -1, d)
               for t in qkv.split([hq * d, hkv * d, hkv * d], dim=-1))
    # rope_kv_append rotates q AND k in place (k also lands rotated in
    # the paged cache); the dense varlen attention consumes them directly
    k = k.contiguous()
    return rope_kv_append(q, k, v, *cache), k, v


def linear_heads(x: torch.Tensor, weight: torch.Tensor,
                 bias: Optional[torch.Tensor],
                 cache: Cache) -> Optional[torch.Tensor]:
    """rope_kv_append of F.linear's columns as heads, in one kernel: the
    rotated queries, or None where it is not made for that."""
    few = _few_rows(x, weight, bias, True)
    n = weight.shape[0]
    if few is None or not cache.takes(x, n):
        return None
    rows, ext = few
    q = rows.new_empty(*_columns(rows.shape[0], n, False, cache))
    ext.rows_heads(q, rows, weight, bias, *cache)
    return q


def norm_goes_in(delta: torch.Tensor, h: torch.Tensor,
                 norm: torch.Tensor) -> bool:
    """Whether a product may make its rows itself, as the RMSNorm of
    h + delta. Up to 4 rows of 8192 numbers in all: every workgroup makes them
    for itself."""
    ext = _load_ext()
    return (ext is not None and h.dim() == 2 and h.shape == delta.shape
            and norm.shape == h.shape[1:] and h.numel() > 0
            and ext.norm_rows_take(*h.shape)
            and all(t.is_cuda and t.device == h.device
                    and t.dtype == torch.bfloat16 and t.is_contiguous()
                    and t.data_ptr() % 16 == 0 for t in (delta, h, norm))
            and inference_only(delta, h, norm))


def linear_normed(delta: torch.Tensor, h: torch.Tensor, norm: torch.Tensor,
                  eps: float, weight: torch.Tensor,
                  bias: Optional[torch.Tensor], gated: bool = False,
                  cache: Optional[Cache] = None):
    """(what becomes of F.linear of norm(h + delta), h + delta) in one kernel,
    or None where it is not made for that: the product, gated as
    linear_gated's, or with a cache linear_heads' queries."""
    if not norm_goes_in(delta, h, norm):
        return None
    few = _few_rows(h, weight, bias, gated or cache is not None)
    m, n = h.shape[0], weight.shape[0]
    if few is None or cache is not None and not cache.takes(h, n):
        return None
    y, total = h.new_empty(*_columns(m, n, gated, cache)), torch.empty_like(h)
    few[1].rows_normed(y, total, delta, h, norm, eps, weight, bias, gated,
                       *(cache or (None,) * 4 + (0.0,)))
    return y, total


class Undivided(NamedTuple):
    """An RMSNorm's rows but for the division by their deviations: rounded
    h * weight, and sums of parts of every row's squares of h, in 32 bits."""
    rows: torch.Tensor
    squares: torch.Tensor


def may_add(h: torch.Tensor, norm: torch.Tensor, rows: int, n: int) -> bool:
    """Whether a product of these rows and columns may be added to h, and make
    the rows of the norm that follows."""
    return (h.shape == (rows, n) and norm.shape == (n,) and n % 64 == 0
            and all(t.is_cuda and t.device == h.device
                    and t.dtype == torch.bfloat16 and t.is_contiguous()
                    and t.data_ptr() % 16 == 0 for t in (h, norm))
            and inference_only(h, norm))


def room_for_added(h: torch.Tensor,
                   parts: int) -> tuple[torch.Tensor, Undivided]:
    """Room for h + a product, and for its norm's rows."""
    return torch.empty_like(h), Undivided(torch.empty_like(h), h.new_empty(
        h.shape[0], parts, dtype=torch.float32))


def linear_added(x: torch.Tensor, weight: torch.Tensor,
                 bias: Optional[torch.Tensor], h: torch.Tensor,
                 norm: torch.Tensor
                 ) -> Optional[tuple[torch.Tensor, Undivided]]:
    """(h + F.linear, RMSNorm of that by the weight norm, undivided) in one
    kernel, or None where it is not made for that. Up to 16 rows: with more of
    them the products that would take such rows are other kernels'."""
    # a compiler would hold the number of rows to a side of 16
    if _compiling() or x.dim() != 2 or x.shape[0] > 16 \
            or x.device != h.device \
            or not may_add(h, norm, x.shape[0], weight.shape[0]):
        return None
    few = _few_rows(x, weight, bias, False)
    if few is None:
        return None
    total, parts = room_for_added(h, few[1].rows_added_parts(
        x.shape[0], *weight.shape))
    few[1].rows_added(parts.rows, total, parts.squares, few[0], weight, bias,
                      h, norm)
    return total, parts


class Normed(NamedTuple):
    """An RMSNorm's rows."""
    rows: torch.Tensor


def linear_added_norm(x: torch.Tensor, weight: torch.Tensor,
                      bias: Optional[torch.Tensor], h: torch.Tensor,
                      norm: torch.Tensor, eps: float
                      ) -> Optional[tuple[torch.Tensor, Normed]]:
    """(h + F.linear, RMSNorm of that by the weight norm), or None: where
    workgroups share the product's sums, which the norm adds up."""
    if _compiling() or x.dim() != 2 or x.shape[0] <= 16 \
            or x.device != h.device \
            or bias is not None and bias.data_ptr() % 16:
        return None
    few = _few_rows(x, weight, bias, False, True)
    if few is None or not may_add(h, norm, x.shape[0], weight.shape[0]):
        return None
    total, rows = torch.empty_like(h), torch.empty_like(h)
    few[1].mid_normed(rows, total, few[0], weight, bias, h, norm, eps)
    return total, Normed(rows)


def linear_scaled(x: Undivided, eps: float, weight: torch.Tensor,
                  bias: Optional[torch.Tensor], gated: bool = False,
                  cache: Optional[Cache] = None) -> Optional[torch.Tensor]:
    """What becomes of F.linear of x divided, gated as linear_gated's, or with a
    cache linear_heads' queries; or None. Every 16 columns ask for all rows'
    squares, so with more than 8 rows and as many columns as a large vocabulary
    has a norm of its own costs less: a step of llama3-8b's first two layers
    and 16 rows 448 us instead of 431."""
    few = _few_rows(x.rows, weight, bias, gated or cache is not None)
    m, n = x.rows.shape[0], weight.shape[0]
    if few is None or m > 16 or m > 8 and n > 65536 \
            or cache is not None and not cache.takes(x.rows, n):
        return None
    y = x.rows.new_empty(*_columns(m, n, gated, cache))
    few[1].rows_scaled(y, *x, eps, weight, bias, gated,
                       *(cache or (None,) * 4 + (0.0,)))
    return y


def _columns(m: int, n: int, gated: bool, cache: Optional[Cache]) -> tuple:
    if cache is None:
        return m, n // 2 if gated else n
    d = cache.k.shape[3]
    return m, n // d - 2 * cache.k.shape[1], d


def silu_mul(x: torch.Tensor) -> torch.Tensor:
    ext = _dispatch(x)
    if ext is None:
        return ref.silu_mul(x)
    out = x.new_empty(*x.shape[:-1], x.shape[-1] // 2)
    ext.silu_mul(out, x.contiguous())
    return out


def gelu(x: torch.Tensor) -> torch.Tensor:
    ext = _dispatch(x)
    if ext is None:
        return ref.gelu(x)
    out = torch.empty_like(x)
    ext.gelu_tanh(out, x.contiguous())
    return out


def softmax_sample(logits: torch.Tensor, temperature: torch.Tensor,
                   top_k: torch.Tensor, top_p: torch.Tensor,
                   uniform: torch.Tensor) -> torch.Tensor:
    ext = _dispatch(logits)
    if ext is None:
        return ref.softmax_sample(logits, temperature, top_k, top_p, uniform)
    out = torch.empty(logits.shape[0], dtype=torch.int64, device=logits.device)
    ext.softmax_sample(out, logits.contiguous(), temperature, top_k, top_p, uniform)
    return out


def cross_entropy_fwd_bwd(logits: torch.Tensor, targets: torch.Tensor,
                          ignore_index: int = -100) -> tuple[torch.Tensor, torch.Tensor]:
    ext = _dispatch(logits)
    if ext is None:
        return ref.cross_entropy_fwd_bwd(logits, targets, ignore_index)
    loss = torch.zeros((), dtype=torch.float32, device=logits.device)
    dlogits = torch.empty_like(logits)
    ext.cross_entropy_fwd_bwd(loss, dlogits, logits.contiguous(), targets, ignore_index)
    return loss, dlogits


def adamw_step(param: torch.Tensor, grad: torch.Tensor, exp_avg: torch.Tensor,
               exp_avg_sq: torch.Tensor, lr: float, beta1: float, beta2: float,
               eps: float, weight_decay: float, step: int,
               grad_scale: float = 1.0) -> None:
    ext = _dispatch(param)
    if ext is None:
        ref.adamw_step(param, grad, exp_avg, exp_avg_sq, lr, beta1, beta2,
                       eps, weight_decay, step, grad_scale)
        return
    ext.adamw_step(param, grad, exp_avg, exp_avg_sq, lr, beta1, beta2,
                   eps, weight_decay, step, grad_scale)


def _steady(tensors, dtype: torch.dtype) -> bool:
    return all(t.is_cuda and t.device == tensors[0].device
               and t.dtype == dtype and t.is_contiguous()
               and t.data_ptr() % 16 == 0 for t in tensors)


def grad_norm(grads: list[torch.Tensor]) -> torch.Tensor:
    """2-norm of all gradients as one vector, a scalar where they are."""
    if grads and _steady(grads, torch.bfloat16):
        return _dispatch(grads[0]).grad_norm(grads)
    norms = torch._foreach_norm(grads, 2.0)
    return torch.linalg.vector_norm(torch.stack(norms))


def adamw_steps(params: list[torch.Tensor], grads: list[torch.Tensor],
                exp_avgs: list[torch.Tensor], exp_avg_sqs: list[torch.Tensor],
                lr: float, beta1: float, beta2: float, eps: float,
                weight_decay: float, step: int, grad_scale: float = 1.0,
                norm: Optional[torch.Tensor] = None,
                clip: float = 0.0) -> None:
    """adamw_step of several tensors. With a norm the gradients are scaled by
    min(1, clip / (norm + 1e-6)) besides, on the GPU without a wait for it."""
    if (params and _steady(params + grads, torch.bfloat16)
            and _steady([*exp_avgs, *exp_avg_sqs], torch.float32)
            and (norm is None or grad_scale == 1.0 and norm.is_cuda
                 and norm.dtype == torch.float32)):
        _dispatch(params[0]).adamw_steps(
            params, grads, exp_avgs, exp_avg_sqs, lr, beta1, beta2, eps,
            weight_decay, step, grad_scale, norm, clip)
        return
    if norm is not None:
        grad_scale *= min(1.0, clip / (float(norm) + 1e-6))
    for p, g, m, v in zip(params, grads, exp_avgs, exp_avg_sqs):
        adamw_step(p, g, m, v, lr, beta1, beta2, eps, weight_decay, step,
                   grad_scale)


# ---- weight-streaming decode GEMM (ops/hip/wstream_gemm.hip) -------------

def wstream_repack(w: torch.Tensor) -> torch.Tensor:
    """Repack a torch Linear weight W[N, K] (bf16) into the MFMA
    B-fragment-linear layout [N/16][K/32][64 lanes][8 bf16] the wstream
    decode GEMM streams sequentially. Lane l = lhi*16+llo holds
    W[n16*16 + llo][t*32 + lhi*8 + j] — one contiguous uint4 per fragment."""
    n, k = w.shape
    assert n % 16 == 0 and k % 32 == 0, (n, k)
    return (w.view(n // 16, 16, k // 32, 4, 8)
             .permute(0, 2, 3, 1, 4).contiguous().view(-1))


def wstream_supported(m: int, n: int, k: int) -> bool:
    return m <= 256 and n % 128 == 0 and k % 64 == 0


def wstream_linear(x: torch.Tensor, wp: torch.Tensor, n: int,
                   k: int) -> torch.Tensor:
    """Y[M, N] = X[M, K] @ W^T with W pre-repacked by wstream_repack.
    GPU-only (decode path); callers fall back to F.linear when unsupported."""
    ext = _dispatch(x)
    assert ext is not None, "wstream_linear is GPU-only"
    m = x.shape[0]
    y = torch.empty(m, n, dtype=x.dtype, device=x.device)
    ext.wstream_gemm(y, x.contiguous(), wp, n, k)
    return y
