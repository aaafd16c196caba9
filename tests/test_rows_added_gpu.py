"""Products that are added to the residual stream and begin the norm that
follows, and products of such rows, which end it: against 64 bits and against the
product, the sum, the norm and the product one after the other."""

from dataclasses import replace

import pytest
import torch

from substratus_amd import ops
from substratus_amd.models import CausalLM, get_config
from tests.test_rows_normed_gpu import DEV, made

pytestmark = pytest.mark.gpu


def kept(x: torch.Tensor, h: torch.Tensor, norm: torch.Tensor, lin):
    total, parts = lin.added(x, h, norm)
    # the same product, rounded, and the same sum as without it
    assert torch.equal(total, h + lin(x))
    assert torch.equal(parts.rows, total * norm)
    squares = total.double().square().sum(1)
    # 16 squares at a time, rounded to 24 bits each time
    assert torch.allclose(parts.squares.double().sum(1), squares, rtol=2e-6)
    return total, parts


# one row and the most that a kernel has, tiles of 16 of them and parts of one;
# shares of 4 and 8 waves; widths of four parts and of more than a load has
@pytest.mark.parametrize("kind,m,k,n,bias", [
    ("dense", 1, 32, 64, True), ("dense", 1, 5632, 2048, False),
    ("dense", 4, 2048, 192, True), ("dense", 8, 4096, 4096, False),
    ("dense", 16, 1056, 320, False), ("q4_0", 1, 13824, 5120, False),
    ("q4_0", 5, 320, 64, False), ("q8_0", 2, 448, 128, False),
    ("q8_0", 4, 512, 576, False), ("q4_K", 1, 2560, 64, False),
    ("q4_K", 5, 2048, 320, False), ("q4_K", 8, 512, 128, False),
    ("q6_K", 3, 256, 64, False), ("q6_K", 6, 1024, 192, False),
    # workgroups of eight weight rows, the last stage a part of one
    ("dense", 8, 4224, 4160, False), ("q4_0", 3, 4160, 4160, False),
    ("q4_0", 1, 4160, 6144, False), ("q8_0", 4, 4352, 4160, False),
    ("q4_K", 5, 4352, 4160, False),
    # workgroups that begin at different columns
    ("dense", 1, 8448, 4160, False), ("dense", 8, 11008, 4160, False),
    ("dense", 16, 8192, 4160, False)])
@pytest.mark.parametrize("how", ["plain", "gated", "heads"])
@torch.no_grad()
def test_added_and_scaled(kind, m, k, n, bias, how):
    torch.manual_seed(m * k + n)
    first, w = made(kind, k, n, bias)
    x = torch.randn(m, k, device=DEV).bfloat16()
    h = 3 * torch.randn(m, n, device=DEV).bfloat16()
    norm = (1 + 0.3 * torch.randn(n, device=DEV)).bfloat16()
    total, parts = kept(x, h, norm, first)
    if n == 4160 or n == 6144:
        want = h.double() + (x.double() @ w.T)
        # two roundings to bf16, and the sums' own
        assert float((total.double() - want).norm()) <= \
            2.0 ** -7 * float(want.norm())
        if kind.endswith("_K"):
            return

    width = 96
    if kind.endswith("_K") and n % 256 or n % 64:
        kind = "dense"
    lin, w = made(kind, n, width, bias and kind == "dense")
    d, cache = 16, None
    if how == "heads":
        kc, vc = (torch.zeros(m, 1, 16, d, device=DEV).bfloat16()
                  for _ in range(2))
        at = torch.arange(m, device=DEV).int()
        cache = ops.Cache(at, kc, vc, at * 16 + 5, 0.0)
    if type(lin).__name__ == "QuantLinear" and lin.quant == "q8_0" and m == 1:
        assert lin.scaled(parts, 1e-5, how == "gated", cache) is None
        return
    y = lin.scaled(parts, 1e-5, how == "gated", cache)
    t = total.double()
    want = (t * (t.square().mean(1, keepdim=True) + 1e-5).rsqrt()
            * norm.double()) @ w.T
    if getattr(lin, "bias", None) is not None:
        want += lin.bias.double()
    other = lin(ops.rms_norm(total, norm, 1e-5))
    if how == "gated":
        want = torch.nn.functional.silu(want[:, :width // 2]) \
            * want[:, width // 2:]
        other = ops.silu_mul(other)
    elif how == "heads":
        rows = torch.arange(m, device=DEV)
        y = torch.cat([y.reshape(m, -1), kc[rows, 0, 5], vc[rows, 0, 5]], 1)
    # x is rounded once either way, so are the results
    off, most = (float((t.double() - want).norm() / want.norm())
                 for t in (y, other))
    assert off <= 1.3 * most + 2.0 ** -10, (off, most)


@torch.no_grad()
def test_refused():
    lin, _ = made("dense", 128, 256, False)
    x, h = (torch.randn(17, n, device=DEV).bfloat16() for n in (128, 256))
    w = torch.ones(256, device=DEV).bfloat16()
    assert lin.added(x[:16], h[:16], w) is not None
    assert lin.added(x, h, w) is None
    assert lin.added(x[:2], h[:1], w) is None
    assert lin.added(x[:2], h[:2].float(), w) is None
    assert lin.added(x[:2], h[:4:2], w) is None
    assert lin.added(x[:2], h[:2].cpu(), w) is None
    odd, _ = made("dense", 128, 72, False)      # parts in fours
    assert odd.added(x[:2], h[:2, :72].contiguous(), w[:72]) is None
    with torch.enable_grad():
        assert lin.added(x[:2], h[:2], w.requires_grad_()) is None


# a head with more columns than it divides rows for, from 9 rows on; tied
# embeddings, whose product is torch's; rows of either kernel and a norm's own
@pytest.mark.parametrize("vocab,tied", [(65600, False), (512, True),
                                        (512, False)])
@pytest.mark.parametrize("rows", [1, 8, 12, 16, 40])
@torch.no_grad()
def test_last_norm(vocab, tied, rows, monkeypatch):
    """Logits of a step whose last rows come undivided, beside those of a step
    that adds and norms by itself."""
    cfg = replace(get_config("llama-tiny"), vocab_size=vocab, num_layers=2,
                  intermediate_size=8192, tie_word_embeddings=tied)
    model = CausalLM(cfg, device=DEV, dtype=torch.bfloat16)
    model.init_random(3)
    d = cfg.head_dim
    at = torch.arange(rows, device=DEV, dtype=torch.int32)
    tokens = torch.randint(0, vocab, (rows,), device=DEV)

    def step():
        caches = [tuple(torch.zeros(rows, model.n_kv_heads, 16, d,
                                    device=DEV).bfloat16() for _ in range(2))
                  for _ in model.blocks]
        return model.forward_decode(
            tokens, torch.zeros_like(at), caches, at * 16,
            at[:, None].contiguous(), torch.ones_like(at)).double()

    kinds = []
    for name in "linear_added", "linear_added_norm", "linear_scaled":
        def spy(*a, name=name, run=getattr(ops, name), **kw):
            got = run(*a, **kw)
            kinds.append((name, got is not None))
            return got
        monkeypatch.setattr(ops, name, spy)
    got = step()
    assert (("linear_added", True) in kinds) == (rows <= 16)
    assert (("linear_added_norm", True) in kinds) == (rows > 16)
    if vocab > 65536:
        assert (("linear_scaled", False) in kinds) == (9 <= rows <= 16)
    for name in "linear_added", "linear_added_norm":
        monkeypatch.setattr(ops, name, lambda *a: None)
    want = step()
    # rows are rounded to bf16 at another place: 2^-9 of each of some ten
    assert float((got - want).norm()) <= 0.02 * float(want.norm())
