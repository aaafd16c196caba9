"""Products that are added to the residual stream and begin the norm that
follows, and products of such rows, which end it: against 64 bits and against the
product, the sum, the norm and the product one after the other."""

import pytest
import torch

from substratus_amd import ops
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
