"""Products that make their rows themselves, as the norm of a sum, against 64
bits and against the norm and the product one after the other."""

import pytest
import torch

from substratus_amd import ops
from substratus_amd.models.quant import QuantLinear
from substratus_amd.parallel.tp import Linear

pytestmark = pytest.mark.gpu
DEV = "cuda"


def made(kind, k, n, bias):
    lin = Linear(k, n, bias=bias, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        lin.weight.normal_(0, k ** -0.5)
        if bias:
            lin.bias.normal_()
    if kind == "dense":
        return lin, lin.weight.double()
    quant = QuantLinear.from_linear(lin.cpu(), kind).to(DEV)
    return quant, quant.dequant_weight().double()


# stages of 64 and 256 columns for 4 or 8 waves, parts of them, the most that
# fits; rows up to four
@pytest.mark.parametrize("kind,m,k,n,bias", [
    ("dense", 1, 32, 48, True), ("dense", 1, 8192, 48, False),
    ("dense", 2, 4096, 160, True), ("dense", 3, 1056, 96, False),
    ("dense", 4, 2048, 256, True), ("q4_0", 1, 5120, 96, False),
    ("q4_0", 3, 320, 64, False), ("q8_0", 2, 448, 48, False),
    ("q4_K", 1, 2560, 64, False), ("q4_K", 4, 2048, 48, False),
    ("q6_K", 1, 256, 64, False), ("q6_K", 2, 1024, 48, False)])
@pytest.mark.parametrize("how", ["plain", "gated", "heads", "turned heads"])
@torch.no_grad()
def test_normed(kind, m, k, n, bias, how):
    torch.manual_seed(m * k + n)
    lin, w = made(kind, k, n, bias)
    h, delta = (torch.randn(m, k, device=DEV).bfloat16() * s for s in (3, 1))
    norm = (1 + 0.3 * torch.randn(k, device=DEV)).bfloat16()
    d, hkv = 16, 1
    cache = None
    if "heads" in how:
        kc, vc = (torch.zeros(m, hkv, 16, d, device=DEV).bfloat16()
                  for _ in range(2))
        at = torch.arange(m, device=DEV).int()
        cache = ops.Cache(at * 3, kc, vc, at * 16 + 5,
                          1e4 if "turned" in how else 0.0)
    got = lin.normed(delta, h, norm, 1e-5, how == "gated", cache)
    assert got is not None
    y, total = got
    assert torch.equal(total, h + delta)
    x = total.double()
    x = x * (x.square().mean(1, keepdim=True) + 1e-5).rsqrt() * norm.double()
    want = x @ w.T + (lin.bias.double() if bias else 0)
    other = lin(ops.rms_norm(total, norm, 1e-5))
    if how == "gated":
        want = torch.nn.functional.silu(want[:, :n // 2]) * want[:, n // 2:]
        other = ops.silu_mul(other)
    elif how == "turned heads":
        plain = lin.normed(delta, h, norm, 1e-5)[0].view(m, -1, d)
        caches = [torch.zeros_like(kc) for _ in range(2)]
        q = ops.rope_kv_append(
            *(t.contiguous() for t in plain.split([n // d - 2, 1, 1], 1)),
            cache.positions, *caches, cache.slots, 1e4)
        # one rounding of the same 32-bit numbers, whose last bits may differ
        for a, b in ((y, q), (kc, caches[0]), (vc, caches[1])):
            a, b = a.float().view(-1), b.float().view(-1)
            assert bool(((a - b).abs() <=
                         2.0 ** -7 * b.abs() + 2.0 ** -20).all())
        return
    elif how == "heads":
        assert torch.equal(y.view(m, -1), lin.normed(
            delta, h, norm, 1e-5)[0][:, :n - 2 * d])
        for c, lo in ((kc, n - 2 * d), (vc, n - d)):
            rows = c[torch.arange(m), 0, 5]
            assert float((rows.double() - want[:, lo:lo + d]).norm()) <= \
                2.0 ** -6 * float(want[:, lo:lo + d].norm())
        y, want, other = (t.reshape(m, -1)[:, :n - 2 * d]
                          for t in (y, want, other))
    # x is rounded once either way, so are the results
    off, most = (float((t.double() - want).norm() / want.norm())
                 for t in (y, other))
    assert off <= 1.3 * most + 2.0 ** -10, (off, most)


@torch.no_grad()
def test_refused():
    lin, _ = made("dense", 4096, 64, False)
    h = torch.randn(5, 4096, device=DEV).bfloat16()
    w = torch.ones(4096, device=DEV).bfloat16()
    assert lin.normed(h[:2], h[:2], w, 1e-5) is not None
    assert lin.normed(h[:3], h[:3], w, 1e-5) is None      # LDS
    assert lin.normed(h[:2], h[:2].float(), w, 1e-5) is None
    assert lin.normed(h[:2, :2048], h[:2, :2048], w[:2048], 1e-5) is None
    with torch.enable_grad():
        assert lin.normed(h[:2], h[:2], w.requires_grad_(), 1e-5) is None
