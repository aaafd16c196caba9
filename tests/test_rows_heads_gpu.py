"""Projections of heads that rotate and append in the same kernel against the
product and rope_kv_append by themselves, dense and quantized."""

import pytest
import torch

from substratus_amd import ops
from substratus_amd.models.quant import QuantLinear
from substratus_amd.parallel.tp import Linear

pytestmark = pytest.mark.gpu
DEV = "cuda"


def projection(kind, k, n, bias):
    lin = Linear(k, n, bias=bias, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        lin.weight.normal_(0, k ** -0.5)
        if bias:
            lin.bias.normal_()
    if kind == "dense":
        return lin
    return QuantLinear.from_linear(lin.cpu(), kind).to(DEV)


@pytest.mark.parametrize("kind,m,hq,hkv,d,k,bias", [
    ("dense", 1, 2, 1, 16, 32, False), ("dense", 3, 4, 2, 64, 96, True),
    ("dense", 16, 5, 5, 128, 160, False), ("dense", 7, 3, 1, 80, 2048, True),
    ("q4_0", 1, 4, 4, 64, 320, False), ("q4_0", 40, 4, 2, 128, 64, False),
    ("q8_0", 5, 2, 2, 128, 128, False), ("q4_K", 17, 4, 1, 64, 512, False),
    ("q6_K", 2, 4, 4, 128, 256, False)])
@pytest.mark.parametrize("theta,fp8", [(10000.0, False), (0.0, False),
                                       (500.0, True)])
@torch.no_grad()
def test_heads(kind, m, hq, hkv, d, k, bias, theta, fp8):
    torch.manual_seed(m * d + k)
    lin = projection(kind, k, (hq + 2 * hkv) * d, bias)
    x = torch.randn(m, k, device=DEV).bfloat16()
    kind8 = torch.float8_e4m3fn if fp8 else torch.bfloat16
    pages, size = m + 2, 16

    def cache():
        k, v = (torch.zeros(pages, hkv, size, d, device=DEV, dtype=kind8)
                for _ in range(2))
        slots = (torch.arange(m, device=DEV) * 17 + 3).int()
        at = (torch.arange(m, device=DEV) * 211 % 4001).int()
        return ops.Cache(at, k, v, slots, theta)

    here, want = cache(), cache()
    q = lin.heads(x, here)
    assert q is not None and q.shape == (m, hq, d)
    parts = lin(x).split([hq * d, hkv * d, hkv * d], 1)
    qw = ops.rope_kv_append(*(t.reshape(m, -1, d).contiguous()
                              for t in parts), *want)
    # one rounding of the same 32-bit numbers, whose last bits may differ
    for got, ref, step in ((q, qw, 2.0 ** -7),
                           (here.k, want.k, 2.0 ** -3 if fp8 else 2.0 ** -7),
                           (here.v, want.v, 0.0)):
        got, ref = got.float(), ref.float()
        assert bool(((got - ref).abs() <=
                     step * ref.abs() + 2.0 ** -20).all())
        if step and theta > 0:
            assert float((got != ref).float().mean()) < 0.01


@torch.no_grad()
def test_heads_refused():
    """What the kernel does not read goes the general way."""
    lin = projection("dense", 64, 6 * 64, False)
    x = torch.randn(65, 64, device=DEV).bfloat16()
    pos = torch.arange(65, device=DEV).int()
    k, v = (torch.zeros(17, 1, 16, 64, device=DEV).bfloat16()
            for _ in range(2))
    ok = ops.Cache(pos[:4], k, v, pos[:4], 1e4)
    assert lin.heads(x[:4], ok) is not None
    assert lin.heads(x, ops.Cache(pos, k, v, pos, 1e4)) is None
    for other in (ok._replace(slots=pos[:8:2]), ok._replace(slots=pos[:3]),
                  ok._replace(positions=pos[:4].long()),
                  ok._replace(k=k.float(), v=v.float()),
                  ok._replace(v=v[:, :, ::2])):
        assert lin.heads(x[:4], other) is None
    with torch.enable_grad():
        assert lin.heads(x[:4], ok) is None
