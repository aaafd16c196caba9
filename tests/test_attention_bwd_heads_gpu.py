"""The backward of grouped heads at the numbers of heads that a workgroup adds
up (one, two, four; groups that they do not divide) against 64 bits."""

import pytest
import torch

from substratus_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("b,s,hq,hkv,d", [
    (1, 70, 3, 1, 64), (16, 128, 71, 1, 64), (32, 70, 192, 64, 64),
    (64, 65, 66, 22, 64), (16, 100, 64, 16, 128), (16, 200, 71, 1, 64)])
def test_heads(b, s, hq, hkv, d):
    torch.manual_seed(b * s)
    q, k, v = (torch.randn(b, s, h, d, device=DEV).bfloat16()
               .requires_grad_() for h in (hq, hkv, hkv))
    dout = torch.randn(b, s, hq, d, device=DEV).bfloat16()
    out = ops.flash_attn_train(q, k, v, d ** -0.5)
    got = torch.autograd.grad(out, (q, k, v), dout)
    at = [t.detach()[-1:].float().requires_grad_() for t in (q, k, v)]
    kk, vv = (t.repeat_interleave(hq // hkv, 2).transpose(1, 2)
              for t in at[1:])
    sc = (at[0].transpose(1, 2).double() @ kk.double().mT) * d ** -0.5
    mask = torch.ones(s, s, device=DEV, dtype=torch.bool).tril()
    p = torch.softmax(sc.masked_fill(~mask, -torch.inf), -1)
    want = torch.autograd.grad((p @ vv.double()).transpose(1, 2), at,
                               dout[-1:].double())
    # weights and their gradients enter the products as bf16: 2^-9 each, and
    # results are rounded once
    for g, w in zip(got, want):
        off = (g[-1:].double() - w.double()).norm() / w.double().norm()
        assert float(off) < 2.0 ** -7, float(off)


@pytest.mark.parametrize("b,s,hq,hkv,d", [
    (1, 31, 8, 8, 64), (2, 33, 4, 4, 128), (1, 65, 3, 1, 64),
    (2, 255, 2, 1, 128), (1, 300, 5, 5, 64), (16, 128, 71, 1, 64),
    (64, 65, 66, 22, 64), (32, 257, 71, 1, 64), (16, 255, 64, 8, 128),
    (33, 256, 64, 8, 128)])
def test_long_form(b, s, hq, hkv, d, monkeypatch):
    """The keys' and values' kernel for long sequences, at its edges: 32 rows
    of a wave, 64 of a chunk, 256 of a tile."""
    monkeypatch.setenv("SUB_ATTN_DKV_V5", "1")
    test_heads(b, s, hq, hkv, d)


@pytest.mark.parametrize("b,s,hq,hkv,d", [
    (1, 2049, 4, 4, 64), (1, 2111, 3, 3, 128), (1, 8200, 2, 1, 64)])
def test_long(b, s, hq, hkv, d):
    """Lengths from which that kernel is taken."""
    test_heads(b, s, hq, hkv, d)


@pytest.mark.parametrize("scale", [0.125, 0.0, -0.2])
@pytest.mark.parametrize("lens", [[1, 63, 64, 65], [255, 256, 257], [600]])
def test_forward(lens, scale):
    """Rows on both sides of the diagonal's chunks, scales of any sign."""
    torch.manual_seed(sum(lens))
    ss = torch.tensor([0] + lens).cumsum(0).int()
    q, k, v = (torch.randn(sum(lens), h, 64, device=DEV).bfloat16()
               for h in (4, 2, 2))
    got = ops.attn_prefill(q, k, v, ss.to(DEV), scale)
    for lo, hi in zip(ss[:-1].tolist(), ss[1:].tolist()):
        qq, kk, vv = (t[lo:hi].double().transpose(0, 1) for t in (
            q, *(t.repeat_interleave(2, 1) for t in (k, v))))
        mask = torch.ones(hi - lo, hi - lo, device=DEV,
                          dtype=torch.bool).tril()
        p = torch.softmax((torch.matmul(qq, kk.mT.contiguous()) * scale)
                          .masked_fill(~mask, -torch.inf), -1)
        want = torch.matmul(p, vv).transpose(0, 1)
        off = (got[lo:hi].double() - want).norm() / want.norm()
        assert float(off) < 2.0 ** -7, float(off)   # bf16 weights and results
