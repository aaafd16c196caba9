"""Forward and backward of packed sequences at the edges of its tiles: 32 keys or queries
of a wave, 64 taken at a time (32 keys of 128 columns), 128 of a workgroup."""

import pytest
import torch

from substratus_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def reference(q, k, v, dout, scale):
    """Output and gradients of one sequence, in 64 bits."""
    q, k, v = (t.double().requires_grad_() for t in (q, k, v))
    group = q.shape[1] // k.shape[1]
    kk, vv = (t.repeat_interleave(group, 1).transpose(0, 1) for t in (k, v))
    sc = (q.transpose(0, 1) @ kk.mT) * scale
    mask = torch.ones(sc.shape[-2:], dtype=torch.bool).tril()
    p = torch.softmax(sc.masked_fill(~mask, -torch.inf), -1)
    out = (p @ vv).transpose(0, 1)
    return out.detach(), *torch.autograd.grad(out, (q, k, v), dout.double())


@pytest.mark.parametrize("scale", [None, -0.2])
@pytest.mark.parametrize("hq,hkv,d", [(2, 2, 64), (3, 1, 64), (2, 2, 128),
                                      (4, 2, 128)])
@pytest.mark.parametrize("lens", [[1, 31, 32, 33], [64, 65, 63, 2],
                                  [127, 128, 129], [96, 0, 97, 160],
                                  [255, 257], [513]])
def test_packed(lens, hq, hkv, d, scale):
    scale = d ** -0.5 if scale is None else scale
    g = torch.Generator().manual_seed(sum(lens) + hq + d)
    n = sum(lens)
    q, dout = (torch.randn(n, hq, d, generator=g).bfloat16()
               for _ in range(2))
    k, v = (torch.randn(n, hkv, d, generator=g).bfloat16() for _ in range(2))
    starts = torch.tensor([0] + lens).cumsum(0)
    dev = [t.to(DEV) for t in (q, k, v, dout)]
    starts_dev = starts.to(DEV, torch.int32)
    out, lse = ops._flash_fwd(*dev[:3], starts_dev, max(lens), scale)
    got = ops._flash_bwd(*dev[:3], out, dev[3], lse, starts_dev, max(lens),
                         scale)
    want = [torch.zeros(t.shape, dtype=torch.float64) for t in (q, q, k, v)]
    for a, b in zip(starts[:-1], starts[1:]):
        if a < b:
            for w, r in zip(want, reference(q[a:b], k[a:b], v[a:b],
                                            dout[a:b], scale)):
                w[a:b] = r
    # weights and their gradients enter the products as bf16: 2^-9 each; the
    # outputs that Delta is made from and the results are rounded once
    for x, w in zip((out, *got), want):
        off = (x.cpu().double() - w).norm() / w.norm()
        assert float(off) < 2.0 ** -7, float(off)
