"""The optimizer's launches over many tensors: sizes around the elements of a
workgroup, more tensors than a launch takes, norms that clip and that do not."""

import pytest
import torch

from substratus_amd import ops
from substratus_amd.ops import ref

pytestmark = pytest.mark.gpu
DEV = "cuda"
SIZES = [1, 7, 8, 8191, 8192, 8193, 32767, 32769, 100003] + [33] * 38


@pytest.mark.parametrize("norm,clip", [(None, 0.0), (1e-3, 1.0), (40.0, 1.0),
                                       (float("inf"), 1.0),
                                       (float("nan"), 1.0)])
def test_adamw_steps(norm, clip):
    torch.manual_seed(1)
    given = [[torch.randn(n).bfloat16(), torch.randn(n).bfloat16(),
              torch.randn(n), torch.rand(n)] for n in SIZES]
    here = [[t.to(DEV) for t in four] for four in given]
    scale = 1.0 if norm is None else min(1.0, clip / (norm + 1e-6))
    ops.adamw_steps(*([f[i] for f in here] for i in range(4)), 1e-2, 0.9,
                    0.95, 1e-8, 0.1, 3,
                    norm=None if norm is None else torch.tensor(norm,
                                                                device=DEV),
                    clip=clip)
    for four, got in zip(given, here):
        p, g, m, v = four
        ref.adamw_step(p, g, m, v, 1e-2, 0.9, 0.95, 1e-8, 0.1, 3, scale)
        # 32-bit moments to some steps, the parameter to its own
        assert torch.allclose(got[2].cpu(), m, rtol=1e-5, atol=1e-6)
        assert torch.allclose(got[3].cpu(), v, rtol=1e-5, atol=1e-6)
        assert torch.allclose(got[0].cpu().float(), p.float(),
                              rtol=2.0 ** -7, atol=1e-5)


def test_grad_norm():
    torch.manual_seed(2)
    gs = [torch.randn(n, device=DEV).bfloat16() * 3 for n in SIZES]
    exact = sum(g.double().square().sum() for g in gs).sqrt()
    got = ops.grad_norm(gs)
    assert got.dtype == torch.float32 and got.dim() == 0
    # 128 squares a thread in 32 bits, then few sums
    assert abs(float(got) / float(exact) - 1) < 2.0 ** -18
    gs[3][5] = torch.inf
    assert float(ops.grad_norm(gs)) == float("inf")
    # what the kernel does not read goes to torch's
    off = [torch.randn(65, device=DEV).bfloat16()[1:], gs[0]]
    assert abs(float(ops.grad_norm(off)) /
               float(torch.cat(off).double().norm()) - 1) < 2.0 ** -7
