"""Products and training ops run where their operands are, whichever device is
the current one."""

import pytest
import torch

from substratus_amd import ops
from substratus_amd.ops import train

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(
    torch.cuda.device_count() < 2, reason="one GPU")]


def test_operands_device():
    def rand(*shape):
        return torch.randn(*shape, generator=g).bfloat16().to("cuda:1") \
            .requires_grad_()

    def results():
        x, w, many = rand(3, 256), rand(64, 256), rand(4165, 4096)
        big, h, d, n = rand(12288, 4096), rand(5, 64), rand(5, 64), rand(64)
        with torch.no_grad():
            out = [ops.linear(x, w), ops.linear_gated(x, w)]
        y = ops.linear(many, big)
        out += [y, *torch.autograd.grad(y, (many, big), y.detach())]
        a, _ = train.add_norm(h, (d,), n, None, 1e-5)
        a = train.silu_mul(a)
        out += [a, *torch.autograd.grad(a, (h, d, n), a.detach()),
                ops.grad_norm([w.detach(), x.detach()])]
        torch.cuda.synchronize("cuda:1")
        return out
    g = torch.Generator().manual_seed(0)
    got = results()
    g.manual_seed(0)
    with torch.cuda.device(1):
        want = results()
    for a, b in zip(got, want):
        assert a.device == torch.device("cuda:1") and torch.equal(a, b)
