"""A prompt's rows on the GPU: fused rows split, rotated and appended in one
kernel against rope_kv_append, and what goes the general way."""

import pytest
import torch

from substratus_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("rows,hq,hkv,d", [(1, 1, 1, 16), (5, 71, 1, 64),
                                           (33, 4, 2, 128), (300, 3, 3, 32),
                                           (7, 3, 1, 80)])
@pytest.mark.parametrize("theta", [10000.0, 0.0])
@pytest.mark.parametrize("fp8", [False, True])
@torch.no_grad()
def test_rope_split_append(rows, hq, hkv, d, theta, fp8):
    torch.manual_seed(rows * d)
    qkv = torch.randn(rows, (hq + 2 * hkv) * d, device=DEV).bfloat16()
    kind = torch.float8_e4m3fn if fp8 else torch.bfloat16
    pages = (rows + 15) // 16 + 1

    def cache():
        k, v = (torch.zeros(pages, hkv, 16, d, device=DEV, dtype=kind)
                for _ in range(2))
        at = torch.arange(rows, device=DEV)
        return ops.Cache((at * 37 % 4001).int(), k, v, (at + 9).int(), theta)

    here, want = cache(), cache()
    before = qkv.clone()
    got = ops.rope_split_append(qkv, hq, hkv, here)
    if d != 80:                         # which the kernel does not take
        assert torch.equal(qkv, before)
    q, k, v = (t.reshape(rows, -1, d).contiguous()
               for t in before.split([hq * d, hkv * d, hkv * d], 1))
    q = ops.rope_kv_append(q, k, v, *want)
    # one rounding of the same 32-bit numbers, whose last bits may differ
    for a, b, step in ((got[0], q, 2.0 ** -7), (got[1], k, 2.0 ** -7),
                       (got[2], v, 0.0),
                       (here.k, want.k, 2.0 ** -3 if fp8 else 2.0 ** -7),
                       (here.v, want.v, 0.0)):
        a, b = a.float(), b.float()
        assert bool(((a - b).abs() <= step * b.abs() + 2.0 ** -20).all())
        assert float((a != b).float().mean()) < 0.01
