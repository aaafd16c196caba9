"""Decode attention of grouped heads against 64 bits: groups around the 16
columns of a matrix instruction, contexts around pages and chunks."""

import pytest
import torch

from substratus_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("hq,hkv,d", [(4, 2, 128), (6, 2, 64), (8, 1, 64),
                                      (32, 2, 128), (17, 1, 128),
                                      (71, 1, 64)])
@pytest.mark.parametrize("contexts", [[1], [15, 16, 17, 31, 32, 33, 64, 65],
                                      [700, 3, 1025]])
def test_groups(hq, hkv, d, contexts):
    torch.manual_seed(hq * d + len(contexts))
    pages = [(c + 15) // 16 for c in contexts]
    order = torch.randperm(sum(pages)).tolist()
    k, v = (torch.randn(sum(pages), hkv, 16, d, device=DEV).bfloat16()
            for _ in range(2))
    table = torch.zeros(len(contexts), max(pages) + 2, dtype=torch.int32)
    at = 0
    for i, n in enumerate(pages):
        table[i, :n] = torch.tensor(order[at:at + n])
        at += n
        if contexts[i] % 16:        # no key is there, whatever the page holds
            for cache in (k, v):
                cache[table[i, n - 1], :, contexts[i] % 16:] = torch.nan
    # queries as columns of a wider projection
    wide = torch.randn(len(contexts), (hq + 2 * hkv) * d, device=DEV) \
        .bfloat16()
    q = wide[:, :hq * d].view(len(contexts), hq, d)
    got = ops.paged_attn_decode(
        q, k, v, table.to(DEV),
        torch.tensor(contexts, dtype=torch.int32, device=DEV), d ** -0.5)
    for i, c in enumerate(contexts):
        kk, vv = (t[table[i, :pages[i]].long()].transpose(1, 2)
                  .reshape(-1, hkv, d)[:c].double()
                  .repeat_interleave(hq // hkv, 1).transpose(0, 1)
                  for t in (k, v))
        s = torch.matmul(kk, q[i].double()[:, :, None])[..., 0] * d ** -0.5
        want = torch.matmul(torch.softmax(s, 1)[:, None], vv)[:, 0]
        # half a bf16 step of the result; weights keep 16 bits, scores' 32-bit
        # sums are off by less
        room = 2.0 ** -8 * want.abs() + 2.0 ** -14 * vv.abs().amax(1)
        assert bool(((got[i].double() - want).abs() <= room).all())
