"""Decode attention of a head at a time: ends of steps, of waves and of shares,
against the sums in 64 bits."""

import pytest
import torch

from substratus_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("hq,hkv,d,fp8", [(4, 4, 128, False), (5, 5, 64, False),
                                          (3, 3, 128, True), (7, 1, 64, True)])
@pytest.mark.parametrize("contexts,copies", [
    ([0, 1, 15, 16, 17, 31, 32, 33, 127, 128, 129, 257], 1),   # alone
    ([250, 16, 1, 33], 90),                 # four waves, more than 1024 heads
    ([650, 3, 1300], 1),                    # eight shares
    ([4100, 40], 1),                        # sixteen
])
def test_heads(hq, hkv, d, fp8, contexts, copies):
    torch.manual_seed(hq * d + len(contexts))
    contexts = contexts * copies
    pages = [(c + 15) // 16 for c in contexts]
    order = torch.randperm(sum(pages)).tolist()
    k, v = (torch.randn(sum(pages), hkv, 16, d, device=DEV).bfloat16()
            for _ in range(2))
    # what is behind a sequence's pages is no page
    table = torch.full((len(contexts), max(pages) + 2), 2 ** 30,
                       dtype=torch.int32)
    at = 0
    for i, n in enumerate(pages):
        table[i, :n] = torch.tensor(order[at:at + n])
        at += n
        if contexts[i] % 16:        # no key is there, whatever the page holds
            for cache in (k, v):
                cache[table[i, n - 1], :, contexts[i] % 16:] = torch.nan
    if fp8:
        k, v = k.to(torch.float8_e4m3fn), v.to(torch.float8_e4m3fn)
    # queries as columns of a wider projection
    wide = torch.randn(len(contexts), (hq + 2 * hkv) * d, device=DEV) \
        .bfloat16()
    q = wide[:, :hq * d].view(len(contexts), hq, d)
    got = ops.paged_attn_decode(
        q, k, v, table.to(DEV),
        torch.tensor(contexts, dtype=torch.int32, device=DEV), d ** -0.5)
    k, v = k.double(), v.double()
    for i, c in enumerate(contexts[:len(contexts) // copies]):
        for j in range(0, copies, 17):
            r = i + j * (len(contexts) // copies)
            if c == 0:
                assert not got[r].any()
                continue
            kk, vv = (t[table[r, :pages[r]].long()].transpose(1, 2)
                      .reshape(-1, hkv, d)[:c]
                      .repeat_interleave(hq // hkv, 1).transpose(0, 1)
                      for t in (k, v))
            s = torch.matmul(kk, q[r].double()[:, :, None])[..., 0] * d ** -0.5
            want = torch.matmul(torch.softmax(s, 1)[:, None], vv)[:, 0]
            # half a bf16 step of the result; weights and scores have 32 bits
            room = 2.0 ** -8 * want.abs() + 2.0 ** -14 * vv.abs().amax(1)
            assert bool(((got[r].double() - want).abs() <= room).all())
