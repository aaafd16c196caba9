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
        # half a bf16 step of the result; weights and scores are 32-bit numbers
        room = 2.0 ** -8 * want.abs() + 2.0 ** -14 * vv.abs().amax(1)
        assert bool(((got[i].double() - want).abs() <= room).all())


@pytest.mark.parametrize("group", [3, 4, 8, 17])
def test_weights_keep_their_bits(group):
    """Two values that nearly cancel, so that what is left of a result is as
    small as what 16 bits leave out of a weight."""
    torch.manual_seed(group)
    n, hkv, d = 16, 4, 64
    q = (torch.randn(n, hkv * group, d, device=DEV) * 0.3).bfloat16()
    k, v = (torch.zeros(n, hkv, 16, d, device=DEV).bfloat16()
            for _ in range(2))
    k[:, :, :2] = torch.randn(n, hkv, 2, d, device=DEV).bfloat16() * 0.3
    first = q.view(n, hkv, group, d)[:, :, 0].double()
    s = (k[:, :, :2].double() * first[:, :, None]).sum(-1) * d ** -0.5
    a, b = torch.softmax(s, -1)[..., None].unbind(2)      # [n, hkv, 1]
    some = (1 + torch.rand(256, n, hkv, d, device=DEV)).bfloat16().double()
    against = -(some * a / b).bfloat16().double()
    best = (some * a + against * b).abs().argmin(0, keepdim=True)
    v[:, :, 0], v[:, :, 1] = (t.gather(0, best)[0] for t in (some, against))
    got = ops.paged_attn_decode(
        q, k, v, torch.arange(n, device=DEV, dtype=torch.int32)[:, None]
        .contiguous(), torch.full((n,), 2, device=DEV, dtype=torch.int32),
        d ** -0.5).view(n, hkv, group, d)[:, :, 0].double()
    want = v[:, :, 0].double() * a + v[:, :, 1].double() * b
    # 32-bit scores and exponentials: some 2^-23 of either product, about 1
    off = (got - want).abs() - 2.0 ** -8 * want.abs()
    assert float(off.max()) <= 2.0 ** -20


@pytest.mark.parametrize("shares", [2, 3, 4, 5, 8, 9, 12, 16])
@pytest.mark.parametrize("d", [64, 128])
def test_merged_shares(shares, d):
    """As many shares as fill what the merge loads at once, and one more."""
    test_groups(4, 2, d, [64 * shares - 71])
