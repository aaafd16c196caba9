"""Decode attention of more workgroups than the chip holds: each sequence has its
own keys, whatever the lengths are."""

import pytest
import torch

from substratus_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


# sequences of a part of a wave, of one, of two and of all four; all lengths
# equal, none, the table's room; grouped heads and heads by themselves
@pytest.mark.parametrize("batch", [2, 63, 64, 65, 129, 256, 257])
@pytest.mark.parametrize("hq,hkv,d", [(64, 16, 64), (32, 8, 128), (64, 64, 64)])
@pytest.mark.parametrize("how", ["unlike", "equal", "one", "none"])
@torch.no_grad()
def test_own_keys(batch, hq, hkv, d, how):
    g = torch.Generator().manual_seed(batch + d)
    room = 62 if batch < 100 else 60
    most = room * 16
    lens = torch.randint(1, most + 1, (batch,), generator=g)
    if how == "equal":
        lens[:] = most - 3
    elif how == "one":
        lens[:] = 5
        lens[batch // 2] = most
    elif how == "none":
        lens[::3] = 0
    check(batch, hq, hkv, d, room, lens, g)


def check(batch, hq, hkv, d, room, lens, g):
    # few pages, shared by sequences: what tells them apart is their tables
    kc, vc = (torch.randn(70, hkv, 16, d, device=DEV).bfloat16()
              for _ in range(2))
    table = torch.randint(0, 70, (batch, room), generator=g).int().to(DEV)
    q = torch.randn(batch, hq, d, device=DEV).bfloat16()
    n = lens.int().to(DEV)
    out = ops.paged_attn_decode(q, kc, vc, table, n, d ** -0.5)
    per = hq // hkv
    for b in {0, 1, batch // 2, batch - 1, int(lens.argmax()),
              int(lens.argmin())}:
        if lens[b] == 0:
            assert not out[b].any()
            continue
        k, v = (c[table[b].long()].transpose(0, 1).reshape(hkv, -1, d)
                [:, :lens[b]].double().repeat_interleave(per, 0)
                for c in (kc, vc))
        s = torch.einsum("hd,hnd->hn", q[b].double(), k) * d ** -0.5
        want = torch.einsum("hn,hnd->hd", s.softmax(-1), v)
        # results are rounded to bf16, weights have 24 bits
        assert float((out[b].double() - want).norm()) <= \
            2.0 ** -8 * float(want.norm()), b


# long and short ones in a table with room for more, in shares or not
@pytest.mark.parametrize("batch,hq,hkv,d,room,most", [
    (40, 32, 8, 128, 256, 2000), (33, 128, 8, 64, 256, 4096),
    (64, 32, 8, 128, 157, 961), (64, 32, 8, 128, 256, 960),
    (40, 71, 71, 64, 300, 1500), (64, 71, 1, 64, 120, 1900),
    (16, 32, 8, 128, 40, 600), (24, 32, 8, 128, 157, 1500),
    (24, 192, 24, 64, 20, 300), (24, 200, 25, 64, 20, 300),
    (32, 128, 32, 128, 20, 300)])
@torch.no_grad()
def test_shares_in_order(batch, hq, hkv, d, room, most):
    g = torch.Generator().manual_seed(batch + d)
    lens = torch.randint(1, most + 1, (batch,), generator=g)
    lens[batch // 3] = most
    check(batch, hq, hkv, d, room, lens, g)


@pytest.mark.parametrize("hq", [2, 4])
@torch.no_grad()
def test_more_sequences_than_a_grid_side(hq):
    batch, d = 65535 + 9, 64
    kc, vc = (torch.randn(50, 2, 16, d, device=DEV).bfloat16()
              for _ in range(2))
    table = torch.randint(0, 50, (batch, 1), device=DEV).int()
    q = torch.randn(batch, hq, d, device=DEV).bfloat16()
    n = torch.randint(1, 17, (batch,), device=DEV).int()
    out = ops.paged_attn_decode(q, kc, vc, table, n, 0.125)
    for part in (slice(0, 9), slice(batch - 18, batch)):
        assert torch.equal(out[part], ops.paged_attn_decode(
            q[part].contiguous(), kc, vc, table[part].contiguous(),
            n[part].contiguous(), 0.125))


# about 1024 heads, where a sequence's come in turn; heads that share keys or not;
# as many sequences as a grid's second side takes
@pytest.mark.parametrize("batch,hq,hkv,d", [
    (63, 16, 16, 64), (64, 16, 16, 64), (65, 16, 16, 64), (85, 12, 12, 64),
    (86, 12, 12, 64), (1024, 1, 1, 128), (25, 41, 41, 128), (40, 71, 1, 64),
    (64, 96, 2, 128), (65535, 2, 2, 64)])
@pytest.mark.parametrize("fp8", [False, True])
@torch.no_grad()
def test_heads_in_turn(batch, hq, hkv, d, fp8):
    if fp8 and hq // hkv not in (1, 71):
        pytest.skip("other kernels'")
    g = torch.Generator().manual_seed(batch)
    kc, vc = (torch.randn(40, hkv, 16, d, device=DEV).bfloat16()
              for _ in range(2))
    if fp8:
        kc, vc = (t.to(torch.float8_e4m3fn) for t in (kc, vc))
    table = torch.randint(0, 40, (batch, 3), generator=g).int().to(DEV)
    q = torch.randn(batch, hq, d, device=DEV).bfloat16()
    n = torch.randint(0, 49, (batch,), generator=g).int().to(DEV)
    out = ops.paged_attn_decode(q, kc, vc, table, n, 0.125)
    for at in range(0, batch, 512):
        part = slice(at, at + 512)
        k, v = (c.float()[table[part].long()].transpose(1, 2).flatten(2, 3)
                .repeat_interleave(hq // hkv, 1) for c in (kc, vc))
        s = (k @ q[part].float().unsqueeze(-1)).squeeze(-1) * 0.125
        none = torch.arange(48, device=DEV) >= n[part, None, None]
        s = s.masked_fill(none, -torch.inf).softmax(-1).nan_to_num(0.0)
        want = (v * s.unsqueeze(-1)).sum(2)
        # results are rounded to bf16, weights have 24 bits
        assert float((out[part].float() - want).norm()) <= \
            2.0 ** -8 * float(want.norm()), at
