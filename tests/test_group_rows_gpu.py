"""Grouped products of few rows: ends of stages, rings, tiles and columns, tails
copied by pieces, gates fetched ahead, against the products in 64 bits."""

import pytest
import torch

from substratus_amd.models.layers import MoESpec
from substratus_amd.ops import hybrid as ops
from test_hybrid_ops_gpu import close, rand

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.mark.parametrize("tile", [16, 32, 64])
@pytest.mark.parametrize("k,n,act", [(128, 16, "none"), (160, 44, "gelu"),
                                     (1056, 24, "silu"), (2080, 72, "none"),
                                     (2048, 8, "gelu"), (128, 1040, "none"),
                                     (1056, 472, "silu"), (1312, 472, "none")])
def test_experts_of_few_rows(tile, k, n, act):
    counts = [1, 15, 0, 16, 17, 31, 32, 33, 2, 48, 49, 64, 65]
    total, e = sum(counts), len(counts)
    g = torch.Generator().manual_seed(k + n)
    ids = torch.repeat_interleave(torch.arange(e), torch.tensor(counts))
    ids = ids[torch.randperm(total, generator=g)].int()[:, None].contiguous()
    x = rand(total, k, seed=1, dtype=BF16)
    w = rand(e, n, k, seed=2, dtype=BF16, scale=k ** -0.5)
    i32 = dict(dtype=torch.int32, device="cuda")
    at, src = torch.empty(total, 1, **i32), torch.empty(total, **i32)
    start = torch.empty(e + 1, **i32)
    tiles = torch.empty(1 + 2 * ((total + tile - 1) // tile + e), **i32)
    ext = ops._ext()
    ext.moe_sort(at, src, start, tiles, ids.cuda(), tile)
    assert start.tolist() == torch.tensor([0] + counts).cumsum(0).tolist()
    cols = n // 2 if act == "silu" else n
    out = torch.full((total, cols), 9.0, dtype=BF16, device="cuda")
    ext.expert_linear(out, x.cuda(), w.cuda(), src, start, tiles, tile, act,
                      0.0)
    want = torch.empty(total, cols, dtype=torch.float64)
    for i in range(e):
        r = ids[:, 0] == i
        y = x[r].double() @ w[i].double().T
        if act == "gelu":
            y = torch.nn.functional.gelu(y)
        if act == "silu":           # columns are gate and up in turn
            y = torch.nn.functional.silu(y[:, ::2]) * y[:, 1::2]
        want[r] = y
    close(out[at[:, 0].long()], want.float(), BF16)


# Rows that are looked for by their ids: fewer than experts, of one expert more than
# a tile holds, of a token twice the same (scores that were no numbers), experts
# without any where weights are asked for first, and the most ids; the packed rows'
# kernel has the same bits.
@pytest.mark.parametrize("tile", [16, 32])
@pytest.mark.parametrize("k,ff,act", [(128, 160, "none"), (1056, 128, "silu"),
                                      (2080, 1312, "gelu")])
@pytest.mark.parametrize("rows,top,e", [(1, 2, 5), (3, 1, 5), (3, 2, 6),
                                        (5, 2, 7), (40, 1, 3), (64, 8, 9),
                                        (128, 4, 4)])
def test_experts_by_ids(tile, k, ff, act, rows, top, e):
    g = torch.Generator().manual_seed(rows + k)
    ids = torch.stack([torch.randperm(max(e, top), generator=g)[:top] % e
                       for _ in range(rows)]).int()
    ids[ids == e - 2] = 0                   # an expert without rows
    if rows > 2:
        ids[1] = ids[1, 0]
    ids = ids.cuda()
    n, each = rows * top, 2 if act == "silu" else 1
    x = rand(rows, k + 8, seed=1, dtype=BF16).cuda()[:, :k]
    up = rand(e, each * ff, k, seed=2, dtype=BF16, scale=k ** -0.5).cuda()
    down = rand(e, k, ff, seed=3, dtype=BF16, scale=ff ** -0.5).cuda()
    ext = ops._ext()
    h, out = (torch.full((n, c), 9.0, dtype=BF16, device="cuda")
              for c in (ff, k))
    if not ext.experts_chosen(h, out, x, up, down, ids, tile, act, 0.0, True):
        assert tile == 16 and n == 512      # many blocks of short rows
        pytest.skip("another kernel's")
    assert bool((h == 9).all())
    assert ext.experts_chosen(h, out, x, up, down, ids, tile, act, 0.0, False)
    i32 = dict(dtype=torch.int32, device="cuda")
    at, src = torch.empty(rows, top, **i32), torch.empty(n, **i32)
    start = torch.empty(e + 1, **i32)
    tiles = torch.empty(1 + 2 * ((n + tile - 1) // tile + min(e, n)), **i32)
    ext.moe_sort(at, src, start, tiles, ids, tile)
    h2, out2 = torch.empty_like(h), torch.empty_like(out)
    ext.expert_linear(h2, x, up, src, start, tiles, tile, act, 0.0)
    ext.expert_linear(out2, h2, down, None, start, tiles, tile, "none", 0.0)
    where = at.view(-1).long()
    assert torch.equal(h, h2[where]) and torch.equal(out, out2[where])


@pytest.mark.parametrize("rows", [1, 32, 33, 100])
def test_tokens_of_the_same_experts(rows):
    """All choose alike: an expert's rows are one tile of up to 32, or packed, where
    its tiles lie side by side."""
    spec = MoESpec(8, 2, 128)
    y = rand(1, 256, seed=1, dtype=BF16).repeat(rows, 1)
    y += rand(rows, 256, seed=2, dtype=BF16, scale=2.0 ** -6)
    router = rand(8, 256, seed=3, dtype=BF16)
    up = rand(8, 128, 256, seed=4, dtype=BF16, scale=2.0 ** -4)
    down = rand(8, 256, 128, seed=5, dtype=BF16, scale=2.0 ** -3.5)
    want = ops.experts(y, router, up, down, spec)
    got = ops.experts(y.cuda(), router.cuda(), up.cuda(), down.cuda(), spec)
    kept = torch.arange(2 * rows, dtype=torch.int32).view(rows, 2)
    if rows > 1:
        assert torch.equal(got.at.cpu(), kept) == (rows <= 32)
    close(got.rows[got.at.long()], want.rows[want.at.long()], BF16)


def test_experts_that_are_packed():
    """Too many ids, tiles of 64 rows, rows that are no whole chunks, float."""
    ext = ops._ext()

    def asks(rows, k, ff, tile, dtype=BF16):
        z = dict(dtype=dtype, device="cuda")
        return ext.experts_chosen(
            torch.empty(rows * 2, ff, **z), torch.empty(rows * 2, k, **z),
            torch.empty(rows, k, **z), torch.empty(4, ff, k, **z),
            torch.empty(4, k, ff, **z),
            torch.zeros(rows, 2, dtype=torch.int32, device="cuda"), tile,
            "none", 0.0, True)
    assert asks(256, 128, 160, 32) and not asks(257, 128, 160, 32)
    assert not asks(4, 128, 160, 64) and not asks(4, 144, 160, 32)
    assert not asks(4, 128, 160, 32, torch.float32)


@pytest.mark.parametrize("rows", [1, 16, 48, 65, 300])
@pytest.mark.parametrize("k,n,tail,each", [(512, 128, 0, True),
                                           (512, 72, 0, False),
                                           (128, 512, 64, None),
                                           (256, 40, 24, True),
                                           (128, 64, 12, None)])
def test_heads_of_few_rows(rows, k, n, tail, each):
    heads = 3
    x = rand(rows, heads * (k + tail), seed=1, dtype=BF16)
    w = rand(heads, n, k, seed=2, dtype=BF16, scale=k ** -0.5)
    gate = None if each is None else rand(
        rows, heads * n if each else heads, seed=3, dtype=BF16)
    v = x.view(rows, heads, k + tail)
    got = ops.head_linear(v.cuda(), w.cuda(),
                          None if gate is None else gate.cuda(), tail)
    want = torch.einsum("rhk,hnk->rhn", v[..., :k].double(), w.double())
    if gate is not None:
        want *= torch.sigmoid(gate.double().view(rows, heads, -1))
    close(got[..., :n], want.float(), BF16)
    assert torch.equal(got[..., n:].cpu(), v[..., k:])


@pytest.mark.parametrize("rows", [1, 17, 48])
def test_side_gate_of_few_columns(rows):
    y = rand(rows, 1088, seed=1, dtype=BF16)
    w = rand(40, 1088, seed=2, dtype=BF16, scale=1088 ** -0.5)
    table = rand(50, 80, seed=3, dtype=BF16)
    tok = torch.randint(0, 50, (rows,), dtype=torch.int32)
    got = ops.side_gate(y.cuda(), w.cuda(), tok.cuda(), table.cuda(), 40)
    want = torch.nn.functional.gelu(y.double() @ w.double().T,
                                    approximate="tanh") \
        * table[tok.long(), 40:].double()
    close(got, want.float(), BF16)
