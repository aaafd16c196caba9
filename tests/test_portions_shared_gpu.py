"""Prompt portions by waves that share their rows (few tiles) and by waves of their
own (many heads): ends of 32 rows, of tiles and of steps of keys, a wave without keys,
every kind of weight, against the products in 64 bits."""

import pytest
import torch

from substratus_amd.ops import hybrid as ops
from test_hybrid_ops_gpu import BS, make_batch, on_gpu, rand

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16
# first position and rows; single ones come first in a batch
SPANS = [(0, 1), (0, 32), (31, 33), (40, 127), (0, 128), (63, 129), (0, 31)]
# contexts long enough to be shared, one whose shares have no step each
LONG = [(900, 33), (0, 2), (511, 65), (100, 3)]
# several steps for each share, a portion on both sides of a chunk's end
LONGER = [(3060, 33), (0, 2), (1501, 65), (700, 3)]


def wide(q, k, v, first, scale, kind):
    """One head of one portion in 64 bits."""
    n, keys = q.shape[0], k.shape[0]
    i = first + torch.arange(n)[:, None]
    j = torch.arange(keys)[None]
    s = scale * q.double() @ k.double().T
    if kind.get("softcap"):
        s = kind["softcap"] * torch.tanh(s / kind["softcap"])
    bias = kind["bias"].double()
    s = s + bias[(i - j).clamp(0, bias.shape[0] - 1)]
    seen = j <= i
    if kind.get("window"):
        seen &= (i - j < kind["window"]) | (j < kind["keep"])
    if kind.get("chunk"):
        seen &= i // kind["chunk"] == j // kind["chunk"]
    if kind.get("weight_bias") is not None:
        w = torch.sigmoid(s + kind["weight_bias"].double()) * seen
    else:
        s = s.masked_fill(~seen, -torch.inf)
        if kind.get("sink") is not None:
            s = torch.cat([s, kind["sink"].double().expand(n, 1)], 1)
        w = torch.softmax(s, 1)[:, :keys]
    return w @ v.double()


@pytest.mark.parametrize("dim,vdim", [(64, 64), (128, 128), (96, 40),
                                      (192, 72), (256, 256)])
@pytest.mark.parametrize("kind", ["plain", "sink", "sigmoid", "cap", "window",
                                  "chunk"])
@pytest.mark.parametrize("times,spans", [(1, SPANS), (32, SPANS), (1, LONG)])
def test_portions(dim, vdim, kind, times, spans):
    portions(dim, vdim, kind, times, spans, dict(window=37, keep=5), 48)


# Shares of three steps and more, which begin within a context, behind a window, kept
# keys or a chunk's first key too.
@pytest.mark.parametrize("dim,vdim", [(64, 64), (128, 128), (192, 72), (256, 256)])
@pytest.mark.parametrize("kind,times", [
    ("plain", 1), ("sink", 1), ("sigmoid", 1), ("cap", 1), ("sink", 8),
    ("window", 8), ("chunk", 8)])
def test_shares_of_several_steps(dim, vdim, kind, times):
    span = {"window": 970, "chunk": 1024}.get(kind, 3093)
    rows = sum(n for _, n in LONGER)
    shares = ops._ext().attn_ctx_prefill_splits(len(LONGER), rows, 4 * times,
                                                vdim, span)
    assert 1 < shares <= span // 64 // 3
    portions(dim, vdim, kind, times, LONGER, dict(window=900, keep=70), 1024)


def test_shares_of_low_scores():
    """Lower than any number that stands for no score."""
    portions(128, 128, "plain", 1, LONG, None, 0, add=-2e30)


def portions(dim, vdim, kind, times, spans, window, chunk, add=0.0):
    g, h = 2, 4
    blocks = max(128, sum((f + n) // BS + 1 for f, n in spans))
    batch = make_batch(spans, blocks)
    n = batch.tokens.shape[0]
    # one sharp score per row, so that a wrong key shows
    q = rand(n, h, dim, seed=1, dtype=BF16, scale=2.0)
    kc = rand(blocks, g, BS, dim, seed=2, dtype=BF16)
    vc = rand(blocks, g, BS, vdim, seed=3, dtype=BF16)
    bias = rand(h, 77, seed=4) + add
    per_head = rand(h, seed=5)
    kinds = {"sink": dict(sink=per_head), "sigmoid": dict(weight_bias=per_head),
             "cap": dict(softcap=3.0), "window": window,
             "chunk": dict(chunk=chunk)}.get(kind, {})
    scale = dim ** -0.5
    want = torch.empty(n, h, vdim, dtype=torch.float64)
    row = 0
    for e, (first, m) in enumerate(spans):
        pages, at = batch.block_table[e].long(), row
        for x in range(h):
            k = kc[pages, x // 2].reshape(-1, dim)[:first + m]
            v = vc[pages, x // 2].reshape(-1, vdim)[:first + m]
            one = {a: (b[x] if torch.is_tensor(b) else b)
                   for a, b in kinds.items()}
            want[at:at + m, x] = wide(q[at:at + m, x], k, v, first, scale,
                                      dict(one, bias=bias[x]))
        row += m

    def more(t, at):                    # the same heads again and again
        return t.repeat_interleave(times, at).cuda()
    args = {a: (more(b, 0) if torch.is_tensor(b) else b)
            for a, b in kinds.items()}
    got = ops.attn_ctx(more(q, 1).flatten(1), None, more(kc, 1), more(vc, 1),
                       more(bias, 0), on_gpu(batch), scale, **args)
    got = got.view(n, h, times, vdim).cpu().double()
    # half a step of the result: 2^-8 of the power of two below it (8 bits of
    # significand); weights of 16 bits and 32-bit sums before
    room = 2.0 ** -8 * want.abs() + 2.0 ** -13 * 4 * want.abs().amax()
    assert bool(((got - want[:, :, None]).abs() <= room[:, :, None]).all())


@pytest.mark.parametrize("dim,vdim,shared", [(64, 64, 16), (192, 128, 64),
                                             (256, 256, 8)])
@pytest.mark.parametrize("window", [0, 37])
@pytest.mark.parametrize("times", [1, 32])
def test_unpaged(dim, vdim, shared, window, times):
    h, spans = 4, SPANS[1:]
    own, i32 = dim - shared, dict(dtype=torch.int32, device="cuda")
    ends = torch.tensor([0] + [m for _, m in spans]).cumsum(0)
    froms = [max(f - window + 1, 0) if window else 0 for f, _ in spans]
    starts = torch.tensor([0] + [f + m - c for (f, m), c in
                                 zip(spans, froms)]).cumsum(0)
    n, keys = int(ends[-1]), int(starts[-1])
    q = rand(n, h, dim, seed=1, dtype=BF16, scale=2.0)
    k = rand(keys, h, own, seed=2, dtype=BF16)
    v = rand(keys, h, vdim, seed=3, dtype=BF16)
    kr = rand(keys, shared, seed=4, dtype=BF16)
    gate = rand(n, h, seed=5, dtype=BF16)
    want = torch.empty(n, h, vdim, dtype=torch.float64)
    for e, (first, m) in enumerate(spans):
        at, ks = slice(int(ends[e]), int(ends[e + 1])), \
            slice(int(starts[e]), int(starts[e + 1]))
        for x in range(h):
            # keys ahead of the first that lies there are seen by no row
            pad = (froms[e], 0)
            kx = torch.cat([k[ks, x], kr[ks]], 1)
            kx, vx = (torch.nn.functional.pad(t, (0, 0) + pad)
                      for t in (kx, v[ks, x]))
            want[at, x] = wide(q[at, x], kx, vx, first, dim ** -0.5, dict(
                bias=torch.zeros(1), window=window, keep=0))
    want *= torch.sigmoid(gate.double())[:, :, None]

    def more(t):
        return t.repeat_interleave(times, 1)
    out = torch.empty(n, h * times * vdim, dtype=BF16, device="cuda")
    kv = torch.cat([more(k).flatten(1), more(v).flatten(1)], 1).cuda()
    pos = torch.cat([f + torch.arange(m) for f, m in spans])
    ops._ext().attn_flat(
        out, more(q).flatten(1).cuda(), more(gate).cuda(), kv, kr.cuda(),
        pos.to(**i32), ends.to(**i32), starts.to(**i32), h * times, vdim,
        dim ** -0.5, window, max(m for _, m in spans))
    got = out.view(n, h, times, vdim).cpu().double()
    room = 2.0 ** -8 * want.abs() + 2.0 ** -13 * 4 * want.abs().amax()
    assert bool(((got - want[:, :, None]).abs() <= room[:, :, None]).all())


def latent_shares(n, most, dim, vdim):
    h = 16
    spans = [(most - 1 - i * (most - 3) // n, 1) for i in range(n)]
    blocks = sum(f // BS + 1 for f, _ in spans)
    batch = make_batch(spans, blocks)
    q = rand(n, h * dim, seed=1, dtype=BF16, scale=2.0)
    cache = rand(blocks, 1, BS, dim, seed=2, dtype=BF16)
    on = cache.cuda()
    got = ops.attn_ctx(q.cuda(), None, on, on[..., :vdim], None,
                       on_gpu(batch), dim ** -0.5).view(n, h, vdim)
    for e, (first, _) in enumerate(spans):
        k = cache[batch.block_table[e].long(), 0].reshape(-1, dim)[:first + 1]
        s = q[e].view(h, dim).double() @ k.double().T * dim ** -0.5
        want = torch.softmax(s, 1) @ k[:, :vdim].double()
        room = 2.0 ** -8 * want.abs() + 2.0 ** -13 * 4 * want.abs().amax()
        assert bool(((got[e].cpu().double() - want).abs() <= room).all())


# Contexts in shares whose number is no power of two, some without a step
@pytest.mark.parametrize("n,most", [(1, 450), (19, 900), (37, 700), (85, 450),
                                    (129, 300)])
def test_latent_shares(n, most):
    latent_shares(n, most, 192, 128)


# Keys that leave a CU room for two workgroups, with four shares, and larger ones: three
# shares of contexts with a round and a half of workgroups, the most shares
@pytest.mark.parametrize("n,most,dim,vdim", [
    (120, 1300, 72, 64), (130, 960, 320, 256), (130, 900, 576, 512),
    (1, 2800, 576, 512)])
def test_latent_shares_by_size(n, most, dim, vdim):
    latent_shares(n, most, dim, vdim)
