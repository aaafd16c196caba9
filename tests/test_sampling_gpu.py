"""The sampling kernel against 64 bits: which tokens may be drawn, and which
one a number in [0, 1) stands for, at sizes where its rounds and loads end."""

import pytest
import torch

from substratus_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def draw(logits, t, k, p, u):
    """(tokens that may be drawn, cumulated weights in token order, draw)."""
    x = logits.double() / t
    x = x.nan_to_num(nan=-torch.inf, posinf=torch.inf, neginf=-torch.inf)
    w = torch.where(x == x.max(), 1.0, torch.exp(x - x.max()))
    keep = ~logits.isnan()
    if 0 < k < len(x):      # equals go together, the largest in any case
        below = x.topk(k + 1).values[-1]
        keep &= (x > below) | (x == x.max())
    if 0 < p < 1:
        goal = p * w[keep].sum()
        by_size, at = w.masked_fill(~keep, 0).sort(descending=True)
        n = int((by_size.cumsum(0) < goal * (1 - 1e-6)).sum())
        keep &= w >= by_size[min(n, len(x) - 1)] * (1 - 1e-9)
    w = w.masked_fill(~keep, 0)
    return keep, w.cumsum(0), u * w.sum()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("vocab", [1, 7, 8, 1000, 8191, 8192, 8200, 32769,
                                   39936, 50257, 57352, 79872])
def test_draws(vocab, dtype):
    if vocab * dtype.itemsize > 156 * 1024:
        pytest.skip("refused: larger than a workgroup's memory")
    torch.manual_seed(vocab)
    settings = [(1.0, 0, 1.0), (0.7, 1, 1.0), (0.9, 40, 1.0), (1.3, 0, 0.9),
                (0.5, 30, 0.5), (1.0, vocab - 1, 0.999), (2.0, 5000, 0.3)]
    n = 8 * len(settings)
    logits = (torch.randn(n, vocab, device=DEV) * 3).to(dtype)
    u = torch.rand(n, device=DEV)
    u[0], u[1] = 0.0, 1.0 - 2.0 ** -24
    t, k, p = (torch.tensor([settings[i % len(settings)][j]
                             for i in range(n)], device=DEV)
               for j in range(3))
    got = ops.softmax_sample(logits, t, k.int(), p, u).tolist()
    for i in range(n):
        keep, cum, goal = draw(logits[i].cpu(), float(t[i]), int(k[i]),
                               float(p[i]), float(u[i]))
        a = got[i]
        assert 0 <= a < vocab and bool(keep[a])
        # 32-bit sums of weights: 2^-24 per addend, of which a thread has at
        # most 80 in a row and partial sums a few hundred
        slack = 2e-5 * float(cum[-1])
        assert float(cum[a]) >= float(goal) - slack
        assert a == 0 or float(cum[a - 1]) <= float(goal) + slack


def test_rows_that_are_not_ordinary():
    """The smallest index of several largest; NaN and -inf are never drawn;
    an infinite logit always is; rows of one value."""
    v = 20000
    rows = torch.randn(6, v, device=DEV).bfloat16()
    rows[0, 5000] = rows[0, 12345] = 50.0
    rows[1] = -torch.inf
    rows[1, 17] = 1.0
    rows[2, ::2] = torch.nan
    rows[3, 777] = torch.inf
    rows[4] = 3.0
    rows[5, 1:] = -torch.inf
    for temp in (0.0, 0.8):
        t = torch.full((6,), temp, device=DEV)
        for k, p in ((0, 1.0), (3, 1.0), (0, 0.5)):
            got = ops.softmax_sample(
                rows, t, torch.full((6,), k, device=DEV).int(),
                torch.full((6,), p, device=DEV),
                torch.full((6,), 0.4, device=DEV)).tolist()
            assert got[0] == 5000 if temp == 0 else got[0] in (5000, 12345)
            assert got[1] == 17 and got[2] % 2 == 1 and got[3] == 777
            assert got[5] == 0
            if temp == 0:
                assert got[4] == 0
            elif p == 1:
                assert abs(got[4] - 0.4 * v) <= 1


@pytest.mark.parametrize("k,p", [(0, 1.0), (2, 1.0), (0, 0.9)])
@pytest.mark.parametrize("temp", [0.6, 0.7, 0.9, 1.3])
def test_neighbouring_numbers_share_the_draws(temp, k, p):
    """Two logits a unit of the last place apart weigh the same but for 1e-6,
    also where they are equal once divided by the temperature."""
    n, vocab = 64, 3000
    g = torch.Generator().manual_seed(1)
    low = torch.rand(n, generator=g) * 25 + 5
    top = torch.nextafter(low, torch.tensor(100.0))
    assert int((low * (1 / torch.tensor(temp)) ==
                top * (1 / torch.tensor(temp))).sum()) > 0
    rows = torch.full((n, vocab), -100.0)
    first, second = 17, 2500
    odd = torch.arange(n) % 2 == 1
    rows[:, first] = torch.where(odd, top, low)
    rows[:, second] = torch.where(odd, low, top)
    of = lambda v, **how: torch.full((n,), v, device=DEV, **how)
    for u, token in ((0.25, first), (0.75, second)):
        got = ops.softmax_sample(rows.to(DEV), of(temp),
                                 of(k, dtype=torch.int32), of(p), of(u))
        assert got.tolist() == [token] * n


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("k,p", [(3, 1.0), (200, 1.0), (0, 0.6), (500, 0.97)])
@pytest.mark.parametrize("kind", ["close", "equal", "steps", "below zero"])
def test_thresholds_among_like_weights(dtype, k, p, kind):
    """Many logits that share their upper 16 bits, or all of them, where a
    threshold lies: more, and fewer, than are sorted out at once."""
    n, vocab = 24, 9000
    g = torch.Generator().manual_seed(k + vocab)
    x = torch.randn(n, vocab, generator=g)
    if kind == "close":
        x = 4 + x * 1e-3
    elif kind == "equal":
        x = torch.where(torch.rand(n, vocab, generator=g) < 0.01, 5.0, 3.0)
    elif kind == "steps":
        # a step's 1000 to 3600 tokens are 3e-5 apart, some 2^-20 of a logit
        # near 4: weights of 32 bits still differ. (At 1e-4 a step they are
        # not all told apart, and a threshold takes or leaves several.)
        x = (x * 2).round() + torch.rand(n, vocab, generator=g) * 0.1
    else:
        x = -x.abs() * 8 - 0.1
    x = x.to(dtype)
    u = torch.rand(n, generator=g)
    of = lambda v: torch.full((n,), v, device=DEV)
    got = ops.softmax_sample(x.to(DEV), of(0.9), of(k).int(), of(p),
                             u.to(DEV)).tolist()
    for i in range(n):
        keep, cum, goal = draw(x[i], 0.9, k, p, float(u[i]))
        a = got[i]
        # as above; a step of the sums may take or leave a weight at the edge
        slack = 2e-5 * float(cum[-1])
        assert bool(keep[a])
        assert float(cum[a]) >= float(goal) - slack
        assert a == 0 or float(cum[a - 1]) <= float(goal) + slack
