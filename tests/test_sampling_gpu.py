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


@pytest.mark.parametrize("temp", [0.6, 0.7, 0.9, 1.3])
@pytest.mark.parametrize("vocab", [3000, 20000])
def test_equal_once_scaled(temp, vocab):
    """One token asked for is the larger of two logits that are a unit of the
    last place apart, also where they are equal once scaled and rounded."""
    n = 64
    g = torch.Generator().manual_seed(1)
    low = torch.rand(n, generator=g) * 25 + 5
    top = torch.nextafter(low, torch.tensor(100.0))
    inv = 1 / torch.tensor(temp)
    assert int((low * inv == top * inv).sum()) > 0
    rows = torch.full((n, vocab), -100.0)
    rows[:, 17], rows[:, 2500] = low, top
    of = lambda v, **how: torch.full((n,), v, device=DEV, **how)
    for u in 0.0, 0.25, 0.75:
        got = ops.softmax_sample(rows.to(DEV), of(temp),
                                 of(1, dtype=torch.int32), of(1.0), of(u))
        assert got.tolist() == [2500] * n


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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("k", [1, 5, 40])
@pytest.mark.parametrize("top", [0.0, -0.0, -1e-6, 1e-6])
def test_largest_logit_next_to_zero(top, k, dtype):
    """Log-probabilities of an all but certain token, rows less their largest:
    the number after the largest logit weighs 1 as well."""
    n, vocab = 64, 32000
    g = torch.Generator().manual_seed(k)
    x = torch.randn(n, vocab, generator=g).to(dtype)
    at = x.float().argmax(1, keepdim=True)
    x = (x.float() - x.float().gather(1, at)).to(dtype)
    x[x == 0] = -0.5                        # equals of the largest
    x.scatter_(1, at, top)
    u = torch.rand(n, generator=g)
    of = lambda v: torch.full((n,), v, device=DEV)
    for p in (1.0, 0.5):
        got = ops.softmax_sample(x.to(DEV), of(0.8), of(k).int(), of(p),
                                 u.to(DEV)).tolist()
        for i in range(n):
            keep, cum, goal = draw(x[i], 0.8, k, p, float(u[i]))
            a = got[i]
            slack = 2e-5 * float(cum[-1])   # as above
            assert bool(keep[a])
            assert float(cum[a]) >= float(goal) - slack
            assert a == 0 or float(cum[a - 1]) <= float(goal) + slack


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("vocab", [32000, 39936])
def test_number_between_a_run_and_its_edge(vocab, dtype):
    """Weights that vanish one by one beside all before them, but not their sum:
    a number that falls to it stands for one of them, not for the row's last
    token. Runs are 256 of equal length."""
    run = (vocab + 255) // 256
    at = 200 * run                  # a weight of 1 each, so sums are exact
    x = torch.zeros(1, vocab)
    x[:, at:at + run] = -7.25       # 7e-4 each, of 2^-9 = 0.002 a step of sums
    x[:, at + run - 3:at + run] = -torch.inf
    x[:, at + run:] = -torch.inf
    x[:, -50:] = 0.0
    w = torch.exp(x.double())
    z = float(w.sum())
    # from 25000 on, and to 32768, a step of 32-bit sums is 2^-9; a number's own
    # is 2^-24 of them
    for part in (0.3, 0.5, 0.7):
        goal = at + part * float(w[0, at:at + run].sum())
        got = ops.softmax_sample(
            x.to(dtype).to(DEV), torch.ones(1, device=DEV),
            torch.zeros(1, device=DEV).int(), torch.ones(1, device=DEV),
            torch.tensor([goal / z], device=DEV))
        assert at <= int(got) < at + run - 3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_number_at_the_last_edge(dtype):
    """Stands for the last token that has a weight."""
    x = torch.full((1, 1000), -torch.inf)
    x[0, :700] = torch.randn(700, generator=torch.Generator().manual_seed(0))
    got = ops.softmax_sample(
        x.to(dtype).to(DEV), torch.ones(1, device=DEV),
        torch.zeros(1, device=DEV).int(), torch.ones(1, device=DEV),
        torch.full((1,), 2.0, device=DEV))
    assert int(got) == 699


@pytest.mark.parametrize("k", [1, 509, 510, 511, 512, 513, 600])
@pytest.mark.parametrize("p", [1.0, 0.3, 0.9999])
def test_thresholds_at_the_last_key_that_is_counted(k, p):
    """One token for each of the numbers from 4 down, among others far below:
    thresholds a little before and behind the 512th of them."""
    n, vocab = 16, 9000
    g = torch.Generator().manual_seed(k)
    x = torch.full((n, vocab), -30.0).bfloat16()
    bits = torch.tensor(4.0).bfloat16().view(torch.int16) - \
        torch.arange(700, dtype=torch.int16)
    at = torch.rand(n, vocab, generator=g).argsort(1)[:, :700]
    x.scatter_(1, at, bits.view(torch.bfloat16).expand(n, -1))
    x[::4, at[0, 0]] = -torch.inf
    u = torch.rand(n, generator=g)
    of = lambda v: torch.full((n,), v, device=DEV)
    got = ops.softmax_sample(x.to(DEV), of(0.8), of(k).int(), of(p),
                             u.to(DEV)).tolist()
    for i in range(n):
        keep, cum, goal = draw(x[i], 0.8, k, p, float(u[i]))
        a = got[i]
        slack = 2e-5 * float(cum[-1])
        assert bool(keep[a])
        assert float(cum[a]) >= float(goal) - slack
        assert a == 0 or float(cum[a - 1]) <= float(goal) + slack


def test_largest_of_rows_that_are_not_usual():
    """The first of equals, zeros of either sign; NaN of either sign, infinities
    and rows of nothing else beside usual ones."""
    vocab = 20000
    x = torch.full((8, vocab), -3.0)
    x[0, 700], x[0, 15000] = -0.0, 0.0
    x[1, 700], x[1, 15000] = 0.0, -0.0
    x[2, 5], x[2, 9], x[2, 19999] = torch.nan, 7.0, 7.0
    x[3, 5], x[3, 9] = -torch.nan, 2.0
    x[4, 12345] = torch.inf
    x[5] = -torch.inf
    x[6] = torch.nan
    x[7] = -torch.inf
    x[7, 19998] = -2e38
    x = x.bfloat16().to(DEV)
    zeros = torch.zeros(8, device=DEV)
    got = ops.softmax_sample(x, zeros, zeros.int(), zeros + 1, zeros)
    assert got.tolist() == [700, 700, 9, 9, 12345, 0, 0, 19998]
    # and as a draw that leaves one token
    got = ops.softmax_sample(x, zeros + 1, zeros.int() + 1, zeros + 1,
                             zeros + 0.5)
    # (all of a row are equal where all are -inf, and none is a token of NaN)
    assert got[2] in (9, 19999)
    assert got[3:].tolist() == [9, 12345, 10000, 0, 19998]
    assert got[0] in (700, 15000) and got[1] in (700, 15000)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("vocab", [1000, 9000, 32000])
@pytest.mark.parametrize("k,p", [(0, 1.0), (40, 1.0), (0, 0.9), (600, 0.3)])
def test_infinite_temperature(vocab, dtype, k, p):
    """All tokens but those of -inf, which are none whatever the temperature:
    in masked rows and past a row's end."""
    n = 16
    g = torch.Generator().manual_seed(vocab)
    x = (torch.randn(n, vocab, generator=g) * 3).to(dtype)
    x[1::2, ::7] = -torch.inf
    x[2::4, vocab // 3:] = -torch.inf
    u = torch.rand(n, generator=g)
    of = lambda v: torch.full((n,), v, device=DEV)
    got = ops.softmax_sample(x.to(DEV), of(torch.inf), of(k).int(), of(p),
                             u.to(DEV)).tolist()
    for i in range(n):
        keep, cum, goal = draw(x[i], torch.inf, k, p, float(u[i]))
        # equal weights: whole numbers, and a number that is rounded once
        assert bool(keep[got[i]])
        assert float(cum[got[i]]) >= float(goal) * (1 - 1e-6)
        assert float(cum[got[i]]) <= float(goal) * (1 + 1e-6) + 1
