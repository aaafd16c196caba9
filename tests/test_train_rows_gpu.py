"""A training step's row work on the GPU against 64 bits: widths around the
vectors a thread holds, rows around the workgroups of a launch."""

import pytest
import torch
import torch.nn.functional as F

from substratus_amd.ops import train

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rand(*shape, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed + sum(shape))
    return torch.randn(*shape, device=DEV, generator=g).bfloat16()


def near(got, want, terms):
    """Two bf16 steps of the result, and 32-bit sums over `terms`."""
    room = 2.0 ** -7 * want.abs() + 2.0 ** -18 * terms
    assert got.dtype == torch.bfloat16
    assert bool(((got.double() - want).abs() <= room).all()), \
        float(((got.double() - want).abs() / room).max())


@pytest.mark.parametrize("rms", [True, False])
@pytest.mark.parametrize("n", [0, 1, 2])
@pytest.mark.parametrize("rows,width", [(1, 8), (513, 768), (3, 2048),
                                        (1030, 2056), (514, 4544),
                                        (511, 8192)])
def test_add_norm(rows, width, n, rms):
    h, *ds = (rand(rows, width, seed=i).requires_grad_() for i in range(n + 1))
    w = (1 + 0.5 * rand(width, seed=7)).detach().requires_grad_()
    b = None if rms else rand(width, seed=8).requires_grad_()
    gy, gs = rand(rows, width, seed=9), rand(rows, width, seed=10)
    y, total = train.add_norm(h, ds, w, b, 1e-5)
    exact = h.detach()
    for d in ds:
        exact = exact + d.detach()
    assert torch.equal(total, exact)
    inputs = [t for t in (h, w, b, *ds) if t is not None]
    got = torch.autograd.grad([y, total], inputs, [gy, gs])

    x, w64 = exact.double().requires_grad_(), w.detach().double()
    w64.requires_grad_()
    b64 = None if rms else b.detach().double().requires_grad_()
    want = (F.rms_norm(x, (width,), w64, 1e-5) if rms
            else F.layer_norm(x, (width,), w64, b64, 1e-5))
    near(y, want.detach(), 1 + want.abs().max())
    leaves = [t for t in (x, w64, b64) if t is not None]
    dx, *dp = torch.autograd.grad(want, leaves, gy.double())
    # the norm's gradient may cancel against the residual's
    size = gs.abs().double() + dx.abs()
    for g in (got[0], *got[len(leaves):]):
        near(g, dx + gs.double(), 2.0 ** 10 * size + width)
    for g, p in zip(got[1:], dp):
        near(g, p, 4.0 * rows)


def test_add_norm_again():
    """Only one of the results used, gradients that are no rows, gradients of
    gradients."""
    w, b, h, d = (rand(*s).requires_grad_()
                  for s in ((64,), (64,), (5, 64), (5, 64)))
    y, total = train.add_norm(h, (d,), w, b, 1e-5)
    g, = torch.autograd.grad(total.sum(), h, retain_graph=True)
    assert bool((g == 1).all())
    torch.autograd.grad(y.sum(), (h, w, b, d), retain_graph=True)
    want = train._norm(h + d, w, b, 1e-5)
    pair = []
    for out in (y, want):
        first, = torch.autograd.grad(out.float().square().sum(), h,
                                     create_graph=True)
        pair.append(torch.autograd.grad(first.float().square().sum(),
                                        (w, d)))
    for a, c in zip(*pair):
        assert torch.allclose(a, c, rtol=2.0 ** -4, atol=0.5)


@pytest.mark.parametrize("b,s,hq,hkv,d", [(1, 1, 1, 1, 64), (2, 33, 71, 1, 64),
                                          (3, 50, 4, 2, 128)])
@pytest.mark.parametrize("turned", [True, False])
def test_attend(b, s, hq, hkv, d, turned):
    qkv = rand(b, s, (hq + 2 * hkv) * d).requires_grad_()
    cos = sin = None
    if turned:
        a = torch.arange(s, device=DEV)[:, None] * 0.9 ** torch.arange(
            d // 2, device=DEV)
        cos, sin = a.cos(), a.sin()
    dout = rand(b, s, hq * d, seed=1)
    got = [train.attend(qkv, cos, sin, hq, hkv, d ** -0.5)]
    got += torch.autograd.grad(got[0], qkv, dout)
    q64 = qkv.detach().double().cpu().requires_grad_()
    turns = (None, None) if not turned else (cos.double().cpu(),
                                             sin.double().cpu())
    want = [train._attend(q64, *turns, hq, hkv, d ** -0.5)]
    want += torch.autograd.grad(want[0], q64, dout.double().cpu())
    # the general form rounds in the same places and more
    other = [train._attend(qkv, cos, sin, hq, hkv, d ** -0.5)]
    other += torch.autograd.grad(other[0], qkv, dout)
    for g, w, o in zip(got, want, other):
        size = w.norm()
        off, most = ((t.double().cpu() - w).norm() / size for t in (g, o))
        assert off <= 1.02 * most + 2.0 ** -12


@pytest.mark.parametrize("b,s,hq,hkv,d", [(2, 33, 4, 1, 64),
                                          (1, 20, 2, 2, 128)])
@pytest.mark.parametrize("turned", [True, False])
@pytest.mark.parametrize("fused", [True, False])
def test_attend_again(b, s, hq, hkv, d, turned, fused):
    """Gradients of gradients, and batches of gradients, of the attention and
    of what is around it."""
    qkv = rand(b, s, (hq + 2 * hkv) * d).requires_grad_()
    dout = rand(b, s, hq * d, seed=1).requires_grad_()
    cos = sin = None
    if turned:
        a = torch.arange(s, device=DEV)[:, None] * 0.9 ** torch.arange(
            d // 2, device=DEV)
        cos, sin = a.cos(), a.sin()
    form = train.attend if fused else train._attend

    def twice(form, qkv, dout, cos, sin):
        out = form(qkv, cos, sin, hq, hkv, d ** -0.5)
        one, = torch.autograd.grad(out, qkv, dout, create_graph=True)
        weigh = torch.linspace(-1, 1, one.numel(), device=one.device)
        return one, *torch.autograd.grad(
            (one * weigh.view_as(one).to(one.dtype)).float().square().sum(),
            (qkv, dout))

    def exact(qkv, cos, sin, hq, hkv, scale):
        q, k, v = (t.view(b, s, -1, d).transpose(1, 2) for t in qkv.split(
            [hq * d, hkv * d, hkv * d], -1))
        if cos is not None:
            q, k = train.rope(q, cos, sin), train.rope(k, cos, sin)
        k, v = (t.repeat_interleave(hq // hkv, 1) for t in (k, v))
        later = torch.ones(s, s, dtype=torch.bool).triu(1)
        a = (q @ k.mT * scale).masked_fill(later, -torch.inf).softmax(-1) @ v
        return a.transpose(1, 2).reshape(b, s, hq * d)

    got = twice(form, qkv, dout, cos, sin)
    want = twice(exact, *(t if t is None else
                          t.detach().double().cpu().requires_grad_(
                              t.requires_grad)
                          for t in (qkv, dout, cos, sin)))
    for g, w in zip(got, want):     # bf16 between the steps
        g, w = g.detach().double().cpu(), w.detach()
        assert float((g - w).norm()) <= 0.03 * float(w.norm())
    out = form(qkv, cos, sin, hq, hkv, d ** -0.5)
    many = torch.stack([dout.detach(), 2 * dout.detach()])
    both, = torch.autograd.grad(out, qkv, many, is_grads_batched=True,
                                retain_graph=True)
    alone, = torch.autograd.grad(out, qkv, dout)
    for i in range(2):
        assert float((both[i].float() - (i + 1) * alone.float()).norm()) <= \
            0.02 * float((i + 1) * alone.float().norm())


@pytest.mark.parametrize("rows,f", [(1, 8), (3, 2056), (700, 5632)])
def test_silu_mul(rows, f):
    x = (4 * rand(rows, 2 * f)).detach().requires_grad_()
    dy = rand(rows, f, seed=3)
    y = train.silu_mul(x)
    dx, = torch.autograd.grad(y, x, dy)
    x64 = x.detach().double().requires_grad_()
    want = train._silu_mul(x64)
    dw, = torch.autograd.grad(want, x64, dy.double())
    near(y, want.detach(), want.detach().abs())
    # the slope is a difference of terms near 1 around its zero
    near(dx, dw, torch.cat([x.detach()[:, f:] * dy, dy], 1).abs().double()
         * 16)


@pytest.mark.parametrize("n,rows,width", [(1, 5, 8), (255, 3, 64),
                                          (257, 1000, 2056), (3000, 40, 2048),
                                          (8192, 9, 72), (700, 5000, 8192)])
def test_lookup(n, rows, width):
    """Numbers that come once, often and on both sides of a workgroup."""
    torch.manual_seed(n)
    table = torch.nn.Embedding(rows, width, device=DEV,
                               dtype=torch.bfloat16)
    tokens = torch.randint(rows, (2, n), device=DEV)[:, :(n + 1) // 2]
    out = train.lookup(tokens, table)
    assert out.grad_fn.name().startswith("_Lookup")
    assert torch.equal(out, table(tokens))
    dy = rand(*out.shape, seed=2)
    got, = torch.autograd.grad(out, table.weight, dy)
    want = torch.zeros(rows, width, device=DEV, dtype=torch.float64)
    size = want.clone()
    flat = dy.reshape(-1, width).double()
    want.index_add_(0, tokens.reshape(-1), flat)
    size.index_add_(0, tokens.reshape(-1), flat.abs())
    near(got, want, size)
    assert torch.equal(got, torch.autograd.grad(
        train.lookup(tokens, table), table.weight, dy)[0])
    table.register_forward_hook(lambda *a: None)
    assert not train.lookup(tokens, table).grad_fn.name().startswith(
        "_Lookup")


@pytest.mark.parametrize("width", [8, 72, 2056])
def test_lookup_of_frequent_numbers(width):
    """Numbers that come as often as one workgroup takes, and once more; a
    number behind a workgroup's reach of others; one alone."""
    g = torch.Generator().manual_seed(width)
    counts = torch.tensor([31, 32, 33, 64, 65, 0, 1, 300, 257, 2])
    for tokens in (torch.arange(10).repeat_interleave(counts),
                   torch.arange(10).repeat_interleave(counts)[
                       torch.randperm(785, generator=g)],
                   torch.tensor([3] * 700), torch.tensor([9] * 8192)):
        tokens = tokens.to(DEV)
        table = torch.nn.Embedding(10, width, device=DEV,
                                   dtype=torch.bfloat16)
        out = train.lookup(tokens, table)
        assert out.grad_fn.name().startswith("_Lookup")
        dy = rand(len(tokens), width, seed=2)
        got, = torch.autograd.grad(out, table.weight, dy)
        want, size = (torch.zeros(10, width, device=DEV, dtype=torch.float64)
                      .index_add_(0, tokens, t) for t in (
                          dy.double(), dy.double().abs()))
        near(got, want, size)
        assert torch.equal(got, torch.autograd.grad(
            train.lookup(tokens, table), table.weight, dy)[0])
