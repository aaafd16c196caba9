"""Products of many rows (tile_gemm.hip) against 64 bits: either operand
flipped, at the ends of tiles, of steps of 64 of the inner dimension and of
their pairs, with tiles that are left over from a round."""

import pytest
import torch

from substratus_amd import _C, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def close(got, a, b, bias=None):
    """Half a bf16 step (2^-9), and 32-bit sums in any order (2^-18 of the sum
    of magnitudes for some thousands of addends)."""
    want = a.double() @ b.double().T
    room = 2.0 ** -18 * (a.double().abs() @ b.double().abs().T)
    if bias is not None:
        want = want + bias.double()
    assert got.dtype == torch.bfloat16 and got.shape == want.shape
    off = (got.double() - want).abs()
    assert bool((off <= 2.0 ** -8 * want.abs() + room + 1e-30).all())


def operand(rows, k, flipped, pad):
    shape = (k, rows) if flipped else (rows, k)
    whole = torch.full((shape[0], shape[1] + pad), torch.nan, device=DEV)
    whole[:, :shape[1]] = torch.randn(shape, device=DEV)
    return whole.bfloat16()[:, :shape[1]]       # what is beside is no number


# the inner dimension: two steps at least; within a pair, whole, one over
@pytest.mark.parametrize("k", [72, 128, 136, 192, 248, 1096])
@pytest.mark.parametrize("m,n", [(256, 256), (264, 256), (256, 1000),
                                 (776, 520)])
@pytest.mark.parametrize("fa", [False, True])
@pytest.mark.parametrize("fb", [False, True])
def test_tile_gemm(m, n, k, fa, fb):
    torch.manual_seed(m + n + k)
    inner = k + 3 if fa and fb else k           # lines of any number
    a, b = operand(m, inner, fa, 8), operand(n, inner, fb, 16)
    bias = torch.randn(n, device=DEV).bfloat16() if k % 3 == 0 else None
    got = _C.tile_gemm(a, b, bias, fa, fb)
    close(got, a.T if fa else a, b.T if fb else b, bias)


@pytest.mark.parametrize("m,n,k,fa,fb", [
    (1000, 1024, 4544, False, False),           # all shared
    (4360, 4104, 1032, False, True),            # a round, and some
    (2304, 8192, 520, True, True)])
def test_rounds(m, n, k, fa, fb):
    a, b = operand(m, k, fa, 0), operand(n, k, fb, 0)
    got = _C.tile_gemm(a, b, None, fa, fb)
    close(got, a.T if fa else a, b.T if fb else b)
    assert torch.equal(got, _C.tile_gemm(a, b, None, fa, fb))


@pytest.mark.parametrize("m,f,k", [(256, 128, 72), (300, 136, 192),
                                   (1000, 512, 4544), (4360, 2056, 1032)])
@pytest.mark.parametrize("bias", [False, True])
def test_gated(m, f, k, bias):
    torch.manual_seed(m)
    a = operand(m, k, False, 8)
    b = (operand(2 * f, k, False, 0) / k ** 0.5).bfloat16()
    bs = torch.randn(2 * f, device=DEV).bfloat16() if bias else None
    got = _C.tile_gemm(a, b, bs, False, False, True)
    y = a.double() @ b.double().T + (0 if bs is None else bs.double())
    g, u = y.chunk(2, 1)
    want = torch.nn.functional.silu(g) * u
    # half a step of the result; 32-bit sums before, slopes of at most 1.1
    room = 2.0 ** -17 * (g.abs() + 1) * (u.abs() + 1)
    assert bool(((got.double() - want).abs() <=
                 2.0 ** -8 * want.abs() + room).all())


def gated_close(got, a, b):
    g, u = (a.double() @ b.double().T).chunk(2, 1)
    want = torch.nn.functional.silu(g) * u
    room = 2.0 ** -17 * (g.abs() + 1) * (u.abs() + 1)   # as in test_gated
    assert bool(((got.double() - want).abs() <=
                 2.0 ** -8 * want.abs() + room).all())


# Tiles of fewer rows, the last one of a few rows, or of all but one or eight: the first
# numbers of rows, of columns, that are cut into such tiles.
@pytest.mark.parametrize("height", [128, 160, 192, 224])
@pytest.mark.parametrize("over", [5, -1])
@pytest.mark.parametrize("k", [2120, 4168])
@pytest.mark.parametrize("kind", ["plain", "gelu", "gated", "b", "both"])
def test_heights(height, over, k, kind):
    torch.manual_seed(height + k)
    fa, fb = kind == "both", kind in ("b", "both")
    by = 8 if fa else 1
    m, n = next(((m, n) for m in range(3 * height + by * over, 8192, height)
                 for n in (1296, 3600, 4560, 9232)
                 if _C.tile_gemm_rows(m, n, k, fa, fb) == height), (0, 0))
    if m == 0:
        assert (kind, height, over) == ("b", 224, 5)
        pytest.skip("cut into other tiles")
    a, b = operand(m, k, fa, 8), operand(n, k, fb, 8)
    if kind in ("gelu", "gated"):
        b = (b / k ** 0.5).bfloat16()
    bias = torch.randn(n, device=DEV).bfloat16() if kind == "plain" else None
    got = _C.tile_gemm(a, b, bias, fa, fb, kind == "gated", kind == "gelu")
    if kind == "gated":
        gated_close(got, a, b)
    elif kind == "gelu":
        assert torch.equal(got, ops.gelu(_C.tile_gemm(a, b, None, fa, fb)))
    else:
        close(got, a.T if fa else a, b.T if fb else b, bias)


# Tiles of 224 rows of a flipped b whose last one begins early: sizes that are none of
# test_heights'
@pytest.mark.parametrize("m,n,k", [(264, 5544, 1096), (264, 9504, 2120)])
def test_last_tile_of_a_flipped_b(m, n, k):
    torch.manual_seed(n)
    assert _C.tile_gemm_rows(m, n, k, False, True) == 224
    a, b = operand(m, k, False, 8), operand(n, k, True, 8)
    close(_C.tile_gemm(a, b, None, False, True), a, b.T)


def test_rows_of_any_number():
    """Rows that are not flipped need not come in eights."""
    a, b = operand(321, 192, False, 0), operand(264, 192, False, 0)
    close(_C.tile_gemm(a, b, None, False, False), a, b)


@pytest.mark.parametrize("bias", [False, True])
def test_linear_gradients(bias):
    """ops.linear at a size where all three products pay."""
    torch.manual_seed(5)
    t, k, n = 2082, 11008, 4096
    assert all(_C.tile_gemm_good(*s, False) for s in (
        (2 * t, n, k, k, k, False, False), (2 * t, k, n, n, k, False, True),
        (n, k, 2 * t, n, k, True, True)))
    x = torch.randn(2, t, k, device=DEV).bfloat16().requires_grad_()
    w = (torch.randn(n, k, device=DEV) / 64).bfloat16().requires_grad_()
    bs = torch.randn(n, device=DEV).bfloat16().requires_grad_() \
        if bias else None
    y = ops.linear(x, w, bs)
    dy = torch.randn(2, t, n, device=DEV).bfloat16()
    rows, drows = x.detach().view(-1, k), dy.view(-1, n)
    close(y.detach().view(-1, n), rows, w.detach(),
          None if bs is None else bs.detach())
    inputs = [t for t in (x, w, bs) if t is not None]
    got = torch.autograd.grad(y, inputs, dy, retain_graph=True)
    close(got[0].view(-1, k), drows, w.detach().T)
    close(got[1], drows.T, rows.T)
    if bias:
        assert torch.equal(got[2], drows.sum(0))
    # gradients that are no rows, and gradients of gradients
    g, = torch.autograd.grad(y.sum(), x, retain_graph=True)
    close(g.view(-1, k), torch.ones_like(drows), w.detach().T)
    first, = torch.autograd.grad(y, x, dy, create_graph=True)
    again, = torch.autograd.grad(first.float().sum(), w)
    want = torch.nn.functional.linear(x, w, bs)
    first, = torch.autograd.grad(want, x, dy, create_graph=True)
    assert torch.equal(again, torch.autograd.grad(first.float().sum(), w)[0])
