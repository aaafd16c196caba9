"""Products of 17 to 64 rows with thin matrices (rows_gemm.hip) against 64
bits, where their tiles of rows, stages and shares of the inner dimension
end."""

import pytest
import torch

from substratus_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def test_where_it_pays():
    for rows, n, k, want in ((16, 1 << 17, 1 << 14, True),
                             (17, 4096, 4096, True), (32, 4096, 4096, True),
                             (33, 4096, 4096, False), (17, 4097, 64, False),
                             (17, 16, 4128, False), (64, 4096, 2048, True),
                             (65, 16, 32, False), (33, 16, 2080, False)):
        assert ops._rows_gemm_pays(rows * k, n, k) == want


# two to four tiles of 16 rows, partly filled; two stages of 64 columns in
# flight for each of four waves: fewer chunks of 32 than waves, half stages, a
# full ring, more than one round
@pytest.mark.parametrize("m", [17, 31, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("k", [32, 96, 160, 544, 2048])
@pytest.mark.parametrize("n", [16, 55, 768])
@torch.no_grad()
def test_rows(m, n, k):
    torch.manual_seed(m * 10000 + n + k)
    w = torch.randn(n, k, device=DEV).bfloat16()
    x = torch.randn(m, k + 64, device=DEV).bfloat16()[:, 32:32 + k]
    b = torch.randn(n, device=DEV).bfloat16()
    assert ops._few_rows(x, w, b, False) is not None
    # half a bf16 step of the result, and 32-bit sums whose order is free:
    # 2^-24 per addend of a wave's share, errors that partly cancel
    prod = x.double() @ w.double().T
    room = 2.0 ** -18 * (x.double().abs() @ w.double().abs().T)
    for bias in (None, b):
        want = prod if bias is None else prod + bias.double()
        off = (ops.linear(x, w, bias).double() - want).abs()
        assert bool((off <= 2.0 ** -8 * want.abs() + room + 1e-30).all())
    y = ops.linear_gated(x, w)
    assert (y is None) == (n % 16 != 0)
    if y is not None:
        g, u = prod.chunk(2, 1)
        rg, ru = room.chunk(2, 1)
        want = torch.nn.functional.silu(g) * u
        # a gate's error reaches the product by silu's slope, at most 1.1
        off = (y.double() - want).abs()
        assert bool((off <= 2.0 ** -8 * want.abs() + 1e-6
                     + 1.1 * (rg * u.abs() + ru * g.abs())).all())


# where matrices are wide or inner sizes long: the last that go here, and the
# first that go elsewhere
@pytest.mark.parametrize("m,n,k", [(48, 4096, 4096), (49, 4096, 3072),
                                   (64, 1024, 4096), (48, 8192, 2048),
                                   (49, 8192, 1024), (32, 12288, 2048),
                                   (32, 6160, 3072), (32, 6160, 4096)])
@torch.no_grad()
def test_larger(m, n, k):
    for rows, cols, inner in ((m, n, k), (m + 1, n, k), (m, n + 16, k),
                              (m, n, k + 32)):
        torch.manual_seed(rows + cols + inner)
        w = torch.randn(cols, inner, device=DEV).bfloat16()
        x = torch.randn(rows, inner, device=DEV).bfloat16()
        prod = x.double() @ w.double().T
        room = 2.0 ** -18 * (x.double().abs() @ w.double().abs().T)
        off = (ops.linear(x, w).double() - prod).abs()
        assert bool((off <= 2.0 ** -8 * prod.abs() + room + 1e-30).all())
        y = ops.linear_gated(x * 0.03125, w)
        if y is not None:
            g, u = (prod * 0.03125).chunk(2, 1)
            rg, ru = (room * 0.03125).chunk(2, 1)
            want = torch.nn.functional.silu(g) * u
            off = (y.double() - want).abs()
            assert bool((off <= 2.0 ** -8 * want.abs() + 1e-6
                         + 1.1 * (rg * u.abs() + ru * g.abs())).all())


@pytest.mark.parametrize("m,hq,hkv,d,k", [(17, 2, 1, 16, 32),
                                          (40, 4, 2, 128, 160),
                                          (64, 3, 1, 64, 2048)])
@torch.no_grad()
def test_heads(m, hq, hkv, d, k):
    torch.manual_seed(m)
    w = (torch.randn((hq + 2 * hkv) * d, k, device=DEV) * k ** -.5).bfloat16()
    x = torch.randn(m, k, device=DEV).bfloat16()
    slots = (torch.arange(m, device=DEV) * 17 + 3).int()
    at = (torch.arange(m, device=DEV) * 211 % 4001).int()
    here, want = (ops.Cache(at, *(torch.zeros(m + 8, hkv, 16, d, device=DEV)
                                  .bfloat16() for _ in range(2)), slots, 1e4)
                  for _ in range(2))
    q = ops.linear_heads(x, w, None, here)
    parts = ops.linear(x, w).split([hq * d, hkv * d, hkv * d], 1)
    qw = ops.rope_kv_append(*(t.reshape(m, -1, d).contiguous()
                              for t in parts), *want)
    # one rounding of the same 32-bit numbers, whose last bits may differ
    for got, ref in ((q, qw), (here.k, want.k)):
        got, ref = got.float(), ref.float()
        assert bool(((got - ref).abs() <=
                     2.0 ** -7 * ref.abs() + 2.0 ** -20).all())
    assert torch.equal(here.v, want.v)
