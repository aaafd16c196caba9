"""gelu of products in their kernel (rows_gemm.hip, mid_gemm.hip, tile_gemm.hip)
against the product and gelu by themselves: the same sums, rounded and taken
through the same function, so the same bits."""

import pytest
import torch

from substratus_amd import _C, ops
from substratus_amd.models.model import gelu_product
from substratus_amd.parallel.tp import Linear

pytestmark = pytest.mark.gpu
DEV = "cuda"


# rows_gemm: a tile of rows to four, widths that end within a workgroup's 16.
# mid_gemm: whole sums and shares, columns stored by fours and by themselves
@pytest.mark.parametrize("m,n,k", [(1, 8, 32), (5, 24, 96), (16, 3072, 768),
                                   (8, 1001, 544), (17, 3072, 768),
                                   (48, 40, 160), (64, 1000, 2048),
                                   (24, 1001, 2080), (17, 4600, 4544),
                                   (40, 18176, 4544), (100, 4600, 4544),
                                   (256, 24, 16416), (248, 3077, 16384)])
@torch.no_grad()
def test_bits(m, n, k):
    torch.manual_seed(m + n + k)
    w = (torch.randn(n, k, device=DEV) * 3 * k ** -.5).bfloat16()
    x = torch.randn(m, k + 64, device=DEV).bfloat16()[:, 32:32 + k]
    b = torch.randn(n, device=DEV).bfloat16()
    # ends of the range, where gelu is the number itself, or none
    x[m // 2, 0] = float("inf")
    for bias in (None, b):
        got = ops.linear_gelu(x, w, bias)
        if ops._few_rows(x, w, bias, False) is None:
            assert got is None
            continue
        y = ops.linear(x, w, bias)
        want = ops.gelu(y)
        assert torch.equal(got.isnan(), want.isnan())
        assert torch.equal(got.nan_to_num(), want.nan_to_num())


# tiles that are partly there, all or some of them shared, whole rounds
@pytest.mark.parametrize("m,n,k", [(256, 256, 72), (264, 1000, 248),
                                   (1000, 1024, 4544), (4360, 4104, 1032),
                                   (2048, 8192, 520)])
@torch.no_grad()
def test_tiles(m, n, k):
    torch.manual_seed(m + n + k)
    w = (torch.randn(n, k, device=DEV) * 3 * k ** -.5).bfloat16()
    x = torch.randn(m, k, device=DEV).bfloat16()
    b = torch.randn(n, device=DEV).bfloat16()
    x[m // 2, 0] = float("inf")
    for bias in (None, b):
        got = _C.tile_gemm(x, w, bias, False, False, False, True)
        want = ops.gelu(_C.tile_gemm(x, w, bias, False, False))
        assert torch.equal(got.isnan(), want.isnan())
        assert torch.equal(got.nan_to_num(), want.nan_to_num())
    y = ops.linear_gelu(x.view(2, m // 2, k), w, b)
    good = _C.tile_gemm_good(m, n, k, k, k, False, False, False)
    assert (y is not None) == good
    if good:
        assert torch.equal(y.view(m, n).nan_to_num(), want.nan_to_num())


@torch.no_grad()
def test_what_stays():
    """Sizes that gelu refuses, gradients and hooks."""
    x, w = (torch.randn(n, 64, device=DEV).bfloat16() for n in (3, 7))
    assert ops.linear_gelu(x, w) is None
    with pytest.raises(RuntimeError):
        ops.gelu(ops.linear(x, w))
    lin = Linear(64, 16, device=DEV, dtype=torch.bfloat16)
    lin.weight.copy_(torch.randn(16, 64))
    want = ops.gelu(lin(x))
    assert torch.equal(gelu_product(lin, x), want)
    with torch.enable_grad():
        assert ops.linear_gelu(x, lin.weight) is None
    seen = []
    lin.register_forward_hook(lambda *a: seen.append(1))
    assert torch.equal(gelu_product(lin, x), want) and seen


def test_one_activation():
    x, w = (torch.randn(n, 64, device=DEV).bfloat16() for n in (3, 16))
    with pytest.raises(RuntimeError):
        _C.rows_gemm(x.new_empty(3, 8), x, w, None, True, True)


def test_every_number():
    """Every bf16 number but NaN, against 64 bits: half a step of the result (2^-8
    of a number that begins with eight bits of 1.0000000), a little for the 32-bit
    steps before (an exponent of up to 88, after seven roundings of 2^-24, is off
    by 2^-14.7 at most), and what is too small: numbers that are not normal, and
    those whose 1 + exp is past the largest number, 2^128 (of -10.0625, whose gelu
    is 2.4 of the least normal number)."""
    bits = torch.arange(1 << 16, dtype=torch.int32).to(torch.int16)
    v = bits.view(torch.bfloat16)
    v = v[~v.isnan() & ~v.isinf()]
    x = v.double()
    t = 2 * (2 / torch.pi) ** 0.5 * (x + 0.044715 * x ** 3)
    want = x * torch.sigmoid(t)
    got = ops.gelu(torch.nn.functional.pad(v, (0, -len(v) % 8)).to(DEV))
    off = (got[:len(v)].cpu().double() - want).abs()
    assert bool((off <= (2.0 ** -8 + 2.0 ** -14) * want.abs()
                 + 2.0 ** -126 + 2.0 ** -128 * x.abs().clamp(max=16)).all())
