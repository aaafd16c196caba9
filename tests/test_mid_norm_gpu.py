"""Products whose shares the norm that follows adds up, against the product, the
sum and the norm one after the other."""

import pytest
import torch

from substratus_amd import ops
from tests.test_rows_normed_gpu import DEV, made

pytestmark = pytest.mark.gpu


# blocks of 32 to 128 rows, the last of them parts; rows of a thread's one quad, of
# two and of four, of part of a workgroup
@pytest.mark.parametrize("m,k,n,bias", [
    (17, 4096, 5120, False), (33, 4128, 256, True), (40, 11008, 2048, False),
    (64, 4096, 4096, False), (100, 4128, 4160, True), (129, 28672, 8256, False),
    (256, 11008, 4096, False), (57, 3104, 1088, True), (96, 3104, 16384, False)])
@torch.no_grad()
def test_added_norm(m, k, n, bias):
    torch.manual_seed(m * k + n)
    lin, w = made("dense", k, n, bias)
    x = torch.randn(m, k, device=DEV).bfloat16()
    h = 3 * torch.randn(m, n, device=DEV).bfloat16()
    norm = (1 + 0.3 * torch.randn(n, device=DEV)).bfloat16()
    assert ops._load_ext().mid_norm_good(m, n, k)
    kept = h.clone()
    total, rows = lin.added_norm(x, h, norm, 1e-5)
    assert torch.equal(h, kept)
    if ops._load_ext().mid_gemm_good(m, n, k, False):   # the same shares
        assert torch.equal(total, h + lin(x))
    want = x.double() @ w.T + h.double()
    if bias:
        want += lin.bias.double()
    # two roundings to bf16, and the sums' own
    assert float((total.double() - want).norm()) <= \
        2.0 ** -7 * float(want.norm())
    t = total.double()
    want = t * (t.square().mean(1, keepdim=True) + 1e-5).rsqrt() * norm.double()
    # rounded to bf16 once; the squares are of rows before they are
    assert torch.allclose(rows.rows.double(), want, rtol=2.0 ** -7, atol=1e-6)


@torch.no_grad()
def test_refused():
    lin, _ = made("dense", 4096, 4096, False)
    x, h = (torch.randn(257, 4096, device=DEV).bfloat16() for _ in range(2))
    w = torch.ones(4096, device=DEV).bfloat16()
    assert lin.added_norm(x[:64], h[:64], w, 1e-5) is not None
    assert lin.added_norm(x, h, w, 1e-5) is None
    assert lin.added_norm(x[:16], h[:16], w, 1e-5) is None
    assert lin.added_norm(x[:64], h[:65], w, 1e-5) is None
    assert lin.added_norm(x[:64], h[:64].float(), w, 1e-5) is None
    assert lin.added_norm(x[:64], h[:128:2], w, 1e-5) is None
    with torch.enable_grad():
        assert lin.added_norm(x[:64], h[:64], w.requires_grad_(), 1e-5) is None


@torch.no_grad()
def test_bias_between_boundaries():
    """Part of a larger tensor: the norm reads four numbers at a time, and the
    product with a norm of its own takes any."""
    torch.manual_seed(3)
    lin, w = made("dense", 4096, 4096, True)
    x, h = (torch.randn(64, 4096, device=DEV).bfloat16() for _ in range(2))
    norm = torch.ones(4096, device=DEV).bfloat16()
    parts = torch.randn(4097, device=DEV).bfloat16()
    lin.bias = torch.nn.Parameter(parts[1:], requires_grad=False)
    assert lin.bias.data_ptr() % 16
    assert lin.added_norm(x, h, norm, 1e-5) is None
    want = x.double() @ w.T + parts[1:].double()
    assert float((lin(x).double() - want).norm()) <= \
        2.0 ** -8 * float(want.norm())
    lin.bias = torch.nn.Parameter(parts[:-1], requires_grad=False)
    assert lin.added_norm(x, h, norm, 1e-5) is not None
