"""Products of a few rows (rows_gemm.hip, rows_quant.hip) against 64 bits, at
the sizes where their tiles, stages and shares of the inner dimension end."""

import pytest
import torch

from substratus_amd import ops
from substratus_amd.models.quant import QuantLinear
from substratus_amd.parallel.tp import Linear

pytestmark = pytest.mark.gpu
DEV = "cuda"


def close(got, x, w, bias=None, extra=0.0):
    """Within what rounding allows: half a bf16 step of the result (2^-9), and
    32-bit sums whose order is free: 2^-24 per addend, of which a wave's share
    has at most some hundreds and their errors partly cancel (2^-18 of the sum
    of magnitudes)."""
    want = x.double() @ w.double().T
    room = 2.0 ** -18 * (x.double().abs() @ w.double().abs().T)
    if bias is not None:
        want = want + bias.double()
    assert got.dtype == torch.bfloat16 and got.shape == want.shape
    off = (got.double() - want).abs()
    assert bool((off <= (2.0 ** -8 + extra) * want.abs() + room + 1e-30).all())


def gated(y):
    g, u = y.chunk(2, -1)
    return torch.nn.functional.silu(g) * u


# chunks of 32 columns for four waves, two to a stage, four stages in flight:
# fewer chunks than waves, half stages, a full ring, more than one round
@pytest.mark.parametrize("m", [1, 3, 16])
@pytest.mark.parametrize("k", [32, 96, 160, 1024, 1056, 4544])
@pytest.mark.parametrize("n", [16, 40, 55, 768])
@torch.no_grad()
def test_rows_gemm(m, n, k):
    torch.manual_seed(m * 10000 + n + k)
    w = torch.randn(n, k, device=DEV).bfloat16()
    x = torch.randn(m, k, device=DEV).bfloat16()
    b = torch.randn(n, device=DEV).bfloat16()
    close(ops.linear(x, w), x, w)
    close(ops.linear(x, w, b), x, w, b)
    # rows of a wider buffer
    wide = torch.randn(m, k + 64, device=DEV).bfloat16()
    close(ops.linear(wide[:, 32:32 + k], w), wide[:, 32:32 + k], w)
    y = ops.linear_gated(x, w)
    assert (y is None) == (n % 16 != 0)
    if y is not None:
        want = gated(x.double() @ w.double().T)
        room = (x.double().abs() @ w.double().abs().T).chunk(2, -1)
        # a gate's error reaches the product by silu's slope, at most 1.1
        full = (x.double() @ w.double().T).abs().chunk(2, -1)
        assert bool(((y.double() - want).abs() <= 2.0 ** -8 * want.abs()
                     + 2.0 ** -18 * 1.1 * (room[0] * full[1]
                                           + room[1] * full[0]) + 1e-6).all())


@torch.no_grad()
def test_linear_forms_that_stay_with_the_library():
    """The same results whichever way a product goes: other shapes of x, rows
    that do not begin on 16 bytes, more rows, other types."""
    torch.manual_seed(1)
    w = torch.randn(64, 128, device=DEV).bfloat16()
    for x in (torch.randn(128, device=DEV).bfloat16(),
              torch.randn(2, 3, 128, device=DEV).bfloat16(),
              torch.randn(128, 5, device=DEV).bfloat16().t(),
              torch.randn(4, 132, device=DEV).bfloat16()[:, 4:],
              torch.randn(4, 131, device=DEV).bfloat16()[:, 3:],
              torch.randn(1, 128, device=DEV).bfloat16().expand(3, 128),
              torch.randn(17, 128, device=DEV).bfloat16()):
        got = ops.linear(x, w)
        assert got.shape == (*x.shape[:-1], 64)
        close(got.reshape(-1, 64), x.reshape(-1, 128), w)
    x = torch.randn(3, 128, device=DEV)
    assert torch.equal(ops.linear(x, w.float()),
                       torch.nn.functional.linear(x, w.float()))
    assert ops.linear(x[:0].bfloat16(), w).shape == (0, 64)


@torch.no_grad()
def test_one_row_of_any_stride():
    """The distance to a next row that is not there tells nothing."""
    torch.manual_seed(2)
    n, k, d = 64, 128, 16
    w = torch.randn(n, k, device=DEV).bfloat16()
    norm = torch.ones(k, device=DEV).bfloat16()
    delta = torch.randn(1, k, device=DEV).bfloat16()
    kc, vc = (torch.zeros(1, 1, 16, d, device=DEV).bfloat16()
              for _ in range(2))
    at = torch.zeros(1, device=DEV, dtype=torch.int32)
    cache = ops.Cache(at, kc, vc, at, 0.0)
    for x in (torch.randn(2, 131, device=DEV).bfloat16()[:1, :k],
              torch.randn(k, 1, device=DEV).bfloat16().t(),
              torch.randn(k, device=DEV).bfloat16().as_strided((1, k), (3, 1))):
        assert x.stride(0) % 8
        close(ops.linear(x, w), x, w)
        whole = x.clone(memory_format=torch.contiguous_format)
        whole = whole.as_strided((1, k), (k, 1))
        assert torch.equal(ops.linear_gated(x, w), ops.linear_gated(whole, w))
        assert torch.equal(ops.linear_heads(x, w, None, cache),
                           ops.linear_heads(whole, w, None, cache))
        for a, b in zip(ops.linear_normed(delta, x, norm, 1e-5, w, None),
                        ops.linear_normed(delta, whole, norm, 1e-5, w, None)):
            assert torch.equal(a, b)


def test_linear_keeps_gradients():
    w = torch.nn.Parameter(torch.randn(64, 128, device=DEV).bfloat16())
    x = torch.randn(3, 128, device=DEV).bfloat16()
    ops.linear(x, w).float().sum().backward()
    assert w.grad is not None
    lin = Linear(128, 64, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        lin.weight.copy_(w)
    lin.gated  # noqa: B018  (there beside the plain product)
    xx = x.clone().requires_grad_()
    (got,) = torch.func.vmap(lambda r: (ops.linear(r, w.detach()),))(x)
    close(got, x, w.detach())
    ops.linear(xx, w.detach()).float().sum().backward()
    assert xx.grad is not None


# stages of 256 columns: fewer than waves, a last one in part (q4_0, q8_0), a
# ring's rounds; row tiles of x: 4, 8, 16, 32, twice 32
@pytest.mark.parametrize("quant", ["q4_0", "q8_0", "q4_K", "q6_K"])
@pytest.mark.parametrize("m", [1, 2, 4, 5, 8, 9, 16, 17, 33, 64])
@pytest.mark.parametrize("n,k", [(16, 256), (41, 512), (48, 2304),
                                 (64, 4352), (32, 64), (64, 4544),
                                 (48, 1056)])
@torch.no_grad()
def test_quant_rows(quant, m, n, k):
    if quant.endswith("_K") and k % 256:
        pytest.skip("blocks of 256")
    torch.manual_seed(m * 10000 + n + k)
    lin = Linear(k, n, device=DEV, dtype=torch.bfloat16)
    lin.weight.normal_(0.0, 0.5)
    ql = QuantLinear.from_linear(lin, quant)
    w = ql._dequant_cpu().to(DEV)
    x = torch.randn(m, k, device=DEV).bfloat16()
    # weights unpacked to bf16 on the way (more rows than the vector kernel
    # takes, blocks in odd numbers) are themselves half a step off
    unpacked = k % 64 and m > 8
    got = ql(x)
    want = x.double() @ w.double().T
    room = x.double().abs() @ w.double().abs().T
    slack = (2.0 ** -9 if unpacked else 2.0 ** -18) * room
    assert bool(((got.double() - want).abs()
                 <= 2.0 ** -8 * want.abs() + slack).all())
    # a view of qs that does not begin on 16 bytes
    odd = torch.empty(ql.qs.numel() + 1, dtype=torch.uint8, device=DEV)[1:]
    ql.qs = odd.view(ql.qs.shape).copy_(ql.qs)
    if not k % 64:
        assert torch.equal(ql(x), got)
    if n % 16 == 0:
        y = ql.gated(x)
        want = gated(want)
        assert bool(((y.double() - want).abs() <= 2.0 ** -7 * want.abs()
                     + 2.0 ** -6 * room.mean()).all())


# A single row, whose stages hold nothing of other rows: eight waves with none to
# five stages each, two in flight, a last one in part; workgroups of eight weight
# rows, whose stages are 512 columns, a last one of half or less (4097 to 6144 rows
# of 4096 columns and more); four waves (q4_K, more rows of 4096 columns at most,
# q4_0, more than 12288 of fewer)
@pytest.mark.parametrize("quant", ["q4_0", "q4_K", "q6_K"])
@pytest.mark.parametrize("n,k", [(41, 64), (40, 1984), (48, 4096), (48, 10240),
                                 (48, 4416), (4112, 4096), (4112, 4352),
                                 (4120, 4160), (5000, 12800), (6160, 4096),
                                 (6160, 4352), (6176, 10304), (12304, 64),
                                 (12304, 1984), (12304, 4032), (12304, 4096)])
@torch.no_grad()
def test_quant_one_row(quant, n, k):
    if quant.endswith("_K") and k % 256:
        pytest.skip("blocks of 256")
    torch.manual_seed(n + k)
    lin = Linear(k, n, device=DEV, dtype=torch.bfloat16)
    lin.weight.normal_(0.0, 0.5)
    ql = QuantLinear.from_linear(lin, quant)
    w = ql._dequant_cpu().to(DEV).double()
    x = torch.randn(1, k, device=DEV).bfloat16()
    want, room = x.double() @ w.T, x.double().abs() @ w.abs().T
    assert bool(((ql(x).double() - want).abs()
                 <= 2.0 ** -8 * want.abs() + 2.0 ** -18 * room).all())
    if n % 16 == 0:
        y, want = ql.gated(x), gated(want)
        assert bool(((y.double() - want).abs() <= 2.0 ** -7 * want.abs()
                     + 2.0 ** -6 * room.mean()).all())


def one_column(ql, quant, at, number):
    """Every row's number of column `at`, and its minimum 0."""
    k, qs = ql.in_features, ql.qs
    if quant == "q8_0":
        qs[:, at] = number & 255
    elif quant == "q4_0":
        byte = at // 32 * 16 + at % 16
        high = at % 32 >= 16
        qs[:, byte] = qs[:, byte] & (15 if high else 240) | \
            number + 8 << 4 * high
    elif quant == "q4_K":
        byte, high = k // 16 + at // 64 * 32 + at % 32, at % 64 >= 32
        qs[:, byte] = qs[:, byte] & (15 if high else 240) | \
            number << 4 * high
        qs[:, k // 32 + at // 32] = 0
    else:
        block, half, l = at // 256, at % 256 // 128, at % 128
        low, high = block * 128 + half * 64 + l % 64, l >= 64
        qs[:, low] = qs[:, low] & (15 if high else 240) | \
            (number + 32 & 15) << 4 * high
        pair, turn = k // 2 + block * 64 + half * 32 + l % 32, l // 32 * 2
        qs[:, pair] = qs[:, pair] & (255 - (3 << turn)) | \
            (number + 32 >> 4) << turn


@pytest.mark.parametrize("quant", ["q4_0", "q8_0", "q4_K", "q6_K"])
@pytest.mark.parametrize("m", [2, 5, 16, 33])
@pytest.mark.parametrize("at", [3, 501, 767])
@torch.no_grad()
def test_quant_outliers(quant, m, at):
    """What weights of zero meet leaves nothing behind, however large; what is
    infinite is infinite, by the sign of its weight."""
    torch.manual_seed(m + at)
    n, k = 48, 1024
    lin = Linear(k, n, device=DEV, dtype=torch.bfloat16)
    lin.weight.normal_(0.0, 0.5)
    ql = QuantLinear.from_linear(lin, quant)
    one_column(ql, quant, at, 0)
    w = ql._dequant_cpu().to(DEV).double()
    assert not bool(w[:, at].any())
    x = torch.randn(m, k, device=DEV).bfloat16()
    x[:, at] = 2.0 ** 24
    want = x.double() @ w.T
    room = x.double().abs() @ w.abs().T
    assert bool(((ql(x).double() - want).abs()
                 <= 2.0 ** -8 * want.abs() + 2.0 ** -18 * room).all())
    one_column(ql, quant, at, 5)
    x[:, at] = torch.inf
    w = ql._dequant_cpu().to(DEV)[:, at]
    assert bool((w != 0).all())
    assert torch.equal(ql(x).float(), (w * torch.inf).expand(m, n))


@torch.no_grad()
def test_products_of_few_rows_in_a_graph():
    """Replays with other inputs, eager work between."""
    torch.manual_seed(3)
    lin = Linear(512, 96, device=DEV, dtype=torch.bfloat16)
    lin.weight.normal_()
    ql = QuantLinear.from_linear(lin, "q4_0")
    x = torch.randn(3, 512, device=DEV).bfloat16()

    def step():
        return lin(x), lin.gated(x), ql(x), ql.gated(x)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for seed in range(4):
        x.copy_(torch.randn(3, 512, device=DEV))
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, step()):
            assert torch.equal(a, b)
