"""Products and training ops where torch's own operations are to be seen:
traces, function modes, batches of gradients."""

import pytest
import torch
import torch.nn.functional as F
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.symbolic_shapes import ShapeEnv
from torch.overrides import TorchFunctionMode

from substratus_amd import ops
from substratus_amd.models.model import NormParams, added_product
from substratus_amd.models.quant import QuantLinear
from substratus_amd.ops import train
from substratus_amd.parallel.tp import Linear, RowParallelLinear


class Seen(TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.calls = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.calls.append(func)
        return func(*args, **(kwargs or {}))


def test_plain_tensors():
    x = torch.zeros(2, 2)
    assert ops.plain_tensors(x, None)
    with torch.device("cpu"):           # a mode of torch's own, for factories
        assert ops.plain_tensors(x)
    with Seen():
        assert not ops.plain_tensors(x)
    told = []

    def traced(t):
        told.append(ops.plain_tensors(t))
        return t + 1
    torch.jit.trace(traced, x, check_trace=False)
    assert told == [False]
    assert not ops.plain_tensors(x, x.to_sparse_csr())
    assert not ops.plain_tensors(x.to_sparse())

    class Told(torch.autograd.Function):
        @staticmethod
        def forward(ctx, t):
            return t * 2

        @staticmethod
        def backward(ctx, dy):
            told.append(ops.plain_tensors(dy))
            return dy * 2
    x.requires_grad_()
    torch.autograd.grad(Told.apply(x), x, torch.ones(3, 2, 2),
                        is_grads_batched=True)
    torch.autograd.grad(Told.apply(x), x, torch.ones(2, 2))
    assert told == [False, False, True]


def test_symbolic_trace():
    lin = Linear(32, 16, bias=True)
    torch.nn.init.normal_(lin.weight)
    graph = torch.fx.symbolic_trace(lin)
    x = torch.randn(3, 32)
    assert torch.equal(graph(x), lin(x))


def test_compiled():
    """As one graph, without a break."""
    w = torch.randn(16, 32)

    def fn(x):
        assert not ops.plain_tensors(x, w)
        return train.silu_mul(ops.linear(x, w))
    x = torch.randn(3, 32)
    want = train.silu_mul(ops.linear(x, w))
    got = torch.compile(fn, backend="eager", fullgraph=True)(x)
    assert torch.equal(got, want)


@pytest.mark.parametrize("quant", ["", "q8_0"])
@torch.no_grad()
def test_added_rows_are_not_counted(quant):
    """One graph for a step of any number of rows."""
    dtype = torch.bfloat16 if quant else torch.float32
    lin = RowParallelLinear(64, 128, dtype=dtype)
    torch.nn.init.normal_(lin.weight)
    if quant:
        lin = QuantLinear.from_linear(lin, quant)
    norm = NormParams(128, True, dtype=dtype)
    graphs = []

    def fn(x, h):
        return added_product(lin, x, h, norm, 1e-5)
    compiled = torch.compile(
        fn, backend=lambda graph, _: graphs.append(graph) or graph,
        dynamic=True)
    for rows in (3, 8, 12, 40, 300):
        x, h = (torch.randn(rows, n).to(dtype) for n in (64, 128))
        assert torch.equal(compiled(x, h)[1][0], fn(x, h)[1][0])
        if rows == 3:
            first = len(graphs)
    assert len(graphs) == first


@torch.no_grad()
def test_exported_from_256_rows_on():
    """A product of any number of rows that the library may take."""
    with FakeTensorMode(shape_env=ShapeEnv()):
        lin = Linear(4096, 4096, device="cuda", dtype=torch.bfloat16)
        x = torch.empty(1000, 4096, device="cuda", dtype=torch.bfloat16)
        rows = torch.export.Dim("rows", min=256, max=4096)
        torch.export.export(lin, (x,), dynamic_shapes=({0: rows},))


@pytest.mark.gpu
@pytest.mark.parametrize("rows,k", [(3, 2048), (40, 2048), (4165, 11008)])
@torch.no_grad()
def test_traced_products(rows, k):
    lin = Linear(k, 4096, device="cuda", dtype=torch.bfloat16)
    lin.weight.normal_()
    x, other = (torch.randn(rows, k, device="cuda").bfloat16()
                for _ in range(2))
    traced = torch.jit.trace(lin, x)
    want = F.linear(other.double(), lin.weight.double())
    assert float((traced(other).double() - want).norm()) <= \
        2.0 ** -8 * float(want.norm())
    with Seen() as mode:
        lin(x)
    assert F.linear in mode.calls
    compiled = torch.compile(lambda t: lin(t), backend="eager",
                             fullgraph=True)
    assert float((compiled(other).double() - want).norm()) <= \
        2.0 ** -8 * float(want.norm())


@pytest.mark.gpu
@torch.no_grad()
def test_traced_training_ops():
    h, d, w = (torch.randn(*s, device="cuda").bfloat16()
               for s in ((4, 64), (4, 64), (64,)))
    for fn in (lambda t: train.add_norm(t, (d,), w, None, 1e-5)[0],
               lambda t: train.add_norm(t, (), w, w, 1e-5)[0],
               lambda t: train.silu_mul(t)):
        traced = torch.jit.trace(fn, h)
        want = fn((h * 3).cpu().to(h.device))
        assert float((traced(h * 3).float() - want.float()).abs().max()) \
            <= 2.0 ** -6 * float(want.abs().max())


@pytest.mark.gpu
def test_batches_of_gradients():
    """Each gradient of a batch as it is by itself."""
    torch.manual_seed(0)

    def leaf(*shape):
        return torch.randn(*shape, device="cuda").bfloat16().requires_grad_()
    x, w = leaf(4165, 11008), leaf(4096, 11008)
    h, d, n, b = leaf(5, 64), leaf(5, 64), leaf(64), leaf(64)
    table = torch.nn.Embedding(50, 64, device="cuda", dtype=torch.bfloat16)
    tokens = torch.randint(0, 50, (2, 9), device="cuda")
    for out, given in (
            (ops.linear(x, w), (x, w)),
            (sum(train.add_norm(h, (d,), n, b, 1e-5)), (h, d, n, b)),
            (train.add_norm(h, (), n, None, 1e-5)[0], (h, n)),
            (train.silu_mul(h), (h,)),
            (train.lookup(tokens, table), (table.weight,))):
        dy = torch.randn(2, *out.shape, device="cuda").bfloat16()
        got = torch.autograd.grad(out, given, dy, retain_graph=True,
                                  is_grads_batched=True)
        for i in range(2):
            one = torch.autograd.grad(out, given, dy[i], retain_graph=True)
            for a, c in zip(got, one):
                a, c = a[i].detach().double(), c.detach().double()
                assert float((a - c).norm()) <= 0.01 * float(c.norm())
