"""Portions of linear attention in as many segments as pay, from a chunk each
up, against the token-by-token form on the CPU."""

import pytest
import torch

from substratus_amd.ops import hybrid as ops

from test_hybrid_ops_gpu import close, gla_inputs, make_batch, on_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("parts", [[(0, 64)], [(5, 65)], [(0, 97), (3, 31)],
                                   [(16, 250)], [(0, 513), (7, 100)]])
@pytest.mark.parametrize("shape", [(2, 64, 64, 16), (1, 128, 128, 16)])
def test_segments(parts, shape):
    batch = make_batch(parts, blocks=96)
    x, a2, a2b, norm, state = gla_inputs(shape, batch, torch.bfloat16, 51,
                                         2.0)
    dev = [t.cuda() for t in (x, a2, a2b, norm, state)]
    got = ops.gla(*dev, on_gpu(batch), 16.0, 1e-5)
    want = ops.gla(x, a2, a2b, norm, state, batch, 16.0, 1e-5)
    close(got, want, torch.bfloat16, "out")
    # 32-bit data all the way: high and low parts keep 2^-16
    assert float((dev[4].cpu() - state).abs().max()
                 / state.abs().max()) < 1e-4
