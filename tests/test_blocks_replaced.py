"""Steps of models with a block whose decode_ops is not Block's, or whose norms
are not like the others': it is given sums of outputs, as any block is that
knows nothing of norms that the block before has begun."""

from dataclasses import replace

import pytest
import torch

from substratus_amd import ops
from substratus_amd.models import CausalLM, get_config
from substratus_amd.models.model import Block


class Own(Block):
    def decode_ops(self, h, deltas, positions, k_cache, v_cache, slots,
                   block_table, seq_lens):
        for d in deltas:
            h = h + d
        return (yield from super().decode_ops(
            h, (), positions, k_cache, v_cache, slots, block_table, seq_lens))


def model_of(how, device, dtype):
    # wide enough that products of 40 rows are made by shares
    cfg = replace(get_config("llama-tiny"), num_layers=3,
                  intermediate_size=8192)
    model = CausalLM(cfg, device=device, dtype=dtype)
    model.init_random(5)
    for i, blk in enumerate(model.blocks):
        if how == i:
            blk.__class__ = Own
    if how == "eps":
        model.blocks[1].eps = 0.5
    return model


def step(model, rows, device, dtype):
    g = torch.Generator().manual_seed(rows)
    tokens = torch.randint(0, 512, (rows,), generator=g).to(device)
    at = torch.arange(rows, device=device, dtype=torch.int32)
    caches = [tuple(torch.zeros(rows, model.n_kv_heads, 16, model.cfg.head_dim,
                                device=device, dtype=dtype) for _ in range(2))
              for _ in model.blocks]
    return model.forward_decode(tokens, torch.zeros_like(at), caches, at * 16,
                                at[:, None].contiguous(),
                                torch.ones_like(at)).double()


@pytest.mark.parametrize("how", [0, 1, 2])
@torch.no_grad()
def test_replaced(how):
    got, want = (step(model_of(h, "cpu", torch.float32), 3, "cpu",
                      torch.float32) for h in (how, ""))
    assert torch.allclose(got, want, rtol=1e-4, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("how", [0, 1, 2, "eps"])
@pytest.mark.parametrize("rows", [3, 40])
@torch.no_grad()
def test_replaced_beside_begun_norms(how, rows, monkeypatch):
    model = model_of(how, "cuda", torch.bfloat16)
    got = step(model, rows, "cuda", torch.bfloat16)
    for name in "linear_added", "linear_added_norm":
        monkeypatch.setattr(ops, name, lambda *a: None)
    want = step(model, rows, "cuda", torch.bfloat16)
    # rows are rounded to bf16 at another place: 2^-9 of each of some ten
    assert float((got - want).norm()) <= 0.02 * float(want.norm())
