"""Into how many shares workgroups divide a context's keys."""

import pytest

_hybrid = pytest.importorskip("substratus_amd._hybrid")


@pytest.mark.parametrize("entries,rows", [(0, 1), (3, 0), (0, 0)])
def test_latent_shares_of_nothing(entries, rows):
    """No division by a number of workgroups that is none."""
    assert _hybrid.attn_latent_splits(entries, rows, 16, 900, 576, 512) >= 1


@pytest.mark.parametrize("n,span,dim,vdim,shares", [
    (1, 900, 576, 512, 7), (20, 2000, 576, 512, 12), (1, 4000, 576, 512, 20),
    (128, 900, 576, 512, 2), (130, 900, 576, 512, 3), (170, 900, 320, 256, 3),
    (171, 900, 576, 512, 1), (130, 800, 576, 512, 1), (300, 4000, 576, 512, 1),
    (64, 1600, 192, 128, 4), (100, 900, 192, 128, 3), (120, 1500, 192, 128, 4),
    (200, 900, 72, 64, 2), (230, 500, 72, 64, 1), (1, 60000, 192, 128, 16)])
def test_latent_shares(n, span, dim, vdim, shares):
    """As many as there is room for on the CUs, which small keys leave more of,
    and no share without a chain worth its merge."""
    assert _hybrid.attn_latent_splits(n, 1, 16, span, dim, vdim) == shares


@pytest.mark.parametrize("entries,rows,heads,vdim,span,shares", [
    (1, 100, 16, 128, 2100, 11), (4, 103, 32, 128, 3093, 3),
    (4, 103, 32, 64, 1024, 3), (1, 900, 16, 128, 64, 1),
    (8, 2400, 16, 128, 4000, 1), (0, 0, 16, 128, 0, 1)])
def test_portion_shares(entries, rows, heads, vdim, span, shares):
    """As many as there are CUs for, where a chain of steps is worth them."""
    assert _hybrid.attn_ctx_prefill_splits(entries, rows, heads, vdim,
                                           span) == shares


@pytest.mark.parametrize("entries,rows,heads,vdim,span,window,flat,shared", [
    (1, 900, 16, 128, 900, False, False, True),
    (8, 2400, 16, 128, 300, False, False, False),
    (1, 58, 64, 128, 64, False, False, False),
    (1, 59, 64, 128, 65, False, False, True),
    (1, 14, 4, 64, 14, False, False, True),
    (1, 2682, 8, 256, 168, True, False, False),
    (2, 2214, 8, 256, 250, True, False, False),
    (4, 1973, 16, 64, 1220, True, False, True),
    (2, 2304, 4, 256, 1624, True, False, True),
    (1, 2682, 8, 256, 2682, False, False, True),
    (6, 2400, 16, 128, 480, False, True, False),
    (2, 900, 16, 128, 480, False, True, True)])
def test_portions_whose_waves_share_rows(entries, rows, heads, vdim, span,
                                         window, flat, shared):
    """Where tiles are few, and neither one step nor a round of CUs more."""
    assert _hybrid.attn_ctx_prefill_shared(entries, rows, heads, vdim, span,
                                           window, flat) == shared
