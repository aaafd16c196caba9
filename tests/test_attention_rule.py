"""Into how many shares workgroups divide a context's keys."""

import pytest

_hybrid = pytest.importorskip("substratus_amd._hybrid")


@pytest.mark.parametrize("entries,rows", [(0, 1), (3, 0), (0, 0)])
def test_latent_shares_of_nothing(entries, rows):
    """No division by a number of workgroups that is none."""
    assert _hybrid.attn_latent_splits(entries, rows, 16, 900) >= 1
