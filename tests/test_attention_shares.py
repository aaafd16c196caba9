"""How many shares decode attention cuts a sequence into, by the kernel that
takes it."""

import pytest

_C = pytest.importorskip("substratus_amd._C")


@pytest.mark.parametrize("bsz,hq,hkv,d,pages,grouped,want", [
    # a head at a time: 71 workgroups a sequence
    (1, 71, 1, 64, 256, False, 15), (16, 71, 1, 64, 256, False, 1),
    (64, 24, 2, 64, 256, False, 1), (1, 16, 16, 64, 10, False, 3),
    # 8 heads at a time
    (4, 24, 1, 64, 256, False, 16), (128, 24, 1, 64, 256, False, 3),
    # a group of 4, 8 or 16 at a time, two pages a step
    (16, 32, 8, 128, 10, False, 5), (16, 32, 8, 128, 256, False, 8),
    (16, 32, 8, 128, 4, False, 1), (200, 64, 8, 128, 256, False, 1),
    # 16 heads of any group at a time, four pages a step
    (1, 71, 1, 64, 256, True, 16), (64, 71, 1, 64, 256, True, 4),
    (16, 32, 8, 128, 10, True, 3), (1, 32, 8, 128, 1, True, 1)])
def test_shares(bsz, hq, hkv, d, pages, grouped, want):
    assert _C.paged_attn_nsplit(bsz, hq, hkv, d, pages, grouped) == want
