"""Which products of many rows leave the library: gradients of inputs that the
tiles were measured to be slower at stay, those that gain go."""

import pytest

_C = pytest.importorskip("substratus_amd._C")


@pytest.mark.parametrize("kind,m,n,k,pays", [
    ("plain", 2048, 4096, 4096, False), ("plain", 4096, 12288, 4096, False),
    ("plain", 2331, 4096, 4096, False), ("plain", 2331, 2048, 5632, False),
    ("plain", 2472, 6160, 2048, True), ("plain", 4096, 18176, 4544, True),
    ("plain", 4165, 4096, 11008, True), ("plain", 4485, 12288, 4096, True),
    ("plain", 4096, 4544, 18176, True), ("plain", 2331, 32000, 2048, True),
    ("gated", 4165, 22016, 4096, True), ("gated", 4096, 22016, 4096, True),
    ("inputs", 4165, 2048, 6144, False), ("inputs", 2331, 4096, 22016, False),
    ("inputs", 1777, 5120, 5120, False), ("inputs", 2464, 4096, 32000, False),
    ("inputs", 3000, 4096, 22016, False), ("inputs", 2472, 4544, 18176, False),
    ("inputs", 4096, 4544, 65024, True), ("inputs", 2331, 2048, 6144, True),
    ("inputs", 1777, 4096, 6144, True), ("inputs", 8192, 4096, 4096, True),
    ("inputs", 2331, 5632, 2048, True), ("inputs", 2331, 5120, 15360, True),
    ("weights", 6144, 2048, 4096, True), ("weights", 5120, 5120, 700, True),
    ("weights", 65024, 4544, 4096, True)])
def test_rule(kind, m, n, k, pays):
    a, b = kind == "weights", kind in ("inputs", "weights")
    assert _C.tile_gemm_good(m, n, k, m if a else k, n if b else k, a, b,
                             kind == "gated") == pays
