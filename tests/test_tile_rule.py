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


@pytest.mark.parametrize("m", [20, 40, 80, 200, 250])
@pytest.mark.parametrize("k", [1024, 2048, 4096, 9216, 17408])
def test_few_rows(m, k):
    """Of matrices of long rows the narrow ones leave the library, up to some
    width, whose neighbours are not told apart."""
    widths = [n + by for n in (1024, 4096, 8192, 12288) for by in (-16, 0, 16)]
    good = [_C.mid_gemm_good(m, n, k, False) for n in widths]
    assert good == sorted(good, reverse=True)
    assert good[0] == (k >= (4096 if m <= 40 else 8192)) and not good[-1]


@pytest.mark.parametrize("m", [33, 64, 96])
def test_shares_in_step(m):
    """Four shares of 8192 begin on whole 4 KB of rows of 16 KB; a little wider
    there are three or seven of them, a little longer they begin elsewhere."""
    assert not _C.mid_gemm_good(m, 8192, 8192, False)
    assert _C.mid_gemm_good(m, 8208, 8192, False)
    assert _C.mid_gemm_good(m, 8192, 8448, False)


@pytest.mark.parametrize("m,n,k,pays", [
    (64, 4096, 4096, True), (24, 8192, 28672, True),
    (69, 2560, 3072, False), (128, 2048, 4096, False), (65, 4096, 4096, True),
    (128, 4096, 4096, True), (100, 5120, 4096, True), (128, 5120, 5120, True),
    (100, 2048, 5632, True), (192, 2048, 5632, True), (192, 4096, 4096, True),
    (129, 4544, 6144, False), (162, 5120, 8192, False),
    (217, 2112, 3200, True), (254, 12288, 7584, False),
    (256, 4096, 11008, True), (256, 5632, 24576, True)])
def test_products_with_their_norm(m, n, k, pays):
    """Those that lost by it stay with the library and a norm of its own."""
    assert _C.mid_norm_good(m, n, k) == pays


@pytest.mark.parametrize("n,k,thin", [
    (2048, 512, True), (2112, 512, False), (4096, 8192, False),
    (4160, 2048, False), (4160, 2176, True), (6144, 16384, True),
    (6208, 4096, False), (5120, 768, False), (5120, 2240, False)])
def test_eight_rows_of_weights(n, k, thin):
    """A workgroup has eight of them where that is the faster one."""
    assert _C.rows_added_parts(8, n, k) == n // (8 if thin else 16)
    assert _C.rows_added_parts(9, n, k) == n // 16


@pytest.mark.parametrize("m,n,k,paired,pays", [
    (48, 8192, 4096, True, True), (64, 28672, 4096, True, True),
    (69, 6144, 2048, True, False), (96, 13824, 16384, True, False),
    (96, 2464, 4096, True, False), (135, 4288, 6144, True, False),
    (48, 36864, 2048, True, False), (20, 32000, 2048, False, True),
    (24, 27648, 8192, False, True), (20, 16384, 8192, False, False),
    (20, 57344, 8192, False, False), (64, 33328, 2048, False, False),
    (64, 128256, 4096, False, True), (20, 22016, 8192, False, True),
    (40, 57344, 8192, False, True), (40, 65024, 8192, False, False),
    (34, 33216, 4096, False, True), (48, 36864, 6144, True, True),
    (64, 40960, 10240, False, False), (120, 10880, 8192, True, True),
    (108, 2112, 6144, True, True), (151, 6016, 10240, True, True),
    (132, 4352, 8192, True, False), (230, 6144, 8192, True, False)])
def test_rows_that_meet_in_memory(m, n, k, paired, pays):
    """Rows of a multiple of 4 KB leave the library where that was measured to
    be the faster way, and not at its edges."""
    assert _C.mid_gemm_good(m, n, k, paired) == pays


@pytest.mark.parametrize("m,n,k,a,b,rows", [
    (2048, 4096, 5000, True, True, 256), (4096, 2048, 4096, True, True, 256),
    (5120, 5120, 6000, True, True, 256), (6144, 4096, 2488, True, True, 256),
    (2048, 2048, 4165, True, True, 256), (768, 8192, 32768, False, True, 256),
    (577, 8192, 32768, False, True, 224), (4096, 2048, 4096, False, True, 256),
    (6144, 2048, 2488, True, True, 192), (320, 4544, 65024, False, True, 160),
    (384, 57344, 8192, False, False, 192)])
def test_heights(m, n, k, a, b, rows):
    """Flipped operands are turned more often by tiles of fewer rows: those that
    were slower by it have 256, or the most of the others."""
    assert _C.tile_gemm_rows(m, n, k, a, b) == rows


@pytest.mark.parametrize("kind,m,n,k,pays", [
    ("plain", 256, 8192, 28672, True), ("plain", 512, 8192, 28672, True),
    ("plain", 1333, 8192, 28672, True), ("plain", 1777, 4096, 16384, True),
    ("plain", 1024, 4096, 16384, True), ("plain", 768, 10240, 8192, True),
    ("plain", 900, 8192, 8192, False), ("plain", 768, 8192, 32768, False),
    ("plain", 768, 8192, 27648, True), ("plain", 3000, 4096, 14336, True),
    ("plain", 1536, 16384, 4096, True), ("plain", 1024, 16384, 4096, False),
    ("inputs", 256, 8192, 32000, True), ("inputs", 512, 8192, 10240, True),
    ("inputs", 900, 32768, 8192, True), ("inputs", 640, 8192, 32000, False),
    ("inputs", 768, 8192, 8192, False),
    ("weights", 8192, 32768, 288, False), ("weights", 4096, 16384, 288, False),
    ("weights", 18176, 4544, 256, True), ("weights", 4096, 4096, 257, True),
    ("inputs", 320, 32768, 8192, False), ("weights", 2048, 2048, 3072, False),
    ("weights", 27648, 5120, 320, True), ("weights", 5120, 5120, 416, True)])
def test_products_the_library_is_tuned_for(kind, m, n, k, pays):
    """They stay with it, and their neighbours, which take twice as long there, do
    not; wherever the operands' lines lie."""
    a, b = kind == "weights", kind in ("inputs", "weights")
    for pad in (0, 64):
        assert _C.tile_gemm_good(m, n, k, (m if a else k) + pad,
                                 (n if b else k) + pad, a, b, False) == pays
