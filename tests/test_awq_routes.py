"""CPU: which int4 products of many rows go where: the tiles a plan cuts."""
import pytest

from sglang_security_amd import ops


@pytest.mark.parametrize("gated", [False, True])
def test_tiles_cover_a_product_once(gated):
    """Every row and column lies in one tile, and no tile lies outside; strips of 192 columns that do not divide the rest occur."""
    ragged = 0
    for K in (128, 512, 4096):
        for N in (256, 1024, 2560, 4096, 5120, 6144, 6656, 6784, 7168, 8192, 22016, 27648, 28672):
            for M in (1, 63, 64, 129, 300, 627, 819, 1152, 1600, 2112, 3200, 3700):
                rows, row_tiles, whole, tail, narrow = ops.awq_gemm_prefill_tiles(M, N, K, gated)
                assert rows in (128, 192, 256) and (row_tiles - 1) * rows < M <= row_tiles * rows
                rest = N - 256 * whole
                if tail:
                    assert narrow in ((128,) if gated else (128, 192)) and (tail - 1) * narrow < rest <= tail * narrow
                    ragged += rest % narrow != 0
                else:
                    assert -256 < rest <= 0
    assert gated or ragged > 20
