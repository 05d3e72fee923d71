"""GPU: fp8 products of many rows on the tile kernels, at the edges of their tiles: rows and columns that do not fill a
tile, a single k-block, views with gaps, a bias, and calls the tiles do not take."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _codes(shape, g):
    """Halves from -4 to 4: every sum of their products is exact in fp32."""
    return (torch.randint(-8, 9, shape, generator=g, device=DEV) * 0.5).to(torch.float8_e4m3fn)


# one size for each form the rule picks between: 64 x 64, 64 x 128, 128 x 128 (one and two blocks a unit), 256 x 256
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(65, 4096, 128), (129, 4112, 256), (300, 6160, 384), (300, 7184, 256), (257, 12304, 128),
                                   (513, 12304, 256), (2049, 6160, 128), (700, 16, 1024), (1025, 28688, 128)])
@pytest.mark.parametrize("bias", [False, True])
def test_scaled_products_of_many_rows(M, N, K, dtype, bias):
    from sglang_security_amd import ops

    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    a, w = _codes((M, K + 48), g)[:, :K], _codes((N, K + 16), g)[:, :K]
    sa, sb = (2.0 ** torch.randint(-6, 1, (n,), generator=g, device=DEV).float() for n in (M, N))
    b = (torch.randint(-40, 41, (N,), generator=g, device=DEV) * 0.25).to(dtype) if bias else None
    want = (a.double() @ w.double().t()) * sa.double()[:, None] * sb.double() + (b.double() if bias else 0)
    for out in (None, torch.full((M, N + 24), float("nan"), dtype=dtype, device=DEV)[:, :N],      # rows of whole 16 bytes
                torch.full((M, N + 3), float("nan"), dtype=dtype, device=DEV)[:, :N]):            # rows the tiles do not take
        got = ops.fp8_scaled_mm(a, w.t(), sa, sb, dtype, b, out)
        assert torch.equal(got, want.to(dtype))     # exact up to the one rounding
        assert out is None or out._base[:, N:].isnan().all()      # what lies between the rows stays


# four waves a block: strips of 192 columns alone, of 128 alone, of 256 alone, of 256 with 128 and with 192 behind them; rows and
# columns that do not fill them, an odd and an even number of k-blocks
@pytest.mark.parametrize("M,N,K,bias", [(2048, 6144, 1024, False), (2047, 4112, 1152, True), (700, 6160, 2048, False),
                                        (1700, 8192, 3584, True), (2048, 8208, 2048, False), (1300, 28688, 4096, True)])
def test_blocks_of_four_waves(M, N, K, bias):
    test_scaled_products_of_many_rows(M, N, K, torch.bfloat16, bias)


def test_rule_covers_decode_and_prompts():
    """Single rows stay on the kernels that stream; prompts go to the tiles, with and without the streaming copy."""
    from sglang_security_amd import ops

    assert not ops.fp8_tiled(64, 28672, 4096) and not ops.fp8_tiled(0, 4096, 4096) and not ops.fp8_tiled(2048, 4096, 100)
    assert ops.fp8_tiled(2048, 4096, 4096) and ops.fp8_tiled(256, 28672, 4096)


def test_rule_leaves_narrow_products_alone():
    """Narrow outputs under a long inner dimension stay on the kernels that spread it over idle units (15.8 us against 30.9
    for 1024 x 128 x 14336 on the streaming copy), also where fp8_scaled_mm itself would not take the tiles (256 x 512 x 4608)."""
    from sglang_security_amd import ops

    for size in ((1024, 128, 14336), (1536, 32, 14336), (512, 256, 7168), (256, 512, 4608), (512, 1024, 14336)):
        assert not ops.fp8_tiled(*size)
