"""fp8 products of at most 64 rows (fp8_direct.h): the first and last rows of each form, one row beyond; column counts on
either side of each tile rule and with strips that do not fill a block; k-blocks that do not fill a turn or a stage."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
F8 = torch.float8_e4m3fn


def _fp8(shape, g):
    return (torch.randn(shape, generator=g, device=DEV)).to(F8)


@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32, 33, 64, 65])
@pytest.mark.parametrize("N,K", [(16, 128), (48, 1152), (4096, 512), (4096, 8320), (4112, 640), (16384 - 16, 384), (16384 + 16, 384),
                                 (16384 + 16, 2688), (48, 8320), (1280, 18432), (4080, 14336), (10240, 4096)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16])
def test_products(M, N, K, out_dtype):
    from sglang_security_amd import ops

    g = torch.Generator(device=DEV).manual_seed(M * N + K)
    wide = _fp8((M, K + 64), g)                                 # rows with something behind them
    x, w = wide[:, :K], _fp8((N, K), g)
    sa, sb = (0.05 + 0.1 * torch.rand(n, 1, generator=g, device=DEV) for n in (M, N))
    bias = torch.randn(N, generator=g, device=DEV).to(out_dtype)
    packed = ops.fp8_repack(w)
    exact = x.double() @ w.double().t()
    # the fp8 matrix instructions add products in a fixed point below the largest of them, 2^-12.5 of it at most over one k-block
    # (16x16x32 and 16x16x128 alike, against 64-bit sums); blocks add up like a random walk, one bit in hand
    most = x.double().abs().amax(1, keepdim=True) * w.double().abs().amax(1)
    bound = most * 2.0 ** -11.5 * max(1.0, K / 128) ** 0.5
    splits = ops.fp8_mm_packed_partial_splits(M, N, K)
    part = torch.full((splits, M, N), float("nan"), device=DEV)
    assert ops.fp8_mm_packed_partial(x, packed, part) == splits
    assert ((part.double().sum(0) - exact).abs() <= bound).all()
    want = exact * sa.double() * sb.double().t()
    ulp = 2.0 ** (-8 if out_dtype == torch.bfloat16 else -11)
    ws = torch.empty(max(ops.fp8_mm_packed_workspace_bytes(M, N, K), 16), dtype=torch.uint8, device=DEV)
    for work in (ws, None):
        for b in (None, bias):
            out = torch.full((M + 1, N + 8), 7.0, dtype=out_dtype, device=DEV)
            ops.fp8_scaled_mm_packed(x, packed, sa, sb, out_dtype, b, out[:M, :N], work)
            ref = want if b is None else want + b.double()
            off = (out[:M, :N].double() - ref).abs()
            assert (off <= ref.abs() * ulp + bound * sa.double() * sb.double().t() * 2 + 1e-6).all()
            assert (out[M:] == 7).all() and (out[:, N:] == 7).all()


@pytest.mark.parametrize("M", [1, 40])
def test_codes_that_are_not_numbers_stay_in_their_rows_and_columns(M):
    from sglang_security_amd import ops

    g = torch.Generator(device=DEV).manual_seed(M)
    x, w = _fp8((M, 1024), g), _fp8((4096, 1024), g)
    part = torch.empty(ops.fp8_mm_packed_partial_splits(M, 4096, 1024), M, 4096, device=DEV)
    ops.fp8_mm_packed_partial(x, ops.fp8_repack(w), part)
    clean = part.sum(0).clone()
    x.view(torch.uint8)[M - 1, 77] = 0x7F
    w.view(torch.uint8)[100, 5] = 0xFF
    ops.fp8_mm_packed_partial(x, ops.fp8_repack(w), part)
    got = part.sum(0)
    assert got[M - 1].isnan().all() and got[:, 100].isnan().all()
    keep = torch.ones_like(got, dtype=torch.bool)
    keep[M - 1] = False
    keep[:, 100] = False
    assert torch.equal(got[keep], clean[keep])


@pytest.mark.parametrize("M", [33, 64])
@pytest.mark.parametrize("K", [128, 256, 512, 1024, 1152])
def test_few_stages(M, K):
    """More than 32 rows of one k-block, of two, of one stage, two and three: the weights' ring is no longer than that."""
    test_products(M, 1040, K, torch.bfloat16)
