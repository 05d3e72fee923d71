"""16-bit products, of at most 32 rows (dense_direct.h) and of more: the first and last rows of each form and one beyond; column counts on
either side of each tile rule, with strips that do not fill a block; k-blocks that do not fill a turn or a split."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32, 33])
@pytest.mark.parametrize("N,K", [(512, 128), (528, 1152), (2560, 2688), (4112, 640), (8192 - 16, 384), (8192 + 16, 384), (16384 - 16, 256),
                                 (16384 + 16, 256), (1024, 8320)])
def test_products(M, N, K, dtype):
    from sglang_security_amd import ops

    g = torch.Generator(device=DEV).manual_seed(M * N + K)
    wide = torch.randn(M, K + 64, generator=g, device=DEV).to(dtype)    # rows with something behind them
    x, w = wide[:, :K], torch.randn(N, K, generator=g, device=DEV).to(dtype)
    bias = torch.randn(N, generator=g, device=DEV).to(dtype)
    packed = ops.dense_repack(w)
    exact = x.double() @ w.double().t()
    bound = (x.double().abs() @ w.double().abs().t()) * 2.0 ** -21      # fp32 sums of K products
    splits = ops.dense_gemm_partial_splits(M, N, K)
    part = torch.full((splits, M, N), float("nan"), device=DEV)
    assert ops.dense_gemm_packed_partial(x, packed, part) == splits
    assert ((part.double().sum(0) - exact).abs() <= bound).all()
    ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    for b in (None, bias):
        want = exact if b is None else exact + b.double()
        tol = want.abs() * ulp + bound * 2
        out = torch.full((M + 1, N + 8), 7.0, dtype=dtype, device=DEV)
        ops.dense_gemm_packed(x, packed, b, out[:M, :N])
        assert ((out[:M, :N].double() - want).abs() <= tol).all()
        assert (out[M:] == 7).all() and (out[:, N:] == 7).all()
        ws = torch.empty(max(splits * M * N, 4), device=DEV)
        out = torch.full((M, N), float("nan"), dtype=dtype, device=DEV)
        ops.dense_gemm_packed_ws(x, packed, b, out, ws)
        assert ((out.double() - want).abs() <= tol).all()
        # the row-major weight, with the same bits up to 16 rows
        rows = torch.empty(M, N, dtype=dtype, device=DEV)
        ops.dense_gemm_nt(x, w, b, rows, torch.empty(max(ops.dense_gemm_workspace_bytes(M, N, K), 16), dtype=torch.uint8, device=DEV))
        assert ((rows.double() - want).abs() <= tol).all() and (M > 16 or torch.equal(rows, out))
        assert ((ops.dense_gemm_nt(x, w, b).double() - want).abs() <= tol).all()
        assert M > 16 or torch.equal(ops.dense_gemm_nt(x, w, b), ops.dense_gemm_packed(x, packed, b))


@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(8192, 2688), (8208, 2688), (16400, 1152), (16400, 2688), (65536 + 16, 1152)])
def test_wide_products(M, N, K):
    """Wide outputs with several k-blocks a wave and a last turn that is not full; the last column count of 32 a block and the
    first of 64, inner dimensions on either side of sixteen waves."""
    test_products(M, N, K, torch.bfloat16)


@pytest.mark.parametrize("M", [24, 25])
def test_widest_products_around_the_last_rows_of_the_direct_form(M):
    test_products(M, 65536 + 16, 640, torch.bfloat16)
    test_products(M, 65536 - 16, 640, torch.bfloat16)


@pytest.mark.parametrize("kblocks", [1, 2, 3, 4, 5, 7, 8, 9, 11])
@pytest.mark.parametrize("M,N", [(33, 80), (64, 16384), (64, 16400), (65, 8192), (65, 8208), (64, 24448), (64, 24464), (65, 12176), (130, 8208)])
def test_staged_products(M, N, kblocks):
    """The staged kernel: rounds of two and of four k-blocks that are whole, short and ragged, one and two strips a wave on
    either side of the rule, column counts and row lengths that sixteen-byte stores cannot take, the last strip of a block."""
    from sglang_security_amd import ops

    K, dtype = 128 * kblocks, torch.bfloat16
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x, w = (torch.randn(r, K, generator=g, device=DEV).to(dtype) for r in (M, N))
    bias = torch.randn(N, generator=g, device=DEV).to(dtype)
    want = x.double() @ w.double().t() + bias.double()
    tol = want.abs() * 2.0 ** -8 + (x.double().abs() @ w.double().abs().t()) * 2.0 ** -20
    packed = torch.full((M + 1, N + 8), 7.0, dtype=dtype, device=DEV)
    ops.dense_gemm_packed(x, ops.dense_repack(w), bias, packed[:M, :N])
    assert ((packed[:M, :N].double() - want).abs() <= tol).all()
    assert (packed[M:] == 7).all() and (packed[:, N:] == 7).all()
    rows = torch.full((M + 1, N + 5), 7.0, dtype=dtype, device=DEV)     # single elements
    ops.dense_gemm_nt(x, w, bias, rows[:M, :N])
    assert torch.equal(rows[:M, :N], packed[:M, :N]) and (rows[M:] == 7).all() and (rows[:, N:] == 7).all()
    n = N - 3                                                           # the last piece is not whole
    some = torch.full((M, N), 7.0, dtype=dtype, device=DEV)
    ops.dense_gemm_nt(x, w[:n], bias[:n], some[:, :n])
    assert torch.equal(some[:, :n], packed[:M, :n]) and (some[:, n:] == 7).all()


@pytest.mark.parametrize("M", [1, 16])
@pytest.mark.parametrize("N", [2560, 16384])
def test_rows_and_columns_that_are_not_numbers(M, N):
    from sglang_security_amd import ops

    g = torch.Generator(device=DEV).manual_seed(N)
    x = torch.randn(M, 1280, generator=g, device=DEV).bfloat16()
    w = torch.randn(N, 1280, generator=g, device=DEV).bfloat16()
    clean = ops.dense_gemm_packed(x, ops.dense_repack(w))
    x[M - 1, 7] = float("inf")
    w[100, 5] = float("nan")
    got = ops.dense_gemm_packed(x, ops.dense_repack(w))
    assert not got[M - 1].isfinite().any() and got[:, 100].isnan().all()
    keep = torch.ones_like(got, dtype=torch.bool)
    keep[M - 1] = False
    keep[:, 100] = False
    assert torch.equal(got[keep], clean[keep])


@pytest.mark.parametrize("M,N,K", [(25, 5104, 2560), (26, 5104, 2560), (24, 5120, 5376), (25, 5120, 5376), (32, 6992, 4224), (16, 16384, 5120), (12, 16416, 4096),
                                   (13, 16416, 4096), (1, 16416, 3072), (1, 16416, 3200), (1, 16416, 4224), (16, 22272, 2944), (16, 22288, 4224), (16, 11008, 5120),
                                   (16, 11008, 5248), (1, 11008, 8192), (1, 11008, 8320), (32, 24576, 4096), (32, 24576, 4224), (16, 49136, 1152), (16, 49152, 1152),
                                   (16, 49152, 1280), (16, 49152, 2048), (17, 49152, 1152), (5, 16400, 1536), (16, 8192, 6144), (16, 8192, 6272), (7, 40960, 2560),
                                   (8, 40960, 2560), (16, 20480, 4096), (24, 20480, 4096)])
def test_sides_of_the_rules(M, N, K):
    """The last and the first calls of the staged and the direct kernel, on both layouts: right sums on each, and finished rows of the
    streaming layout are the rounded split sums."""
    from sglang_security_amd import ops

    g = torch.Generator(device=DEV).manual_seed(M * N + K)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = torch.randn(N, K, generator=g, device=DEV).bfloat16()
    bias = torch.randn(N, generator=g, device=DEV).bfloat16()
    packed = ops.dense_repack(w)
    want = x.double() @ w.double().t()
    bound = (x.double().abs() @ w.double().abs().t()) * 2.0 ** -20     # fp32 sums of K products
    splits = ops.dense_gemm_partial_splits(M, N, K)
    part = torch.full((splits, M, N), float("nan"), device=DEV)
    assert ops.dense_gemm_packed_partial(x, packed, part) == splits
    total = part[0]
    for p in part[1:]:
        total = total + p
    assert ((total.double() - want).abs() <= bound).all()
    ws = torch.empty(max(splits * M * N, 4), device=DEV)
    finished = ops.dense_gemm_packed_ws(x, packed, bias, torch.empty(M, N, dtype=torch.bfloat16, device=DEV), ws)
    assert torch.equal(finished, (total + bias.float()).bfloat16())
    want += bias.double()
    tol = want.abs() * 2.0 ** -8 + 2 * bound
    need = max(ops.dense_gemm_workspace_bytes(M, N, K), 16)
    for got in (ops.dense_gemm_packed(x, packed, bias), ops.dense_gemm_nt(x, w, bias),
                ops.dense_gemm_nt(x, w, bias, None, torch.empty(need, dtype=torch.uint8, device=DEV))):
        assert ((got.double() - want).abs() <= tol).all()


@pytest.mark.parametrize("M", [33, 64, 130])
@pytest.mark.parametrize("N,kblocks", [(1040, 1), (1040, 2), (1040, 3), (16640, 1), (65536, 1), (65536 + 16, 2), (65536, 3)])
def test_split_sums_of_few_k_blocks(M, N, kblocks):
    """Rings of one, two and four k-blocks, one and two strips a wave, where the sums stay in 32 bits."""
    from sglang_security_amd import ops

    K = 128 * kblocks
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x, w = (torch.randn(r, K, generator=g, device=DEV).bfloat16() for r in (M, N))
    splits = ops.dense_gemm_partial_splits(M, N, K)
    part = torch.full((splits, M, N), float("nan"), device=DEV)
    assert ops.dense_gemm_packed_partial(x, ops.dense_repack(w), part) == splits
    bound = (x.double().abs() @ w.double().abs().t()) * 2.0 ** -21      # fp32 sums of K products
    assert ((part.double().sum(0) - x.double() @ w.double().t()).abs() <= bound).all()
    rows = ops.dense_gemm_nt(x, w)
    assert torch.equal(rows, ops.dense_gemm_packed(x, ops.dense_repack(w)))
