"""Products of many rows on the tiles of prefill_tile.h: every row height and strip width the plan picks, ragged rows, int4 against 16-bit
weights bit for bit, values that are not finite, pitches beyond 32-bit offsets."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _int4(K, N, dtype, seed, group=128):
    g = torch.Generator(device=DEV).manual_seed(seed)
    word = lambda *shape: torch.randint(-2 ** 31, 2 ** 31, shape, device=DEV, generator=g, dtype=torch.int64).int()
    scales = (torch.rand(K // group, N, device=DEV, generator=g) * 0.02).to(dtype)
    return word(K, N // 8), scales, word(K // group, N // 8), g


def _same(a, b):
    return torch.equal(torch.nan_to_num(a, 7.0), torch.nan_to_num(b, 7.0)) and torch.equal(a.isnan(), b.isnan())


# rows a block and strips: 128 x 128; 192 x 128; 128 x 192; 192 x 192; 256 x 192; whole rounds of 256 columns with 192 and with 128
# behind them; 256 columns alone; an odd number of k-blocks, one k-block, a single row
@pytest.mark.parametrize("M,K,N,group", [(300, 384, 1024, 128), (1152, 1024, 4096, 256), (1000, 256, 6144, 128), (1400, 640, 6144, 128),
                                         (2048, 512, 6144, 512), (1152, 256, 28672, 128), (2048, 128, 28672, 128), (500, 384, 28672, 128),
                                         (1, 128, 128, 128), (257, 1152, 640, 384)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_int4_gives_the_bits_of_its_dequantised_weights(M, K, N, group, dtype):
    """Both kinds add along K in the same order, whatever the tile, so the same weights give the same bits; the 16-bit kind against
    64-bit sums: the result's one rounding and its fp32 sums."""
    from sglang_security_amd import ops

    qw, sc, qz, g = _int4(K, N, dtype, M + K + N, group)
    x = torch.randn(M, K + 16, device=DEV, generator=g).to(dtype)[:, 8: K + 8]
    bias = torch.randn(N, device=DEV, generator=g).to(dtype)
    packed = ops.awq_repack(qw)
    w = ops.awq_dequantize_packed_nk(packed, sc, qz)
    buf = torch.full((M + 1, N + 8), 7.0, dtype=dtype, device=DEV)
    got = ops.awq_gemm_prefill(x, packed, sc, qz, None, buf[:M, :N])
    assert bool((buf[M] == 7).all()) and bool((buf[:, N:] == 7).all())
    assert torch.equal(got, ops.dense_gemm_prefill(x, w))
    got = ops.awq_gemm_prefill(x, packed, sc, qz, bias)
    assert torch.equal(got, ops.dense_gemm_prefill(x, w, bias))
    want = x.double() @ w.double().t() + bias.double()
    unit = 2 ** -8 if dtype == torch.bfloat16 else 2 ** -11   # half a step of 8 or 11 significant bits is at most that of a number
    assert ((got.double() - want).norm() / want.norm()).item() < unit
    assert ((got.double() - want).abs() <= unit * want.abs() + 1e-5 * want.abs().max()).all()


# strips of 192 columns of which the last has 64 or 128: 128, 192 and 256 rows a block, behind whole strips of 256 and without any
@pytest.mark.parametrize("M,K,N,rows,left", [(627, 128, 6784, 128, 64), (627, 256, 6656, 128, 128), (563, 128, 22016, 128, 128),
                                             (1600, 384, 4096, 192, 64), (819, 128, 7424, 192, 128), (2355, 128, 7424, 192, 64),
                                             (2112, 256, 4096, 256, 64), (1100, 256, 7168, 256, 64), (800, 128, 27648, 256, 128),
                                             (3200, 128, 28672, 256, 128), (3700, 128, 28672, 256, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_a_last_strip_that_is_not_full(M, K, N, rows, left, dtype):
    from sglang_security_amd import ops

    block, _, whole, _, narrow = ops.awq_gemm_prefill_tiles(M, N, K)
    assert (block, narrow, (N - 256 * whole) % narrow) == (rows, 192, left)
    test_int4_gives_the_bits_of_its_dequantised_weights(M, K, N, 128, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_scales_and_biases_that_start_anywhere(dtype):
    """Scales off 4 bytes, biases off 8: the same numbers as from aligned copies (the gated form, which asks for whole pairs, refuses)."""
    from sglang_security_amd import ops
    from sglang_security_amd._lib import SglkError

    M, K, N = 300, 256, 512
    qw, sc, qz, g = _int4(K, N, dtype, 11)
    x = torch.randn(M, K, device=DEV, generator=g).to(dtype)
    off = lambda t: torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)
    bias = torch.randn(N, device=DEV, generator=g).to(dtype)
    packed = ops.awq_repack(qw)
    w = ops.awq_dequantize_packed_nk(packed, sc, qz)
    want = x.double() @ w.double().t() + bias.double()
    unit = 2 ** -8 if dtype == torch.bfloat16 else 2 ** -11   # as above
    for got in (ops.awq_gemm_prefill(x, packed, off(sc), qz, bias), ops.awq_gemm_prefill(x, packed, sc, qz, off(bias)),
                ops.dense_gemm_prefill(x, w, off(bias))):
        assert ((got.double() - want).abs() <= unit * want.abs() + 1e-5 * want.abs().max()).all()
    with pytest.raises(SglkError):
        ops.awq_gemm_prefill_silu_mul(x, packed, off(sc), qz, torch.empty(M, N // 2, dtype=dtype, device=DEV))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_values_that_are_not_finite(dtype):
    """Infinite and NaN scales and activations reach what they reach through the dequantised weights, and nothing else."""
    from sglang_security_amd import ops

    qw, sc, qz, g = _int4(512, 1024, dtype, 3)
    sc[1, 5], sc[3, 70], sc[0, 200] = float("inf"), float("nan"), float("-inf")
    x = torch.randn(300, 512, device=DEV, generator=g).to(dtype)
    x[7, 100], x[140, 3] = float("inf"), float("nan")
    packed = ops.awq_repack(qw)
    got = ops.awq_gemm_prefill(x, packed, sc, qz)
    assert _same(got, ops.dense_gemm_prefill(x, ops.awq_dequantize_packed_nk(packed, sc, qz)))
    clean = torch.ones_like(got, dtype=torch.bool)
    clean[[7, 140]] = False
    clean[:, [5, 70, 200]] = False
    assert bool(got[clean].isfinite().all())


def test_pitches_beyond_32_bit_offsets():
    from sglang_security_amd import ops

    qw, sc, qz, g = _int4(256, 128, torch.bfloat16, 4)
    x = torch.randn(5, 256, device=DEV, generator=g).to(torch.bfloat16)
    far = torch.empty(5 * (1 << 23), dtype=torch.bfloat16, device=DEV).as_strided((5, 256), (1 << 23, 1))
    far.copy_(x)
    packed = ops.awq_repack(qw)
    w = ops.awq_dequantize_packed_nk(packed, sc, qz)
    want = (x.double() @ w.double().t()).float()
    for got in (ops.awq_gemm_prefill(far, packed, sc, qz), ops.dense_gemm_prefill(far, w), ops.awq_gemm_prefill(x, packed, sc, qz)):
        torch.testing.assert_close(got.float(), want, rtol=2 ** -8, atol=1e-4)


def test_linear_method_of_many_rows():
    """AWQLinearMethod with more rows than the few-row kernels take, on either side of the rule: the product of the dequantised weight."""
    from types import SimpleNamespace

    from sglang_security_amd import ops
    from sglang_security_amd.quantization.awq import AWQLinearMethod

    for M, K, N in ((300, 4096, 28672), (300, 512, 256)):
        qw, sc, qz, g = _int4(K, N, torch.bfloat16, M)
        packed = ops.awq_repack(qw)
        layer = SimpleNamespace(sglk_shape=(K, N), sglk_fusable=True, sglk_packed=packed, scales=sc, qzeros=qz, qweight=None)
        x = torch.randn(M, K, device=DEV, generator=g).to(torch.bfloat16)
        bias = torch.randn(N, device=DEV, generator=g).to(torch.bfloat16)
        got = AWQLinearMethod(None).apply(layer, x, bias)
        want = (x.double() @ ops.awq_dequantize_packed_nk(packed, sc, qz).double().t()).to(torch.bfloat16) + bias
        assert ((got.double() - want.double()).norm() / want.double().norm()).item() < 2 ** -8


def _linear(M, K, N):
    from types import SimpleNamespace

    from sglang_security_amd import ops

    qw, sc, qz, g = _int4(K, N, torch.bfloat16, M)
    layer = SimpleNamespace(sglk_shape=(K, N), sglk_fusable=True, sglk_packed=ops.awq_repack(qw), scales=sc, qzeros=qz, qweight=None)
    assert ops.awq_prefill_fused(M, N, K)
    return layer, torch.randn(M * K + 8, device=DEV, generator=g).to(torch.bfloat16)


def test_linear_method_takes_rows_that_start_anywhere():
    from sglang_security_amd.quantization.awq import AWQLinearMethod

    layer, flat = _linear(300, 4096, 28672)
    rows = lambda at: flat[at: at + 300 * 4096].view(300, 4096)
    got = AWQLinearMethod(None).apply(layer, rows(1))
    want = AWQLinearMethod(None).apply(layer, rows(1).clone())
    assert ((got.double() - want.double()).norm() / want.double().norm()).item() < 2 ** -8   # a rounding each, sums in another order


def test_linear_method_refuses_rows_of_another_type_or_length():
    from sglang_security_amd.quantization.awq import AWQLinearMethod

    layer, flat = _linear(300, 4096, 28672)
    rows = flat[: 300 * 4096].view(300, 4096)
    for wrong in (rows.half(), rows.float(), rows[:, :2048], rows.view(150, 8192).repeat(2, 1)):
        with pytest.raises(RuntimeError):
            AWQLinearMethod(None).apply(layer, wrong)


def test_linear_method_keeps_the_gradient_of_its_rows():
    from sglang_security_amd import ops
    from sglang_security_amd.quantization.awq import AWQLinearMethod

    layer, flat = _linear(300, 4096, 28672)
    rows = flat[: 300 * 4096].view(300, 4096).clone().requires_grad_()
    out = AWQLinearMethod(None).apply(layer, rows)
    weights = torch.randn_like(out)
    out.backward(weights)
    w = ops.awq_dequantize_packed_nk(layer.sglk_packed, layer.scales, layer.qzeros)
    want = weights.float() @ w.float()
    assert ((rows.grad.float() - want).norm() / want.norm()).item() < 2 ** -8   # one rounding to bf16


def test_linear_method_follows_autocast():
    from sglang_security_amd.quantization.awq import AWQLinearMethod

    layer, flat = _linear(300, 4096, 28672)
    rows = flat[: 300 * 4096].view(300, 4096)
    want = AWQLinearMethod(None).apply(layer, rows)
    for dtype in (torch.bfloat16, torch.float16):
        with torch.autocast("cuda", dtype):
            got = AWQLinearMethod(None).apply(layer, rows)
        assert got.dtype == dtype and ((got.double() - want.double()).norm() / want.double().norm()).item() < 2 ** -8   # `want` has one rounding to bf16


def test_rule_stays_where_it_was_measured():
    from sglang_security_amd import ops

    assert ops.awq_prefill_fused(1152, 28672, 4096) and ops.awq_prefill_fused(256, 28672, 4096)
    assert not ops.awq_prefill_fused(256, 4096, 14336)          # few blocks along a long inner dimension
    assert not ops.awq_prefill_fused(300, 1024, 512) and not ops.awq_prefill_fused(300, 28672, 4000)


@pytest.mark.parametrize("M,K,inter", [(300, 256, 128), (256, 512, 14336), (1152, 256, 14336), (700, 384, 6144), (2048, 128, 14336)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gated_rows_are_those_of_two_launches(M, K, inter, dtype):
    """Strips of 256 and of 128 columns: the activation's bits are those of the product followed by act_and_mul."""
    from sglang_security_amd import ops

    qw, sc, qz, g = _int4(K, 2 * inter, dtype, M + inter)
    x = torch.randn(M, K, device=DEV, generator=g).to(dtype)
    want = torch.empty(M, inter, dtype=dtype, device=DEV)
    ops.act_and_mul(want, ops.awq_gemm_prefill(x, ops.awq_repack(qw), sc, qz), 0)
    qi, si, zi = ops.awq_interleave_gate_up(qw, sc, qz)
    buf = torch.full((M + 1, inter + 8), 7.0, dtype=dtype, device=DEV)
    ops.awq_gemm_prefill_silu_mul(x, ops.awq_repack(qi), si, zi, buf[:M, :inter])
    assert torch.equal(buf[:M, :inter], want)
    assert bool((buf[M] == 7).all()) and bool((buf[:, inter:] == 7).all())
