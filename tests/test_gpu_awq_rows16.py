"""int4 products of at most 16 rows (awq_rows16.h) at the edges of its rule: one row, the last rows of either form, one row
beyond; splits of one stage (a group a wave), two, and many with a remainder; each way out of the kernel."""
import pytest
import torch

from test_gpu_ops import _awq_case, _gemm_close

pytestmark = pytest.mark.gpu
DEV = "cuda"
# (K, N): one group a wave / two / a split of 13 groups in turns of 8, last split shorter / one split of 28 groups
SHAPES = [(512, 128), (4096, 4096), (4096, 6144), (14336, 4096), (3584, 32768)]


def _case(M, K, N, dtype, interleave=False):
    import oracle
    from sglang_security_amd import ops

    x, qw, sc, qz = _awq_case(M, K, N, 128, dtype, seed=M + K + N)
    w = [t.to(DEV) for t in (qw, sc, qz)]
    if interleave:
        w = ops.awq_interleave_gate_up(*w)
    return ops, x.to(DEV), (ops.awq_repack(w[0]), w[1], w[2]), oracle.awq_gemm(x, qw, sc, qz)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17])
@pytest.mark.parametrize("K,N", SHAPES[:4])
def test_products_and_split_sums(M, K, N, dtype):
    ops, x, w, want = _case(M, K, N, dtype)
    wide = torch.randn(M, K + 64, device=DEV).to(dtype)       # rows with something behind them
    wide[:, :K] = x
    part = torch.full((ops.awq_gemm_partial_splits(M, N, K), M, N), float("nan"), device=DEV)
    ops.awq_gemm_partial(wide[:, :K], *w, part)
    _gemm_close(part.sum(0).to(dtype).cpu(), want, dtype)
    bias = torch.randn(N, device=DEV).to(dtype)
    work = torch.zeros(max(ops.awq_gemm_workspace_bytes(M, N, K), 256), dtype=torch.uint8, device=DEV)
    out = torch.full((M + 1, N + 8), 7.0, dtype=dtype, device=DEV)
    for _ in range(2):                                          # the tickets are back at zero
        ops.awq_gemm(x, *w, bias=bias, out=out[:M, :N], workspace=work)
        _gemm_close(out[:M, :N].cpu(), (want.float() + bias.float().cpu()).to(dtype), dtype)
    assert (out[M:] == 7).all() and (out[:, N:] == 7).all()


@pytest.mark.parametrize("M", [1, 8, 9, 16])
@pytest.mark.parametrize("K,N", [(512, 256), (3584, 32768)])
def test_gated_activation(M, K, N):
    ops, x, w, want = _case(M, K, N, torch.bfloat16, interleave=True)
    out = torch.full((M, N // 2), float("nan"), dtype=torch.bfloat16, device=DEV)
    xs = torch.zeros(N // 256, M + 2, device=DEV)
    ops.awq_gemm_silu_mul(x, *w, out, None, xs)
    gate, up = want.float().chunk(2, 1)
    act = torch.nn.functional.silu(gate).to(torch.bfloat16).float() * up
    _gemm_close(out.cpu(), act, torch.bfloat16)
    sums = out.double().view(M, -1, 128).sum(2).t()
    # 64 additions of fp32 in either addend, values below 4
    torch.testing.assert_close(xs[:, :M].double(), sums, rtol=0, atol=128 * 4 * 2 ** -23 * 8)
    assert (xs[:, M:] == 0).all()


@pytest.mark.parametrize("M", [1, 16])
def test_zero_scales_and_rows_that_are_not_numbers(M):
    """A column whose scales are zero is zero; a row of x that is not a number stays with itself."""
    ops, x, (packed, sc, qz), _ = _case(M, 4096, 6144, torch.bfloat16)
    sc = sc.clone()
    sc[:, 5] = 0
    x = x.clone()
    clean = torch.empty(M, 6144, dtype=torch.bfloat16, device=DEV)
    part = torch.empty(ops.awq_gemm_partial_splits(M, 6144, 4096), M, 6144, device=DEV)
    ops.awq_gemm_partial(x, packed, sc, qz, part)
    clean = part.sum(0)
    assert (clean[:, 5] == 0).all() and (clean[:, 6] != 0).any()
    x[M - 1, 100] = float("nan")
    ops.awq_gemm_partial(x, packed, sc, qz, part)
    assert torch.equal(part.sum(0)[: M - 1], clean[: M - 1]) and part.sum(0)[M - 1].isnan().all()


@pytest.mark.parametrize("M", [1, 8, 9, 16, 17])
def test_chain_gives_the_bits_of_the_separate_launches(M):
    """gate_up (+ activation) and down as one call and as two, with the splits and the block sums of either."""
    ops, x, gu, _ = _case(M, 1024, 3072, torch.bfloat16, interleave=True)
    _, _, dn, _ = _case(M, 1536, 1024, torch.bfloat16)
    xs = x.float().view(M, -1, 128).sum(2).t().contiguous()
    act = torch.empty(2, M, 1536, dtype=torch.bfloat16, device=DEV)
    xs_act = torch.zeros(2, 12, M, device=DEV)
    part = torch.full((2, ops.awq_gemm_partial_splits(M, 1024, 1536), M, 1024), float("nan"), device=DEV)
    ops.awq_gemm_silu_mul(x, *gu, act[0], xs, xs_act[0])
    ops.awq_gemm_partial(act[0], *dn, part[0], xs_act[0])
    sync = ops.awq_chain_sync(DEV)
    ops.awq_chain([ops.chain_silu_mul(x, *gu, xs, act[1], xs_act[1]), ops.chain_partial(act[1], *dn, xs_act[1], part[1])], sync)
    assert ops.awq_chain_status(sync) == 0 and int(sync.abs().sum()) == 0
    assert torch.equal(act[0], act[1]) and torch.equal(xs_act[0], xs_act[1]) and torch.equal(part[0], part[1])


@pytest.mark.parametrize("dtype,bound", [(torch.float16, 1.1e-5), (torch.bfloat16, 1.1e-6)])
@pytest.mark.parametrize("M", [1, 16])
def test_distance_from_64_bits(M, dtype, bound):
    """Two sums of about (OFF + z) sqrt(n) are taken off one another, n = 64 (fp16, OFF = 1024) or 128 (bf16, 128) of x at a time,
    each with the roundings of n / 32 steps: 3.5e-4 a half in fp16, 1e-4 a group in bf16, of a group's 74 that is 7e-6 and 1e-6
    (no more than a product whose roundings are all of the last step's size); with some for what rounds inside an instruction.
    Whole groups give 1.22e-5 in fp16."""
    from sglang_security_amd import ops

    K = N = 4096
    shifts = torch.tensor([0, 4, 1, 5, 2, 6, 3, 7], device=DEV) * 4
    nib = lambda t: ((t[..., None] >> shifts) & 15).flatten(-2).double()
    off = of = 0.0
    for seed in range(4):
        g = torch.Generator(device=DEV).manual_seed(seed)
        words = lambda rows: torch.randint(-(2 ** 31), 2 ** 31 - 1, (rows, N // 8), dtype=torch.int32, generator=g, device=DEV)
        qw, qz = words(K), words(K // 128)
        sc = (torch.rand(K // 128, N, generator=g, device=DEV) * 0.01 + 0.001).to(dtype)
        x = torch.randn(M, K, generator=g, device=DEV).to(dtype)
        part = torch.empty(ops.awq_gemm_partial_splits(M, N, K), M, N, device=DEV)
        ops.awq_gemm_partial(x, ops.awq_repack(qw), sc, qz, part)
        want = x.double() @ ((nib(qw) - nib(qz).repeat_interleave(128, 0)) * sc.double().repeat_interleave(128, 0))
        off += (part.double().sum(0) - want).square().sum().item()
        of += want.square().sum().item()
    assert (off / of) ** 0.5 <= bound


@pytest.mark.parametrize("M", [1, 9, 16])
@pytest.mark.parametrize("K,N", [(512, 256), (4096, 128), (4608, 128), (6656, 256), (14336, 128)])
def test_last_block_adds_every_split_in_order(M, K, N, monkeypatch):
    """One to 28 splits of one stage each, counts that are and are no multiple of those asked for at once."""
    ops, x, w, _ = _case(M, K, N, torch.bfloat16)
    monkeypatch.setenv("SGLK_AWQ_WIDE", "2")
    monkeypatch.setenv("SGLK_AWQ_WIDE_SPS", "1")
    part = torch.full((ops.awq_gemm_partial_splits(M, N, K), M, N), float("nan"), device=DEV)
    assert len(part) == K // 512
    ops.awq_gemm_partial(x, *w, part)
    want = part[0].clone()
    for p in part[1:]:
        want += p
    work = torch.zeros(ops.awq_gemm_workspace_bytes(M, N, K), dtype=torch.uint8, device=DEV)
    for _ in range(2):
        assert torch.equal(ops.awq_gemm(x, *w, workspace=work), want.bfloat16())


@pytest.mark.parametrize("batch", [6, 16, 17])
def test_decode_step_makes_only_block_sums_that_are_read(batch):
    """Up to 16 rows the products form the sums of x themselves: the step's norms, attention and gated activation leave the
    block sums alone, and its logits are the bits of a step that makes them."""
    from sglang_security_amd.decode_runner import LlamaConfig, LlamaDecoder

    logits = []
    for forced in (False, True):
        dec = LlamaDecoder(LlamaConfig.tiny(), batch=batch, pool_slots=1 + 64 + batch * 24, max_ctx=96, device=DEV, seed=0)
        dec.setup_shared_prefix_batch(prefix_len=64, suffix_len=5)
        dec.enable_shared_prefix(True)
        assert dec.enable_fusion(True)
        buffers = (dec.xs_hidden, dec.xs_attn, dec.xs_act)
        if forced:
            dec.block_sums = buffers
        for t in buffers:
            t.fill_(float("nan"))
        dec.step()
        torch.cuda.synchronize()
        assert all(bool(t.isnan().all()) for t in buffers) == (batch <= 16 and not forced)
        logits.append(dec.logits.clone())
    assert torch.isfinite(logits[0].float()).all() and torch.equal(logits[0], logits[1])
