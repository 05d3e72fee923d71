"""int4 products of more than 64 rows on blocks of 96 and 128 (awq_tall.h), against the oracle and against 64-bit sums."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(M, K, N, seed):
    from test_gpu_ops import _awq_case

    return _awq_case(M, K, N, 128, torch.bfloat16, seed=seed)


def _weight64(qw, sc, qz):
    shifts = torch.tensor([0, 4, 1, 5, 2, 6, 3, 7], device=qw.device) * 4
    nib = lambda t: ((t[..., None] >> shifts) & 15).flatten(-2).double()
    return (nib(qw) - nib(qz).repeat_interleave(128, 0)) * sc.double().repeat_interleave(128, 0)


def _wide(monkeypatch, call):
    """The same call on the wide kernel."""
    monkeypatch.setenv("SGLK_AWQ_WIDE", "1")
    out = call()
    monkeypatch.delenv("SGLK_AWQ_WIDE")
    return out


def _takes(M, N, K, rows, splits=1, gated=False):
    """The size is one that blocks of so many rows take, K in so many splits, whoever forms the block sums."""
    from sglang_security_amd import ops

    for sums in (False, True):
        assert ops.awq_gemm_tall_rows(M, N, K, gated=gated, sums=sums) == (rows, splits)


@pytest.mark.parametrize("M,K,inter,block", [(65, 4096, 14336, 96), (96, 4096, 14336, 96), (97, 4096, 14336, 128), (128, 4096, 14336, 128),
                                             (200, 4096, 14336, 128), (255, 4096, 14336, 128), (192, 1024, 5632, 96), (65, 512, 8320, 96),
                                             (97, 512, 8320, 128), (65, 1024, 8320, 96), (96, 1536, 14336, 96), (97, 1536, 8320, 128),
                                             (193, 1024, 4224, 128), (128, 2560, 8320, 128)])
def test_gated_rows_and_their_sums(monkeypatch, M, K, inter, block):
    """Every output of the gated form, ragged rows among them, with and without the producer's block sums: the unfused sequence's
    roundings, so half an ulp of bf16 twice (2^-8 each) beside the product's own 1e-6; rows behind M stay as they were.  With the
    producer's sums, rows and the sums left for the next product are the wide kernel's bits."""
    from sglang_security_amd import ops

    _takes(M, 2 * inter, K, block, gated=True)
    x, qw, sc, qz = (t.to(DEV) for t in _case(M, K, 2 * inter, M + K))
    qi, si, zi = ops.awq_interleave_gate_up(qw, sc, qz)
    packed = ops.awq_repack(qi)
    gu = (x.double() @ _weight64(qw, sc, qz)).to(torch.bfloat16).double()
    silu = torch.nn.functional.silu(gu[:, :inter]).to(torch.bfloat16).double()
    want = silu * gu[:, inter:]
    wide = torch.nn.functional.pad(x, (8, 8))[:, 8:-8]  # rows with a pitch of their own
    sums = x.float().view(M, -1, 128).sum(-1).t().contiguous()
    for rows, xs, pitch in ((x, None, inter), (wide, sums, inter), (x, sums, inter + 4)):
        def call():
            buf = torch.full((M + 2, pitch), 7.0, dtype=torch.bfloat16, device=DEV)
            left = torch.zeros(inter // 128, M, device=DEV)
            ops.awq_gemm_silu_mul(rows, packed, si, zi, buf[:M, :inter], xs, left)
            return buf, left

        buf, left = call()
        out = buf[:M, :inter]
        # a sum that falls on the other side of a rounding boundary moves gate or up by an ulp
        torch.testing.assert_close(out.double(), want, rtol=4 * 2 ** -8, atol=2 ** -8 * want.abs().mean().item())
        assert (out.double() - want).norm() / want.norm() < 2 ** -8
        torch.testing.assert_close(left, out.float().view(M, -1, 128).sum(-1).t(), rtol=1e-4, atol=2e-2)
        assert bool((buf[M:] == 7).all()) and bool((buf[:, inter:] == 7).all())
        if xs is not None:
            for mine, theirs in zip((buf, left), _wide(monkeypatch, call)):
                assert torch.equal(mine, theirs)


@pytest.mark.parametrize("M,K,N,rows,splits", [(65, 4096, 28672, 96, 1), (96, 1024, 16640, 96, 1), (97, 1536, 16640, 128, 1),
                                               (128, 2560, 16640, 128, 1), (193, 1024, 8448, 128, 1), (160, 4608, 5632, 96, 2),
                                               (192, 28672, 8192, 96, 2), (97, 10240, 11008, 128, 2), (255, 10240, 5632, 128, 2),
                                               (65, 4608, 8448, 96, 3), (97, 4608, 8448, 128, 3), (193, 4608, 4352, 128, 3),
                                               (192, 12800, 3840, 96, 4), (80, 12800, 5632, 96, 5), (255, 12800, 2816, 128, 5),
                                               (65, 25088, 4352, 96, 7), (97, 25088, 4352, 128, 7)])
def test_finished_rows(monkeypatch, M, K, N, rows, splits):
    """Finished rows with a bias, whole and split along K, twice over one workspace of the size that is asked for, no further from 64
    bits than the wide kernel's: what is left after the rounding to bf16 is that rounding."""
    from sglang_security_amd import ops

    _takes(M, N, K, rows, splits)
    x, qw, sc, qz = (t.to(DEV) for t in _case(M, K, N, K + N))
    bias = torch.randn(N, device=DEV).to(torch.bfloat16)
    packed = ops.awq_repack(qw)
    want = x.double() @ _weight64(qw, sc, qz)
    size = ops.awq_gemm_workspace_bytes(M, N, K)
    work = torch.zeros(size + 4096, dtype=torch.uint8, device=DEV)
    work[size:] = 7
    sums = x.float().view(M, -1, 128).sum(-1).t().contiguous()
    err = lambda t, w: ((t.double() - w).norm() / w.norm()).item()
    finished = lambda: ops.awq_gemm(x, packed, sc, qz, bias, None, work)

    def with_sums():
        buf = torch.full((M + 2, N + 8), 7.0, dtype=torch.bfloat16, device=DEV)
        ops.awq_gemm_xs(x, packed, sc, qz, sums, buf[:M, :N], work)
        assert bool((buf[M:] == 7).all()) and bool((buf[:, N:] == 7).all())
        return buf[:M, :N]

    for call, exact in ((finished, want + bias.double()), (with_sums, want)):
        got, again = call(), call()
        assert torch.equal(got, again)
        assert bool((work[size:] == 7).all()) and not bool(work[: 4 * 4096].any())   # tickets are left at zero
        assert err(got, exact) <= 1.01 * err(_wide(monkeypatch, call), exact)


@pytest.mark.parametrize("M,K,rows", [(96, 512, 96), (100, 512, 128), (96, 1024, 96), (80, 1536, 96), (128, 1536, 128), (100, 2560, 128)])
def test_zero_scales_and_few_stages(monkeypatch, M, K, rows):
    """Columns whose scale is zero in the first, a middle, the last or all groups, over one to three and five stages: nothing from there,
    the rest as before; a capture replays the same bits."""
    from sglang_security_amd import ops

    inter = 8320
    _takes(M, 2 * inter, K, rows, gated=True)
    x, qw, sc, qz = (t.to(DEV) for t in _case(M, K, 2 * inter, K))
    sc[0, 0::7] = 0
    sc[K // 256, 1::7] = 0
    sc[-1, 2::7] = 0
    sc[:, 3::7] = 0
    qi, si, zi = ops.awq_interleave_gate_up(qw, sc, qz)
    packed = ops.awq_repack(qi)
    gu = (x.double() @ _weight64(qw, sc, qz)).to(torch.bfloat16).double()
    want = torch.nn.functional.silu(gu[:, :inter]).to(torch.bfloat16).double() * gu[:, inter:]
    sums = x.float().view(M, -1, 128).sum(-1).t().contiguous()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for xs in (None, sums):
            out = torch.empty(M, inter, dtype=torch.bfloat16, device=DEV)
            ops.awq_gemm_silu_mul(x, packed, si, zi, out, xs)
            eager = out.clone()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                ops.awq_gemm_silu_mul(x, packed, si, zi, out, xs)
            for _ in range(2):
                out.zero_()
                graph.replay()
                stream.synchronize()
                assert torch.equal(out, eager)
            assert (eager.double() - want).norm() / want.norm() < 2 ** -8
            assert bool((eager[:, 3::7] == 0).all())
            if xs is not None:
                assert torch.equal(eager, _wide(monkeypatch, lambda: ops.awq_gemm_silu_mul(x, packed, si, zi, out, xs).clone()))
