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


@pytest.mark.parametrize("M", [65, 96, 97, 128, 192, 200, 255])
@pytest.mark.parametrize("K,inter", [(4096, 14336), (1536, 14336)])
def test_gated_rows_and_their_sums(monkeypatch, M, K, inter):
    """Every output of the gated form, ragged rows among them, with and without the producer's block sums: the unfused sequence's
    roundings, so half an ulp of bf16 twice (2^-8 each) beside the product's own 1e-6; rows behind M stay as they were.  With the
    producer's sums, rows and the sums left for the next product are the wide kernel's bits."""
    from sglang_security_amd import ops

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


@pytest.mark.parametrize("M,K,N", [(65, 4096, 28672), (128, 2048, 28672), (300, 1024, 16384), (96, 1536, 12288)])
def test_finished_rows(monkeypatch, M, K, N):
    """Finished rows with a bias, twice over one workspace, no further from 64 bits than the wide kernel's: what is left after the
    rounding to bf16 is that rounding."""
    from sglang_security_amd import ops

    x, qw, sc, qz = (t.to(DEV) for t in _case(M, K, N, K + N))
    bias = torch.randn(N, device=DEV).to(torch.bfloat16)
    packed = ops.awq_repack(qw)
    want = x.double() @ _weight64(qw, sc, qz) + bias.double()
    work = torch.zeros(max(ops.awq_gemm_workspace_bytes(M, N, K), 256), dtype=torch.uint8, device=DEV)
    call = lambda: ops.awq_gemm(x, packed, sc, qz, bias, None, work)
    got, again = call(), call()
    assert torch.equal(got, again)
    err = lambda t: ((t.double() - want).norm() / want.norm()).item()
    assert err(got) <= 1.01 * err(_wide(monkeypatch, call))


def test_zero_scales_and_few_stages(monkeypatch):
    """Columns whose scale is zero in the first, a middle, the last or all groups, over one to three stages: nothing from there, the
    rest as before; a capture replays the same bits."""
    from sglang_security_amd import ops

    for K in (512, 1024, 1536):
        M, inter = 128, 14336
        x, qw, sc, qz = (t.to(DEV) for t in _case(M, K, 2 * inter, K))
        sc[0, 0::7] = 0
        sc[K // 256, 1::7] = 0
        sc[-1, 2::7] = 0
        sc[:, 3::7] = 0
        qi, si, zi = ops.awq_interleave_gate_up(qw, sc, qz)
        packed = ops.awq_repack(qi)
        gu = (x.double() @ _weight64(qw, sc, qz)).to(torch.bfloat16).double()
        want = torch.nn.functional.silu(gu[:, :inter]).to(torch.bfloat16).double() * gu[:, inter:]
        out = torch.empty(M, inter, dtype=torch.bfloat16, device=DEV)
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            ops.awq_gemm_silu_mul(x, packed, si, zi, out)
            eager = out.clone()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                ops.awq_gemm_silu_mul(x, packed, si, zi, out)
            for _ in range(2):
                out.zero_()
                graph.replay()
                stream.synchronize()
                assert torch.equal(out, eager)
        assert (eager.double() - want).norm() / want.norm() < 2 ** -8
        assert bool((eager[:, 3::7] == 0).all())
