"""Latent-row decode of 32 query heads or more: a block's waves take every fourth tile of 16 tokens and may fold several splits;
sizes around a tile, a wave's turn and a split, scores that outgrow the maximum they were first measured from, and head groups
that leave part of a block's 32 heads empty."""
import math

import pytest
import torch

import sglang_security_amd  # noqa: F401

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _run(lens, Hq, most, dtype, kv, q, cap=0.0, splits=None, sm=1.0 / math.sqrt(192)):
    from sglang_security_amd import ops

    B, total = len(lens), sum(lens)
    gen = torch.Generator().manual_seed(total)
    ind = torch.randperm(total + 5, generator=gen)[:total].to(torch.int32).to(DEV)
    ptr = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    ns = torch.full((B,), splits or most, dtype=torch.int32, device=DEV)
    o = torch.full((B, Hq, 512), float("nan"), dtype=dtype, device=DEV)
    al = torch.full((B, Hq, most, 512), float("nan"), device=DEV)
    lse = torch.full((B, Hq, most), float("nan"), device=DEV)
    ops.decode_attention_fwd(q, kv, kv[..., :512], o, ptr, ind, al, lse, ns, most, sm, cap)
    want, wlse = [], []
    for b in range(B):
        k = kv[ind[ptr[b]: ptr[b + 1]].long(), 0].double()
        s = q[b].double() @ k.T * sm
        if cap:
            s = cap * torch.tanh(s / cap)
        want.append(torch.softmax(s, -1) @ k[:, :512])
        wlse.append(torch.logsumexp(s, -1))
    return o, lse, torch.stack(want), torch.stack(wlse)


def _data(lens, Hq, dtype, seed):
    gen = torch.Generator().manual_seed(seed)
    kv = torch.randn(sum(lens) + 5, 1, 576, generator=gen).to(dtype).to(DEV)
    return kv, (torch.randn(len(lens), Hq, 576, generator=gen) * 0.5).to(dtype).to(DEV)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Hq,lens,most,cap", [
    (32, [1, 15, 16, 17, 63, 64, 65] * 10, 4, 0.0),       # one tile, one turn of the four waves, and a token either side
    (128, [257, 300, 1152, 96, 64] * 2, 8, 0.0),             # splits folded, several blocks a request
    (72, [511, 33] * 50, 3, 30.0),                        # the last tile of heads holds eight; capped
    (64, [960] * 70, 5, 0.0),                        # rows written without a merge
])
def test_sizes(Hq, lens, most, cap, dtype):
    kv, q = _data(lens, Hq, dtype, len(lens) * 1000 + Hq)
    o, lse, want, wlse = _run(lens, Hq, most, dtype, kv, q, cap)
    # a probability is rounded once to the type, and so is the result (relative eps, against |v| <= max|v|)
    eps = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    assert (o.double() - want).abs().max().item() <= eps * (kv.abs().max().double() + want.abs().max()).item() + 1e-4
    # the splits' log-sum-exps, over sums of rounded probabilities
    got = torch.logsumexp(torch.where(lse.isnan(), torch.full_like(lse, -math.inf), lse), -1)
    assert (got.double() - wlse).abs().max().item() <= eps + 1e-4


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_scores_that_outgrow_the_first_maximum(dtype):
    """Rows that grow along the request: every tile's scores lie far above those before it, in both directions."""
    lens = [400, 129] + [65] * 31
    kv, q = _data(lens, 256, dtype, 3)
    ind = torch.randperm(sum(lens) + 5, generator=torch.Generator().manual_seed(sum(lens)))[: sum(lens)].to(DEV)
    grow = torch.cat([torch.linspace(0.1, 6.0, n, device=DEV) for n in lens])
    kv[ind, 0] = (kv[ind, 0].float() * grow[:, None]).to(dtype)
    kv[ind, 0, :8] = (grow[:, None] * 12.0).to(dtype)
    q[:, ::2, :8] = 2.0
    q[:, 1::2, :8] = -2.0
    o, _, want, _ = _run(lens, 256, 1, dtype, kv, q)
    eps = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    assert (o.double() - want).abs().max().item() <= eps * (kv[..., :512].abs().max().double() + want.abs().max()).item() + 1e-4


def test_more_splits_asked_for_than_there_is_room_for():
    """A split count above the slots of the partials leaves out the tokens behind them and writes no others' slots."""
    lens = [256] * 34
    kv, q = _data(lens, 128, torch.bfloat16, 5)
    o, lse, _, _ = _run(lens, 128, 2, torch.bfloat16, kv, q, splits=8)
    assert o.isfinite().all() and lse.isfinite().all()


def test_scores_of_minus_infinity():
    """A run of tokens whose key (beside the value part) makes their score -inf weighs nothing, wherever a wave meets it."""
    lens = [96, 16 + 64] + [40] * 31
    kv, q = _data(lens, 256, torch.bfloat16, 7)
    ind = torch.randperm(sum(lens) + 5, generator=torch.Generator().manual_seed(sum(lens)))[: sum(lens)].to(DEV)
    hidden = torch.zeros(sum(lens), dtype=torch.bool, device=DEV)
    hidden[0:16] = hidden[64:80] = hidden[96 + 16: 96 + 80] = True      # first tiles of waves, and of one request all but a tile
    kv[ind[hidden], 0, 575] = math.inf
    q[..., 575] = -1.0
    o, _, want, _ = _run(lens, 256, 1, torch.bfloat16, kv, q)
    assert o.isfinite().all()
    v = kv[..., :512].abs().max().double()
    assert (o.double() - want).abs().max().item() <= 2.0**-8 * (v + want.abs().max()).item() + 1e-4


@pytest.mark.parametrize("splits", [32, 8])
def test_blocks_of_minus_infinity(splits):
    """Requests of several blocks (of two folded splits, and of one), some of which hold nothing but scores of -inf: the others'
    rows are the result; with none left it is NaN, as a softmax over nothing."""
    lens = [512, 512, 300] + [20] * 6
    kv, q = _data(lens, 32, torch.bfloat16, 11)
    ind = torch.randperm(sum(lens) + 5, generator=torch.Generator().manual_seed(sum(lens)))[: sum(lens)].to(DEV)
    hidden = torch.zeros(sum(lens), dtype=torch.bool, device=DEV)
    hidden[64:192] = hidden[448:512] = True             # of the first request: the second, third and last 64 tokens
    hidden[512: 1024] = True                            # the whole second one
    kv[ind[hidden], 0, 575] = math.inf
    q[..., 575] = -1.0
    o, lse, want, wlse = _run(lens, 32, 32, torch.bfloat16, kv, q, splits=splits)
    assert o[1].isnan().all()
    keep = [b for b in range(len(lens)) if b != 1]
    assert o[keep].isfinite().all()
    v = kv[..., :512].abs().max().double()
    assert (o[keep].double() - want[keep]).abs().max().item() <= 2.0**-8 * (v + want[keep].abs().max()).item() + 1e-4
    got = torch.logsumexp(torch.where(lse.isnan(), torch.full_like(lse, -math.inf), lse), -1)
    assert (got[keep].double() - wlse[keep]).abs().max().item() <= 2.0**-8 + 1e-4


@pytest.mark.parametrize("Hq,lens,most", [
    (128, [300] * 3 + [40] * 8 + [700, 1] + [33] * 6, 8),      # more than the blocks every request has a place for, and fewer
    (128, [1500] + [10] * 69, 8),                              # one long request among more than a wave's lanes
    (64, [20] * 66 + [2000, 900, 0, 1200], 5),                 # ... behind them, and one without tokens
    (32, [700, 30] * 8, 64),                                   # splits that have to be folded eight at a time
    (72, [64, 128, 129, 640] * 6, 16),                         # 85 places of three head tiles
])
def test_blocks_are_found(Hq, lens, most):
    """Requests with more and fewer blocks than they have a place for by their number: every row, and every log-sum-exp."""
    kv, q = _data(lens, Hq, torch.bfloat16, len(lens) + Hq)
    o, lse, want, wlse = _run(lens, Hq, most, torch.bfloat16, kv, q)
    keep = [b for b, n in enumerate(lens) if n]
    assert all(o[b].isnan().all() for b, n in enumerate(lens) if n == 0)
    assert (o[keep].double() - want[keep]).abs().max().item() <= 2.0**-8 * (kv.abs().max().double() + want[keep].abs().max()).item() + 1e-4
    got = torch.logsumexp(torch.where(lse.isnan(), torch.full_like(lse, -math.inf), lse), -1)
    assert (got[keep].double() - wlse[keep]).abs().max().item() <= 2.0**-8 + 1e-4
