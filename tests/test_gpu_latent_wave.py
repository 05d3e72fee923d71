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
    # the result is rounded once to the type, and its probabilities are held closer than that (relative eps, against |v| <= max|v|)
    eps = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    assert (o.double() - want).abs().max().item() <= eps * (kv.abs().max().double() + want.abs().max()).item() + 1e-4
    # the splits' log-sum-exps, over sums of rounded probabilities
    got = torch.logsumexp(torch.where(lse.isnan(), torch.full_like(lse, -math.inf), lse), -1)
    assert (got.double() - wlse).abs().max().item() <= eps + 1e-4


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens,Hq,most", [
    ([400, 129] + [65] * 31, 256, 1),
    ([400, 129] + [65] * 31, 256, 4),                       # splits folded into one block
    ([1000, 400, 129] + [65] * 6, 32, 32),                  # ... and into several: a split's maximum lies above those before it
])
def test_scores_that_outgrow_the_first_maximum(lens, Hq, most, dtype):
    """Rows that grow along the request: every tile's scores lie far above those before it, in both directions."""
    kv, q = _data(lens, Hq, dtype, 3)
    ind = torch.randperm(sum(lens) + 5, generator=torch.Generator().manual_seed(sum(lens)))[: sum(lens)].to(DEV)
    grow = torch.cat([torch.linspace(0.1, 6.0, n, device=DEV) for n in lens])
    kv[ind, 0] = (kv[ind, 0].float() * grow[:, None]).to(dtype)
    kv[ind, 0, :8] = (grow[:, None] * 12.0).to(dtype)
    q[:, ::2, :8] = 2.0
    q[:, 1::2, :8] = -2.0
    o, lse, want, wlse = _run(lens, Hq, most, dtype, kv, q)
    eps = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    assert (o.double() - want).abs().max().item() <= eps * (kv[..., :512].abs().max().double() + want.abs().max()).item() + 1e-4
    # every split's log-sum-exp: 32-bit sums of scores of up to 100 (576 products each: 2^-24 times their size, times a few)
    got = torch.logsumexp(torch.where(lse.isnan(), torch.full_like(lse, -math.inf), lse).double(), -1)
    assert (got - wlse).abs().max().item() <= 2e-3


@pytest.mark.parametrize("lens", [[1152, 800, 960] * 22, [100, 64, 30] * 22])
def test_probabilities_are_carried_in_two_parts(lens):
    """What is left of the error is the rounding of the result, half a unit of its last place (eight bits, so 2^-9 of the power of two
    above it), and 2^-15 of what is summed up for 32-bit sums, exponentials and scores.  Probabilities in one 16-bit number,
    each off by up to 2^-8, leave that bound behind: with them the bound is tried as well."""
    kv, q = _data(lens, 128, torch.bfloat16, 9)
    o, _, want, _ = _run(lens, 128, 8, torch.bfloat16, kv, q)
    gen = torch.Generator().manual_seed(sum(lens))
    ind = torch.randperm(sum(lens) + 5, generator=gen)[: sum(lens)].to(DEV)
    at = 0
    for b, n in enumerate(lens[:6]):
        k = kv[ind[at: at + n], 0].double()
        p = torch.softmax(q[b].double() @ k.T / math.sqrt(192), -1)
        bound = torch.ldexp(torch.ones_like(want[b]), torch.frexp(want[b]).exponent - 9) + 2.0**-15 * (p @ k[:, :512].abs())
        assert ((o[b].double() - want[b]).abs() <= bound).all(), b
        p = p / p.amax(-1, keepdim=True)
        one = (p.to(torch.bfloat16).double() @ k[:, :512]) / p.sum(-1, keepdim=True)
        assert ((one.to(torch.bfloat16).double() - want[b]).abs() > bound).double().mean().item() > 0.05, b
        at += n


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_two_latent_heads_strided_queries_and_odd_rows(dtype):
    """A pool of two latent heads a slot, queries and results that are parts of wider rows; results at odd elements."""
    from sglang_security_amd import ops

    lens, Hq, most = [70, 300, 16, 129] * 10, 80, 4                    # 40 heads a latent head: a tile and a quarter of one
    B, total = len(lens), sum(lens)
    gen = torch.Generator().manual_seed(17)
    kv = torch.randn(total + 3, 2, 592, generator=gen).to(dtype).to(DEV)[..., :576]
    q = (torch.randn(B, Hq + 3, 584, generator=gen) * 0.5).to(dtype).to(DEV)[:, 1: Hq + 1, :576]
    ind = torch.randperm(total + 3, generator=gen)[:total].to(torch.int32).to(DEV)
    ptr = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    ns = torch.full((B,), most, dtype=torch.int32, device=DEV)
    rows = torch.full((B, Hq, 515), -77.0, dtype=dtype, device=DEV)
    o = rows[..., 1: 513]
    al, lse = torch.empty(B, Hq, most, 512, device=DEV), torch.empty(B, Hq, most, device=DEV)
    ops.decode_attention_fwd(q, kv, kv[..., :512], o, ptr, ind, al, lse, ns, most, 1 / math.sqrt(192), 0.0)
    assert (rows[..., 0] == -77).all() and (rows[..., 513:] == -77).all()
    eps = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    for b in range(B):
        for h in range(2):
            k = kv[ind[ptr[b]: ptr[b + 1]].long(), h].double()
            want = torch.softmax(q[b, 40 * h: 40 * h + 40].double() @ k.T / math.sqrt(192), -1) @ k[:, :512]
            assert (o[b, 40 * h: 40 * h + 40].double() - want).abs().max().item() <= eps * (k.abs().max() + want.abs().max()).item() + 1e-4, (b, h)


def test_more_than_64_blocks_a_request():
    """The merge of 150 blocks: its lanes take more than one block each."""
    lens = [9600, 50]
    kv, q = _data(lens, 32, torch.bfloat16, 13)
    o, lse, want, wlse = _run(lens, 32, 300, torch.bfloat16, kv, q)
    assert (~lse[0].isnan()).sum(-1).eq(300).all()
    assert (o.double() - want).abs().max().item() <= 2.0**-8 * (kv.abs().max().double() + want.abs().max()).item() + 1e-4
    got = torch.logsumexp(torch.where(lse.isnan(), torch.full_like(lse, -math.inf), lse), -1)
    assert (got.double() - wlse).abs().max().item() <= 2.0**-8 + 1e-4


@pytest.mark.parametrize("shared", [True, False])
def test_beside_a_shared_plan(shared):
    """Launched beside the kernel for shared prefixes, by whose plan the one or the other leaves: one result, that of float64."""
    from sglang_security_amd import ops

    Hq, most, sizes = 128, 8, [(6, 130), (4, 64), (3, 0)] if shared else [(1, 0)] * 13
    gen = torch.Generator().manual_seed(19)
    B = sum(n for n, _ in sizes)
    rows, at, prefixes = [], 1, []
    for n, prefix in sizes:
        common = torch.arange(at, at + prefix)
        at += prefix
        prefixes.append(prefix)
        for _ in range(n):
            own = int(torch.randint(1, 200, (1,), generator=gen))
            rows.append(torch.cat([common, torch.arange(at, at + own)]))
            at += own
    kv = torch.randn(at, 1, 576, generator=gen).to(torch.bfloat16).to(DEV)
    q = (torch.randn(B, Hq, 576, generator=gen) * 0.5).to(torch.bfloat16).to(DEV)
    ind = torch.cat(rows).int().to(DEV)
    ptr = torch.tensor([0] + torch.tensor([len(r) for r in rows]).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    gi = torch.tensor([0] + torch.tensor([n for n, _ in sizes]).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    plan = ops.decode_shared_plan_buffer(B, Hq, 1, most, DEV)
    ops.decode_shared_plan_from_groups(ptr, ind, gi, torch.tensor(prefixes, dtype=torch.int32, device=DEV), B, Hq, 1, most, plan)
    assert (ops.decode_shared_plan_read(plan, B)["n_items"] > 0) == shared
    ws = ops.decode_shared_workspace(B, Hq, 512, most, DEV)
    ns = torch.full((B,), most, dtype=torch.int32, device=DEV)
    o = torch.full((B, Hq, 512), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.decode_attention_shared_planned(q, kv, kv[..., :512], o, ptr, ind, plan, ws, most, 1 / math.sqrt(192), 0.0, None, ns)
    assert ops.decode_shared_workspace_status(ws, B, Hq) == 0
    for b, r in enumerate(rows):
        k = kv[r.to(DEV), 0].double()
        want = torch.softmax(q[b].double() @ k.T / math.sqrt(192), -1) @ k[:, :512]
        assert (o[b].double() - want).abs().max().item() <= 2.0**-8 * (k.abs().max() + want.abs().max()).item() + 1e-4, b


def test_more_splits_asked_for_than_there_is_room_for():
    """A split count above the slots of the partials leaves out the tokens behind them, and nothing is written behind the last."""
    from sglang_security_amd import ops

    B, Hq, most = 34, 128, 2
    lens = [256] * B
    kv, q = _data(lens, Hq, torch.bfloat16, 5)
    gen = torch.Generator().manual_seed(sum(lens))
    ind = torch.randperm(sum(lens) + 5, generator=gen)[: sum(lens)].to(torch.int32).to(DEV)
    ptr = (torch.arange(B + 1, device=DEV) * 256).int()
    ns = torch.full((B,), 8, dtype=torch.int32, device=DEV)
    whole = [torch.full((n + 4096,), -77.0, dtype=t, device=DEV) for n, t in
             ((B * Hq * 512, torch.bfloat16), (B * Hq * most * 512, torch.float32), (B * Hq * most, torch.float32))]
    o, al, lse = whole[0][:-4096].view(B, Hq, 512), whole[1][:-4096].view(B, Hq, most, 512), whole[2][:-4096].view(B, Hq, most)
    ops.decode_attention_fwd(q, kv, kv[..., :512], o, ptr, ind, al, lse, ns, most, 1 / math.sqrt(192), 0.0)
    assert all((w[-4096:] == -77).all() for w in whole)
    k = kv[ind.view(B, 256)[:, :64].long(), 0].double()                 # two splits of 32 tokens
    s = torch.matmul(q.double(), k.transpose(1, 2).contiguous()) / math.sqrt(192)
    want = torch.matmul(torch.softmax(s, -1), k[..., :512].contiguous())
    assert (o.double() - want).abs().max().item() <= 2.0**-8 * (kv.abs().max().double() + want.abs().max()).item() + 1e-4
    assert (lse.double() - torch.logsumexp(s.view(B, Hq, 2, 32), -1)).abs().max().item() <= 2.0**-8 + 1e-4


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
