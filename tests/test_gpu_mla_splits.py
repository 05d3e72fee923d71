"""Latent-row decode where the launch takes fewer splits than the caller offers: batches whose splits spill into a short
last round, one request much longer than the rest, empty requests, and more requests than the chip has places."""
import math

import pytest
import torch

import sglang_security_amd  # noqa: F401

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hq,max_splits", [(16, 128, 8), (20, 128, 8), (65, 64, 5), (33, 128, 16), (130, 128, 3), (24, 40, 16)])
def test_splits_against_float32(dtype, B, Hq, max_splits):
    from sglang_security_amd import ops

    gen = torch.Generator().manual_seed(B * 100 + Hq)
    lens = torch.randint(90, 161, (B,), generator=gen)
    lens[1], lens[2], lens[B - 1] = 700, 1, 0
    total = int(lens.sum())
    kv = torch.randn(total + 5, 1, 576, generator=gen).to(dtype).to(DEV)
    q = (torch.randn(B, Hq, 576, generator=gen) * 0.5).to(dtype).to(DEV)
    ind = torch.randperm(total + 5, generator=gen)[:total].to(torch.int32).to(DEV)
    ptr = torch.tensor([0] + lens.cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    ns = torch.full((B,), max_splits, dtype=torch.int32, device=DEV)
    ns[0] = 1
    sm = 1.0 / math.sqrt(192)

    o = torch.full((B, Hq, 512), float("nan"), dtype=dtype, device=DEV)
    al = torch.full((B, Hq, max_splits, 512), float("nan"), device=DEV)
    lse = torch.full((B, Hq, max_splits), float("nan"), device=DEV)
    ops.decode_attention_fwd(q, kv, kv[..., :512], o, ptr, ind, al, lse, ns, max_splits, sm, 0.0)
    fast = o.float().cpu()
    rows = [b for b in range(B) if lens[b]]
    kc, qc, ic, pc = kv[:, 0].float().cpu(), q.float().cpu(), ind.cpu().long(), ptr.cpu()
    # each probability is rounded once to the type (relative eps, against |v| <= max|v|), and the result once
    eps = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    for b in rows:
        k = kc[ic[pc[b]:pc[b + 1]]]
        want = torch.softmax(qc[b] @ k.T * sm, -1) @ k[:, :512]
        assert (fast[b] - want).abs().max().item() <= eps * (k.abs().max().item() + want.abs().max().item()) + 1e-4, b


@pytest.mark.parametrize("lens,Hq,most,taken", [
    ([960] * 64, 128, 3, 2),                        # three splits: a round of 512 blocks and half of one
    ([960] * 20 + [1], 128, 8, 6),                  # 480 blocks instead of 640
    ([960] * 16, 128, 8, 8),                        # a whole round as it is
    ([150] * 75, 128, 8, 1),                        # little to read: partials are what the splits cost
    ([960] * 63 + [3000], 128, 3, 2),               # (the last keeps its three)
    ([960] * 64, 16, 8, 8),                         # up to 31 heads a group: as the caller says
    ([960] * 64, 128, 17, 17),                      # more than the rule weighs
    ([0] * 63 + [1], 128, 3, 3),                    # (padding)
])
def test_splits_taken(lens, Hq, most, taken):
    """The slots of the partials that a launch fills: as many as the rule takes, a request much longer than the mean as many
    as the caller offers, and the rows are those of float32 sums."""
    from sglang_security_amd import ops

    gen = torch.Generator().manual_seed(len(lens))
    B, total = len(lens), sum(lens)
    kv = torch.randn(total + 5, 1, 576, generator=gen).to(torch.bfloat16).to(DEV)
    q = (torch.randn(B, Hq, 576, generator=gen) * 0.5).to(torch.bfloat16).to(DEV)
    ind = torch.randperm(total + 5, generator=gen)[:total].to(torch.int32).to(DEV)
    ptr = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    ns = torch.full((B,), most, dtype=torch.int32, device=DEV)
    o = torch.full((B, Hq, 512), float("nan"), dtype=torch.bfloat16, device=DEV)
    al = torch.full((B, Hq, most, 512), float("nan"), device=DEV)
    lse = torch.full((B, Hq, most), float("nan"), device=DEV)
    ops.decode_attention_fwd(q, kv, kv[..., :512], o, ptr, ind, al, lse, ns, most, 1.0 / math.sqrt(192), 0.0)
    filled = (~lse.isnan()).sum(-1)
    for b in range(B):
        per = -(-(-(-lens[b] // (most if lens[b] > 2 * total / B else max(taken, 1)))) // 32) * 32
        assert (filled[b] == (-(-lens[b] // per) if lens[b] else 0)).all(), b
    for b in (0, B - 1):
        if lens[b]:
            k = kv[ind[ptr[b]: ptr[b + 1]].long(), 0].float()
            want = torch.softmax(q[b].float() @ k.T / math.sqrt(192), -1) @ k[:, :512]
            assert (o[b].float() - want).abs().max().item() <= 2.0**-8 * (k.abs().max() + want.abs().max()).item() + 1e-4
