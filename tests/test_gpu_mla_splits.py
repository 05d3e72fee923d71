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
