"""GPU: every mechanism of the Lusatar layers alone and the whole model through the engine, against the plain oracle
(oracle/lusatar.py, float64)."""
import functools
import json
import math
import subprocess
import sys

import pytest
import torch

import lusatar_models as M
from oracle import lusatar as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF16, F32 = torch.bfloat16, torch.float32
TOL = {BF16: 1e-2, F32: 2e-6}


def gen(seed):
    return torch.Generator().manual_seed(seed)


def rnd(g, *shape, dtype=F32):
    return torch.randn(*shape, generator=g).to(dtype)


def i32(*v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


def close(got, want, tol, what=""):
    want = want.double()
    err = (got.double().cpu() - want).abs().max().item()
    assert err <= tol * max(want.abs().max().item(), 1e-3), f"{what}: {err} of {want.abs().max().item()}"


def source(t, splits, dtype):
    """A product [rows, cols] as its consumers may receive it: split sums, or finished rows."""
    from sglang_security_amd.ops_hybrid import Source

    if splits == 0:
        return Source(t.to(dtype).to(DEV), False), t.to(dtype).double()
    parts = torch.stack([t * (0.5 if splits > 1 else 1.0)] + [t * (0.5 / (splits - 1))] * (splits - 1)) if splits > 1 else t[None]
    return Source(parts.contiguous().to(DEV), True), parts.double().sum(0)


# ---- row kernels --------------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("width,pitch", [(84, 128), (128, 128), (2560, 2560), (4100, 4224), (9000, 9088)])
@pytest.mark.parametrize("dtype,splits", [(BF16, 0), (BF16, 3), (BF16, 9), (F32, 1)])
def test_residual_norm(width, pitch, dtype, splits):
    from sglang_security_amd import ops_hybrid as H

    g, rows, eps = gen(width + splits), 5, 1e-4
    wide = lambda t: torch.cat([t, t.new_zeros(*t.shape[:-1], pitch - width)], -1).contiguous()
    x, x0, s = (wide(rnd(g, rows, width)) for _ in range(3))
    wp, wn, step = (wide(rnd(g, width)) for _ in range(3))
    src, sv = source(s, splits, dtype)
    d = lambda t: t.clone().to(DEV)
    h = torch.full((rows, pitch), 7.0, dtype=dtype, device=DEV)
    xd = d(x)
    H.residual_norm(xd, width, eps, h, d(wn), src, d(wp), x0=d(x0), add_x0=True, step=d(step), dtype=dtype)
    want = x.double()[:, :width] + O.rms_norm(sv[:, :width], wp.double()[:width], eps) + x0.double()[:, :width] + step.double()[:width]
    close(xd[:, :width], want, 2e-6, "x")
    close(h[:, :width], O.rms_norm(want, wn.double()[:width], eps), 2 * TOL[dtype], "h")
    assert not xd[:, width:].any() and not h[:, width:].any()
    # embedding in front, saved; then picked rows without storing
    table, ids = wide(rnd(g, 11, width, dtype=dtype)), i32(3, 10, 0, 0, 7)
    keep = torch.empty(rows, pitch, device=DEV)
    H.residual_norm(xd, width, eps, h, d(wn), embed=table.to(DEV), ids=ids, embed_scale=1.25, x0=keep, step=d(step), dtype=dtype)
    e = table.double()[ids.cpu().long()] * 1.25
    close(keep, e, 1e-6, "embedding output")
    close(xd, e + step.double(), 1e-6, "embedded")
    before = xd.clone()
    H.residual_norm(xd, width, eps, h, d(wn), src, d(wp), rows=i32(4, 1), dtype=dtype)
    want = (before.double().cpu()[:, :width] + O.rms_norm(sv[:, :width], wp.double()[:width], eps))[[4, 1]]
    close(h[:2, :width], O.rms_norm(want, wn.double()[:width], eps), 2 * TOL[dtype], "picked rows")
    assert torch.equal(before, xd)


@pytest.mark.parametrize("pitch", [128, 2056, 4096, 4104, 8192])
@pytest.mark.parametrize("dtype", [BF16, F32])
def test_residual_norm_of_few_and_many_rows(pitch, dtype):
    """512 rows take a thread a piece, 513 take 256 threads a row: the same sums in another grouping."""
    from sglang_security_amd import ops_hybrid as H

    g, eps = gen(pitch), 1e-5
    d = lambda t: t.clone().to(DEV)
    x, s, x0, wp, wn, step = rnd(g, 513, pitch), rnd(g, 513, pitch), rnd(g, 513, pitch), rnd(g, pitch), rnd(g, pitch), rnd(g, pitch)
    for rows in (512, 513):
        src, sv = source(s[:rows], 2, dtype)
        xd, h = d(x[:rows]), torch.empty(rows, pitch, dtype=dtype, device=DEV)
        H.residual_norm(xd, pitch, eps, h, d(wn), src, d(wp), x0=d(x0[:rows]), add_x0=True, step=d(step), dtype=dtype)
        want = x[:rows].double() + O.rms_norm(sv, wp.double(), eps) + x0[:rows].double() + step.double()
        close(xd, want, 2e-6, "x")
        close(h, O.rms_norm(want, wn.double(), eps), 2 * TOL[dtype], "h")


@pytest.mark.parametrize("splits", [2, 3, 8])
def test_residual_norm_of_wide_rows_and_many_splits(splits):
    """From 257 rows on, wide rows of more than two split sums take 256 threads a row."""
    from sglang_security_amd import ops_hybrid as H

    pitch, eps = 4104, 1e-5
    g = gen(splits)
    d = lambda t: t.clone().to(DEV)
    x, s, wp, wn = rnd(g, 257, pitch), rnd(g, 257, pitch), rnd(g, pitch), rnd(g, pitch)
    for rows in (256, 257):
        src, sv = source(s[:rows], splits, BF16)
        xd, h = d(x[:rows]), torch.empty(rows, pitch, dtype=BF16, device=DEV)
        H.residual_norm(xd, pitch, eps, h, d(wn), src, d(wp), dtype=BF16)
        want = x[:rows].double() + O.rms_norm(sv, wp.double(), eps)
        close(xd, want, 2e-6, "x")
        close(h, O.rms_norm(want, wn.double(), eps), 2 * TOL[BF16], "h")


@pytest.mark.parametrize("dtype,splits", [(BF16, 0), (BF16, 5), (F32, 1)])
def test_activations_and_capped_logits(dtype, splits):
    from sglang_security_amd import ops_hybrid as H

    g = gen(splits)
    t, bias = rnd(g, 7, 48) * 3, rnd(g, 48)
    src, sv = source(t, splits, dtype)
    for act, f in ((H.ACT_NONE, lambda z: z), (H.ACT_RELU2, O.relu2), (H.ACT_GELU_TANH, O.gelu_tanh)):
        out = torch.empty(7, 48, dtype=dtype, device=DEV)
        close(H.source_act(src, out, act, bias.to(DEV)), f(sv + bias.double()), TOL[dtype], f"activation {act}")
    for cap in (None, 2.5):
        out = torch.empty(7, 43, device=DEV)
        close(H.capped_logits(src, out, cap, dtype), O.softcap(sv[:, :43], cap), 2e-6, "logits")


# ---- latent attention -----------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype,splits", [(BF16, 0), (BF16, 4), (F32, 1)])
@pytest.mark.parametrize("q_rank,R,rot_dim,rot_dims", [(72, 104, 24, 24), (28, 36, 8, 4), (1536, 512, 64, 64), (130, 70, 70, 40)])
def test_latent_prep_and_query_rotation(dtype, splits, q_rank, R, rot_dim, rot_dims):
    from sglang_security_amd import ops_hybrid as H
    from sglang_security_amd.layers.linear import pad, vector
    from sglang_security_amd.layers.rotary import rotary_table

    g, rows, eps = gen(q_rank), 6, 1e-5
    Qp, Rp, rp = pad(q_rank, 128), pad(R, 64), pad(rot_dim, 64)
    s = torch.zeros(rows, Qp + Rp + rp)
    s[:, :q_rank], s[:, Qp: Qp + R] = rnd(g, rows, q_rank), rnd(g, rows, R)
    s[:, Qp + Rp: Qp + Rp + rot_dim] = rnd(g, rows, rot_dim)
    wq, wkv = rnd(g, q_rank), rnd(g, R)
    src, sv = source(s, splits, dtype)
    pos = torch.tensor([0, 1, 63, 64, 500, 999])
    table = rotary_table(rot_dims, 1000.0, 1000, DEV, M.YARN)
    pool = torch.full((9, Rp + rp), 5.0, dtype=dtype, device=DEV)
    cq = torch.empty(rows, Qp, dtype=dtype, device=DEV)
    loc = i32(8, 1, 3, 2, 7, 5)
    H.latent_prep(src, vector(wq, Qp).to(DEV), vector(wkv, Rp).to(DEV), cq, pool, loc, table, pos.int().to(DEV), q_rank, R, Rp, rot_dim,
                  rot_dims, eps)
    close(cq[:, :q_rank], O.rms_norm(sv[:, :q_rank], wq.double(), eps), 2 * TOL[dtype], "query latent")
    row = pool[loc.long()]
    close(row[:, :R], O.rms_norm(sv[:, Qp: Qp + R], wkv.double(), eps), 2 * TOL[dtype], "latent")
    close(row[:, Rp: Rp + rot_dim], O.rotate(sv[:, Qp + Rp: Qp + Rp + rot_dim], pos, 1000.0, rot_dims, M.YARN), TOL[dtype], "rotated key")
    assert not cq[:, q_rank:].any() and not row[:, R: Rp].any() and not row[:, Rp + rot_dim:].any()
    assert bool((pool[[0, 4, 6]] == 5.0).all())
    q = rnd(g, rows, 3, rot_dim, dtype=dtype)
    qd = q.to(DEV).clone()
    H.latent_rope_q(qd, qd, table, pos.int().to(DEV), rot_dims)
    close(qd, O.rotate(q.double(), pos, 1000.0, rot_dims, M.YARN), TOL[dtype], "rotated query")


@pytest.mark.parametrize("M_,H_,N,K", [(1, 3, 20, 64), (64, 2, 512, 128), (70, 5, 128, 512), (130, 1, 36, 448)])
def test_head_products_and_merge(M_, H_, N, K):
    from sglang_security_amd import ops_hybrid as H
    from sglang_security_amd.layers.linear import pad, padded

    g, Np = gen(N), pad(N, 16)
    a, w = rnd(g, M_, H_, K + 64, dtype=BF16), rnd(g, H_, N, K, dtype=BF16) / math.sqrt(K)
    want = torch.einsum("mhk,hnk->mhn", a[..., :K].double(), w.double())
    wp = H.pack_heads(padded(w, H_, Np, K)).to(DEV)
    out = torch.zeros(M_, H_, N, dtype=BF16, device=DEV)
    close(H.head_gemm(a.to(DEV)[..., :K], wp, out, K, Np), want, 1e-2, "tiles")
    of = torch.zeros(M_, H_, N, device=DEV)
    wf = padded(w.float(), H_, Np, K).to(DEV)
    close(H.head_gemm(a.float().to(DEV)[..., :K], wf, of, K, Np), want, 1e-5, "rows")
    # merged split partials, one split empty
    S = 4
    part, lse = rnd(g, M_, H_, S, K), rnd(g, M_, H_, S)
    lse[:, :, 2] = -math.inf
    part[:, :, 2] = math.nan
    wt = torch.softmax(lse.double(), -1)
    merged = (wt[..., None] * torch.nan_to_num(part.double())).sum(2)
    for dt in (BF16, F32):
        got = torch.empty(M_, H_, K, dtype=dt, device=DEV)
        close(H.latent_merge(part.to(DEV), lse.to(DEV), got), merged, TOL[dt], "merged")


def _pool_case(g, lengths, Rp, rotp, R, rot, dtype, loud=()):
    """Requests of the given lengths with scattered slots.  loud: (request, position) whose key is made to stand out."""
    total = sum(lengths)
    slots = torch.randperm(total + 7, generator=g)[:total] + 1
    r2t = torch.zeros(len(lengths) + 1, max(lengths) + 3, dtype=torch.int32)
    pool = torch.zeros(total + 9, Rp + rotp)
    at = 0
    for b, n in enumerate(lengths):
        r2t[b + 1, :n] = slots[at: at + n].int()          # request row b + 1: row 0 is nobody's
        pool[slots[at: at + n].long(), :R] = 0.3 * rnd(g, n, R)
        pool[slots[at: at + n].long(), Rp: Rp + rot] = 0.3 * rnd(g, n, rot)
        at += n
    for b, p in loud:
        pool[int(r2t[b + 1, p])] *= 6.0
    return r2t, pool.to(dtype)


@pytest.mark.parametrize("H_,R,rot", [(6, 104, 24), (16, 512, 64), (40, 512, 64), (3, 36, 8), (33, 200, 64), (1, 320, 64)])
@pytest.mark.parametrize("window", [1, 21, 64, 90, None])
def test_latent_decode(H_, R, rot, window):
    """Rows at, just inside and just outside the window's edge; one key stands out just inside or just outside."""
    from sglang_security_amd import ops_hybrid as H
    from sglang_security_amd.layers.linear import pad

    g = gen(R + (window or 0))
    Rp, rotp, scale = pad(R, 64), 64, 0.9 / math.sqrt(R)
    w = window or 40
    lengths = [1, w, w + 1, w + 2, 2 * w + 33, 130, 65]
    loud = [(b, n - 1 - d) for b, n, d in ((1, w, w - 1), (2, w + 1, w), (3, w + 2, w - 1), (4, 2 * w + 33, w), (5, 130, 0)) if 0 <= n - 1 - d]
    r2t, pool = _pool_case(g, lengths, Rp, rotp, R, rot, BF16, loud)
    q = torch.zeros(len(lengths), H_, Rp + rotp, dtype=BF16)
    q[..., :R], q[..., Rp: Rp + rot] = rnd(g, len(lengths), H_, R), rnd(g, len(lengths), H_, rot)
    for b, p in loud:                                       # every query points at its request's loud key
        q[b] += 1.5 * pool[int(r2t[b + 1, p])]
    want = torch.zeros(len(lengths), H_, Rp).double()
    for b, n in enumerate(lengths):
        k = pool[r2t[b + 1, :n].long()].double()
        o = O.window_attention(q[b].double()[None].expand(n, -1, -1), k[:, None].expand(n, H_, -1), k[:, None, :Rp].expand(n, H_, -1),
                               scale, window)
        want[b] = o[-1]
    req, pos = i32(*range(1, len(lengths) + 1)), i32(*[n - 1 for n in lengths])
    args = (q.to(DEV), pool.to(DEV), r2t.to(DEV), req, pos)
    for S in (1, 3, 8):
        part = torch.full((len(lengths), H_, S, Rp), math.nan, device=DEV)
        lse = torch.full((len(lengths), H_, S), math.nan, device=DEV)
        H.latent_decode(*args, part, lse, Rp, window, scale)
        out = torch.empty(len(lengths), H_, Rp, dtype=BF16, device=DEV)
        H.latent_merge(part, lse, out)
        close(out, want, 1e-2, f"{S} splits")
    for dt, tol in ((BF16, 1e-2), (F32, 1e-5)):
        out = torch.empty(len(lengths), H_, Rp, dtype=dt, device=DEV)
        H.latent_attention_rows(args[0].to(dt), args[1].to(dt), *args[2:], out, window, scale)
        close(out, want, tol, f"rows {dt}")


@pytest.mark.parametrize("H_,kp,vp,vdim", [(6, 64, 64, 64), (3, 128, 128, 128), (2, 64, 128, 70), (5, 192, 64, 20), (2, 256, 256, 250),
                                           (1, 128, 256, 201), (2, 192, 256, 256), (2, 256, 64, 64), (2, 64, 256, 129)])
@pytest.mark.parametrize("window", [1, 21, 64, 90, None])
def test_latent_prefill(H_, kp, vp, vdim, window):
    """Portions of unequal length behind prefixes of unequal length; loud keys inside and outside the windows."""
    from sglang_security_amd import ops_hybrid as H

    g = gen(kp + vp + (window or 0))
    scale = 0.8 / math.sqrt(kp + 64)
    seqs = [(0, 2), (0, 131), (70, 64), (33, 65), (1, 17), (200, 3)]        # (tokens before the portion, rows)
    lo = [max(0, s - window + 1) if window else 0 for s, _ in seqs]
    ahead = [s - l for (s, _), l in zip(seqs, lo)]
    row0 = [4]                                                              # rows in front belong to somebody else
    tok0 = [0]
    for (s, n), a in zip(seqs, ahead):
        row0.append(row0[-1] + n)
        tok0.append(tok0[-1] + a + n)
    T, N, D = row0[-1], tok0[-1], kp + 64
    q, k, v = rnd(g, T, H_, D), 0.5 * rnd(g, N, H_, D), rnd(g, N, H_, vp)
    v[..., vdim:] = 0
    k[..., kp:] = k[:, :1, kp:]                                            # the rotated part is shared by the heads
    for b, (s, n) in enumerate(seqs):
        if window:
            for i in {n - 1, n // 2, 0}:
                for j in (ahead[b] + i - window + 1, ahead[b] + i - window):
                    if j >= 0:
                        k[tok0[b] + j] *= 3.0
                        q[row0[b] + i] += 0.7 * k[tok0[b] + j]
    q, k, v = (t.to(BF16) for t in (q, k, v))
    k[..., kp:] = k[:, :1, kp:]
    out = torch.full((T, H_ * vdim + 8), 3.0, dtype=BF16, device=DEV)
    kd = torch.cat([k[..., :kp].reshape(N, -1), v.reshape(N, -1)], 1).contiguous().to(DEV)
    kr = torch.cat([torch.zeros(N, 64, dtype=BF16), k[:, 0, kp:]], 1).contiguous().to(DEV)
    H.latent_prefill(q.reshape(T, -1).contiguous().to(DEV), kd[:, : H_ * kp], kd[:, H_ * kp:], kr[:, 64:], out, i32(*row0[:-1]),
                     i32(*[n for _, n in seqs]), i32(*tok0[:-1]), i32(*ahead), max(n for _, n in seqs), H_, kp, vp, vdim, window, scale)
    for b, (s, n) in enumerate(seqs):
        kk, vv = k[tok0[b]: tok0[b] + ahead[b] + n].double(), v[tok0[b]: tok0[b] + ahead[b] + n].double()
        qq = torch.cat([q.new_zeros(ahead[b], H_, D), q[row0[b]: row0[b] + n]]).double()
        want = O.window_attention(qq, kk, vv, scale, window)[ahead[b]:, :, :vdim]
        close(out[row0[b]: row0[b] + n, : H_ * vdim].view(n, H_, vdim), want, 1.2e-2, f"sequence {b}")
    assert bool((out[:4] == 3.0).all()) and bool((out[:, H_ * vdim:] == 3.0).all())


# ---- gated linear recurrence -----------------------------------------------------------------------------------------------
def _rglru(width, blocks, taps, dtype, D=64, seed=0):
    from sglang_security_amd.layers.rglru import Rglru
    from sglang_security_amd.mem_cache.memory_pool import RecurrentStatePool

    cfg = M.config([M.recurrent(width, blocks, taps)], width=D)
    w = {k[len("l0.mix."):]: v for k, v in M.weights(cfg, seed).items() if k.startswith("l0.mix.")}
    layer = Rglru(cfg["layers"][0]["mixer"], lambda n: w[n].to(dtype).to(DEV), 128, dtype)
    return layer, RecurrentStatePool(5, layer.W, taps, dtype, DEV), w, cfg["layers"][0]["mixer"]


class _Batch:
    """Rows of a step for a layer alone: [(slot, position of the first row, rows)], single rows first."""

    def __init__(self, seqs):
        from sglang_security_amd.ops_hybrid import RowSeqs

        self.singles = sum(1 for s in seqs if s[2] == 1)
        row0, row_seq, tile0, tr, tn = [], [], [], [], []
        r = 0
        for s, (_, _, n) in enumerate(seqs):
            row0.append(r)
            row_seq += [s] * n
            tile0.append(len(tr))
            if n > 1:
                tr += range(r, r + n, 64)
                tn += [min(64, n - t) for t in range(0, n, 64)]
            r += n
        self.seqs = RowSeqs(i32(*row_seq), i32(*row0), i32(*[n for _, _, n in seqs]), i32(*[p for _, p, _ in seqs]),
                            i32(*[s for s, _, _ in seqs]))
        self.tile0, self.tile_row, self.tile_rows = i32(*tile0), i32(*tr), i32(*tn)


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("width,blocks,taps", [(60, 3, 4), (64, 1, 1), (192, 2, 2), (128, 4, 4), (96, 8, 7), (512, 2, 4)])
def test_rglru_portions_and_slots(dtype, width, blocks, taps):
    """Four sequences of which pieces of every length run together, slots reused for later sequences."""
    layer, cache, w, c = _rglru(width, blocks, taps, dtype)
    cache.state.fill_(1e3)                                                     # what an earlier owner left
    cache.conv.fill_(1e3)
    g = gen(width)
    seqs = [rnd(g, n, 64, dtype=dtype) for n in (200, 70, 66, 5)]
    want = [O.rglru(x.double(), {k: v.double() for k, v in w.items()}, c) for x in seqs]
    slot, at, got = [3, 0, 4, 1], [0] * 4, [[] for _ in seqs]
    plan = [{0: 64, 1: 2}, {0: 1, 1: 1, 2: 1, 3: 2}, {0: 67, 2: 63, 1: 3}, {0: 2, 1: 1, 3: 1, 2: 2}, {3: 2, 1: 63, 0: 1}, {0: 65}]
    for step in plan:
        order = sorted(step, key=lambda s: step[s] > 1)
        b = _Batch([(slot[s], at[s], step[s]) for s in order])
        h = torch.zeros(sum(step.values()), 128, dtype=dtype)
        h[:, :64] = torch.cat([seqs[s][at[s]: at[s] + step[s]] for s in order])
        out = layer.forward(h.to(DEV), b, cache).data
        out = (out.sum(0) if out.dim() == 3 else out).double().cpu()[:, :64]
        r = 0
        for s in order:
            got[s].append(out[r: r + step[s]])
            at[s] += step[s]
            r += step[s]
    tol = 2e-5 if dtype == F32 else 2.5e-2
    for s in range(4):
        close(torch.cat(got[s]), want[s][: at[s]], tol, f"sequence {s}")
    # a slot given to a new sequence behaves as if it had been cleared
    b = _Batch([(3, 0, 5)])
    h = torch.zeros(5, 128, dtype=dtype)
    h[:, :64] = seqs[3]
    out = layer.forward(h.to(DEV), b, cache).data
    close((out.sum(0) if out.dim() == 3 else out)[:, :64], want[3], tol, "reused slot")


def test_recurrent_memory_reaches_far_back():
    """Decays close to one: the first token still shows after a thousand, whichever way the rows were cut."""
    layer, cache, w, c = _rglru(64, 2, 4, F32)
    w["lam"].fill_(-11.0)
    layer, cache, _, _ = _rglru(64, 2, 4, F32)
    layer.w.sp.copy_(torch.nn.functional.softplus(torch.tensor(-11.0)).expand_as(layer.w.sp))
    x = torch.zeros(1000, 64)
    x[0] = 5.0
    want = O.rglru(x.double(), {k: v.double() for k, v in w.items()}, c)
    h = torch.zeros(1000, 128)
    h[:, :64] = x
    out = torch.cat([layer.forward(h[a:b].to(DEV), _Batch([(2, a, b - a)]), cache).data[0] for a, b in ((0, 130), (130, 999), (999, 1000))])
    close(out[:, :64], want, 3e-5, "whole")
    quiet = O.rglru(torch.zeros_like(x).double(), {k: v.double() for k, v in w.items()}, c)
    assert (want[-1] - quiet[-1]).abs().max() > 1e-2 * want[-1].abs().max()


# ---- the whole model through the engine ------------------------------------------------------------------------------------
@functools.lru_cache(None)
def oracle_logits(name, seed, n):
    cfg = M.CONFIGS[name]
    return O.forward(cfg, M.weights(cfg), M.tokens(cfg, n, seed))


@pytest.fixture(scope="module")
def engines():
    from sglang_security_amd.engine import Engine
    from sglang_security_amd.model_loader import Weights
    from sglang_security_amd.models import model_class

    made = {}

    def get(name, dtype, max_tokens=640, max_requests=4, **kw):
        key = (name, dtype)
        if key not in made:
            cfg = M.CONFIGS[name]
            ws = Weights(M.weights(cfg), dtype, torch.device(DEV, 0))
            made[key] = model_class(cfg)(cfg, ws, dtype, torch.device(DEV, 0), 640)
            ws.check_all_used()
        return Engine(made[key], max_tokens, max_requests, **kw)

    return get


CASES = [(n, d) for n in M.CONFIGS for d in (F32, BF16)]


def agrees(err, dtype, noise, what):
    """Relative errors per row.  bf16: rounding is amplified at single tokens of a random model; `noise` is what a small
    disturbance of the oracle does to each row."""
    limit = torch.full_like(err, 1e-4) if dtype == F32 else 0.02 + 5 * noise[: len(err)]
    at = int((err / limit).argmax())
    says = f"{what}: {float(err[at]):.4g} at row {at} of {len(err)}, limit {float(limit[at]):.4g}, mean {float(err.mean()):.4g}"
    assert bool((err <= limit).all()) and float(err.mean()) <= (1e-4 if dtype == F32 else 0.035), says


@functools.lru_cache(None)
def oracle_noise(name, seed, n):
    """Largest relative change of each logits row over three runs with norm outputs disturbed by 2^-9."""
    cfg, plain = M.CONFIGS[name], O.rms_norm
    want, worst = oracle_logits(name, seed, n)[0], torch.zeros(n, dtype=torch.float64)
    try:
        for k in range(3):
            g = gen(k)
            O.rms_norm = lambda x, w, e: plain(x, w, e) * (1 + 2 ** -9 * torch.randn(x.shape, generator=g, dtype=torch.float64))
            worst = torch.maximum(worst, M.rel_rms(O.forward(cfg, M.weights(cfg), M.tokens(cfg, n, seed))[0], want))
    finally:
        O.rms_norm = plain
    return worst


def run(engine, name, plan, check=True):
    """plan: steps of {sequence id: (seed, total length, rows now)}; a sequence closes when its tokens are through.
    Returns {id: logits} and compares them with the oracle."""
    from sglang_security_amd.engine import Entry

    cfg, live, got, meta = M.CONFIGS[name], {}, {}, {}
    for step in plan:
        entries, ids = [], []
        for sid, (seed, total, n) in step.items():
            if sid not in live:
                live[sid] = engine.open()
                got[sid], meta[sid] = [], (seed, total)
            at = live[sid].length
            entries.append(Entry(live[sid], M.tokens(cfg, total, seed)[at: at + n], range(n)))
            ids.append(sid)
        out = engine.step(entries).cpu()
        r = 0
        for sid, e in zip(ids, entries):
            got[sid].append(out[r: r + len(e.tokens)])
            r += len(e.tokens)
            if live[sid].length == meta[sid][1]:
                engine.close(live.pop(sid))
    got = {sid: torch.cat(v) for sid, v in got.items()}
    if check:
        for sid, (seed, total) in meta.items():
            err = M.rel_rms(got[sid], oracle_logits(name, seed, total)[0][: len(got[sid])])
            agrees(err, engine.model.dtype, oracle_noise(name, seed, total), f"{name} {sid}")
    return got


def cut(seed, total, parts):
    out, at, i = [], 0, 0
    while at < total:
        n = min(parts[i % len(parts)], total - at)
        out.append((seed, total, n))
        at, i = at + n, i + 1
    return out


@pytest.mark.parametrize("name,dtype", CASES)
def test_whole_prompts_and_residual_stream(engines, name, dtype):
    from sglang_security_amd.engine import Entry

    e = engines(name, dtype)
    for seed, n in enumerate((1, 2, 3, 150, 300)):
        run(e, name, [{0: (seed, n, n)}])
    s, col = e.open(), []
    e.step([Entry(s, M.tokens(M.CONFIGS[name], 150, 3), [149])], collect=col)
    stream = oracle_logits(name, 3, 150)[1]
    assert len(col) == len(stream)
    for i, (a, b) in enumerate(zip(col, stream)):
        agrees(M.rel_rms(a, b), dtype, oracle_noise(name, 3, 150), f"layer run {i}")
    e.close(s)


@pytest.mark.parametrize("name,dtype", CASES)
def test_token_by_token_equals_the_prompt(engines, name, dtype):
    e = engines(name, dtype)
    run(e, name, [{0: p} for p in cut(3, 150, [1])])                      # graph replays from the third step on
    run(e, name, [{0: p} for p in cut(4, 300, [180] + [1] * 120)])


@pytest.mark.parametrize("name,dtype", CASES)
@pytest.mark.parametrize("parts", [[2], [3, 2, 37], [64, 1, 63, 65], [5, 40, 2, 130]])
def test_portions(engines, name, dtype, parts):
    run(engines(name, dtype), name, [{0: p} for p in cut(3, 150, parts)])


@pytest.mark.parametrize("name,dtype", CASES)
def test_mixed_batches_with_reused_slots(engines, name, dtype):
    """Unequal requests come and go; portions beside single tokens; some are left out of steps; 640 slots serve more
    than a thousand tokens."""
    e = engines(name, dtype)
    queue = [(i, cut(seed, n, parts)) for i, (seed, n, parts) in enumerate(
        [(4, 300, [100, 1, 1, 1, 50, 2]), (0, 1, [1]), (3, 150, [37, 3, 24, 2]), (5, 90, [60] + [1] * 30), (6, 97, [97]),
         (7, 66, [64, 2]), (8, 120, [1, 2, 40, 1]), (9, 200, [150] + [1] * 50), (3, 150, [149, 1]), (2, 3, [2, 1])])]
    live, plan, t = [], [], 0
    while queue or live:
        while queue and len(live) < 4:
            live.append(queue.pop(0))
        step = {}
        for k, (sid, parts) in enumerate(live):
            if len(live) > 1 and (t + k) % 5 == 4:
                continue
            step[sid] = parts.pop(0)
        live = [x for x in live if x[1]]
        plan.append(step)
        t += 1
    run(e, name, plan)
    assert e.free_tokens() == 640 and e.cache.req_pool.available_size() == 4


@pytest.mark.parametrize("name", list(M.CONFIGS))
def test_batches_equal_each_alone(engines, name):
    """bf16: the same requests alone, together, and on other slots differ by rounding only."""
    e = engines(name, BF16)
    alone = {s: run(e, name, [{s: p} for p in cut(s, n, [n - 4, 1, 1, 1, 1])])[s] for s, n in ((3, 150), (5, 90), (6, 97))}
    steps = [dict(zip((3, 5, 6), ps)) for ps in zip(*[cut(s, n, [n - 4, 1, 1, 1, 1]) for s, n in ((3, 150), (5, 90), (6, 97))])]
    both = run(e, name, steps)
    for s, n in ((3, 150), (5, 90), (6, 97)):
        agrees(M.rel_rms(both[s], alone[s].double()), BF16, oracle_noise(name, s, n), f"{name} {s}")


def test_graph_replays_equal_eager_steps(engines):
    from sglang_security_amd.engine import Entry

    name = "mixed"
    a, b = engines(name, BF16), engines(name, BF16, use_graph=False)
    sa, sb = [a.open() for _ in range(3)], [b.open() for _ in range(3)]
    t = M.tokens(M.CONFIGS[name], 120, 1)
    for e, s in ((a, sa), (b, sb)):
        e.step([Entry(q, t[:n]) for q, n in zip(s, (40, 1, 9))])
    for i in range(24):
        want = [[0], [], [0]] if i % 3 else [[0]] * 3
        n = 3 if i % 4 else 2
        la, lb = (e.step([Entry(q, [t[50 + i + j]], w) for j, (q, w) in enumerate(zip(s[:n], want))]) for e, s in ((a, sa), (b, sb)))
        assert torch.equal(la, lb), f"step {i}"
        torch.randn(1000, device=DEV).sum().item()                        # the program's own work between the replays
    assert set(a.graphs) == {2, 3} and not b.graphs


@pytest.mark.parametrize("name", list(M.CONFIGS))
def test_greedy_generation_through_the_scheduler(engines, name):
    from sglang_security_amd.engine import SamplingParams, Scheduler

    cfg = M.CONFIGS[name]
    prompts = [M.tokens(cfg, n, 50 + n) for n in (3, 41, 70, 1, 25, 9)]
    outs = Scheduler(engines(name, F32), prefill_budget=32).generate(prompts, SamplingParams(max_new_tokens=12))
    for p, o in zip(prompts, outs):
        lg, _ = O.forward(cfg, M.weights(cfg), p + o)
        for i, t in enumerate(o):
            row = lg[len(p) - 1 + i]
            assert float(row[t]) >= float(row.max()) - 1e-3, f"token {i}"      # the arg-max, ties aside
    # bf16: every pick lies within rounding of the best logit, greedy runs repeat themselves
    sched = Scheduler(engines(name, BF16), prefill_budget=32)
    outs = sched.generate(prompts, SamplingParams(max_new_tokens=12))
    for p, o in zip(prompts, outs):
        lg, _ = O.forward(cfg, M.weights(cfg), p + o)
        spread = float((lg ** 2).mean().sqrt())
        for i, t in enumerate(o):
            row = lg[len(p) - 1 + i]
            assert float(row[t]) >= float(row.max()) - 0.3 * spread
    assert sched.generate(prompts, SamplingParams(max_new_tokens=12)) == outs


def test_sampled_generation(engines):
    from sglang_security_amd.engine import SamplingParams, Scheduler

    cfg = M.CONFIGS["mixed"]
    prompts = [M.tokens(cfg, 20, s) for s in range(4)]
    greedy = Scheduler(engines("mixed", BF16)).generate(prompts, SamplingParams(max_new_tokens=6))
    assert Scheduler(engines("mixed", BF16)).generate(prompts, SamplingParams(max_new_tokens=6, temperature=0.7, top_k=1)) == greedy
    assert Scheduler(engines("mixed", BF16)).generate(prompts, SamplingParams(max_new_tokens=6, temperature=0.7, min_p=1.0)) == greedy
    draw = lambda seed: Scheduler(engines("mixed", BF16), seed=seed).generate(prompts, SamplingParams(max_new_tokens=6, temperature=2.0, top_p=0.95))
    assert draw(1) == draw(1) and draw(1) != draw(2)


def test_command_line_and_trace(tmp_path):
    """generate and trace from a checkpoint folder, in processes of their own."""
    import numpy as np

    name = "tail"
    cfg = M.CONFIGS[name]
    folder = M.save(str(tmp_path / "model"), cfg, M.weights(cfg))
    t = M.tokens(cfg, 90, 5)
    r = subprocess.run([sys.executable, "-m", "sglang_security_amd.cli", "generate", "--model", folder, "--dtype", "float32",
                        "--prompt-ids", ",".join(map(str, t[:30])), "--max-new-tokens", "5"], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    out = json.loads(r.stdout.strip().splitlines()[-1])["output_ids"]
    lg, _ = O.forward(cfg, M.weights(cfg), t[:30] + out)
    assert len(out) == 5 and all(float(lg[29 + i].max() - lg[29 + i][v]) < 1e-3 for i, v in enumerate(out))
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": t[:50], "want": [49, 0]}, {"id": "b", "tokens": t[:1], "want": []}], "end": []},
             {"step": 1, "entries": [{"id": "b", "tokens": t[1:4], "want": []}], "end": ["b"]},
             {"step": 2, "entries": [{"id": "c", "tokens": t[:2], "want": [1]}, {"id": "a", "tokens": t[50:51], "want": [0]}], "end": ["a", "c"]}]
    p = subprocess.run(["bin/trace_run", "--model", folder, "--dtype", "float32", "--out", str(tmp_path), "--max-tokens", "128"],
                       input="\n".join(map(json.dumps, steps)) + "\n", capture_output=True, text=True, timeout=100, cwd=_root())
    assert p.returncode == 0, p.stderr[-2000:]
    assert [l for l in p.stdout.splitlines() if l.startswith("done")] == ["done 0", "done 1", "done 2"]
    lg = oracle_logits(name, 5, 90)[0]
    read = lambda n: torch.from_numpy(np.fromfile(tmp_path / f"{n}.f32", "<f4")).view(-1, cfg["vocab"])
    assert float(M.rel_rms(read(0), lg[[49, 0]]).max()) < 1e-4 and not (tmp_path / "1.f32").exists()
    assert float(M.rel_rms(read(2), lg[[1, 50]]).max()) < 1e-4


def _root():
    import os

    return os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
