"""GPU tests of the extend (prefill-with-prefix) forward and of the prefix-cache harness around it: the whole-model
extend against a torch restatement that rounds where the kernels round, a prefix served from the radix cache against
the same request recomputed from scratch, and the SafeKV rule that a private prefix is shared with its owner only."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _tiny(quant="awq"):
    from sglang_security_amd.decode_runner import LlamaConfig, LlamaDecoder

    cfg = LlamaConfig.tiny(quant)
    return LlamaDecoder(cfg, 1, 2, 16, device=DEV)


def _weight(w):
    from sglang_security_amd import ops

    if hasattr(w, "packed"):
        return ops.awq_dequantize_packed(w.packed, w.scales, w.qzeros).float()
    if getattr(w, "wpacked", None) is not None:
        # the streaming layout read back through the product with the identity (exact in 16 bits)
        eye = torch.eye(w.K, dtype=w.wpacked.dtype, device=w.wpacked.device)
        return ops.dense_gemm_packed(eye, w.wpacked).float()
    return w.weight.t().float()


def _r(x):
    return x.to(torch.bfloat16).float()


def _ref_forward(dec, ids):
    """Whole sequence from scratch, fp32 math, rounded to bf16 where the kernel path stores bf16."""
    c = dec.cfg
    T = len(ids)
    x = dec.embed[ids].float()
    pos = torch.arange(T, device=DEV)
    cs = dec.cos_sin[pos]
    half = c.head_dim // 2
    cos, sin = cs[:, :half], cs[:, half:]
    res = None

    def norm(v, w):
        return _r(v * torch.rsqrt((v * v).mean(-1, keepdim=True) + c.eps) * w.float())

    def rope(t):                                         # [T, H, D], neox halves
        a, b = t[..., :half], t[..., half:]
        return _r(torch.cat([a * cos[:, None] - b * sin[:, None], b * cos[:, None] + a * sin[:, None]], -1))

    for li, L in enumerate(dec.layers):
        res = x if li == 0 else _r(res + x)
        h = norm(res, L["ln1"])
        qkv = _r(h @ _weight(L["qkv"]))
        q = rope(qkv[:, : dec.q_size].view(T, c.q_heads, c.head_dim))
        k = rope(qkv[:, dec.q_size: dec.q_size + dec.kv_size].view(T, c.kv_heads, c.head_dim))
        v = qkv[:, dec.q_size + dec.kv_size:].view(T, c.kv_heads, c.head_dim)
        rep = c.q_heads // c.kv_heads
        kk, vv = k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1)
        s = torch.einsum("thd,shd->hts", q, kk) / math.sqrt(c.head_dim)
        s = s.masked_fill(torch.triu(torch.ones(T, T, dtype=torch.bool, device=DEV), 1), float("-inf"))
        o = _r(torch.einsum("hts,shd->thd", torch.softmax(s, -1), vv)).reshape(T, -1)
        x = _r(o @ _weight(L["o"]))
        res = _r(res + x)
        h = norm(res, L["ln2"])
        gu = _r(h @ _weight(L["gate_up"]))
        act = _r(_r(torch.nn.functional.silu(gu[:, : c.inter])) * gu[:, c.inter:])
        x = _r(act @ _weight(L["down"]))
    return x, res


def _rel(a, b):
    return ((a.float() - b.float()).norm() / b.float().norm()).item()


@pytest.mark.parametrize("T,gemm", [(40, "library"), (300, "library"), (300, "fused")])   # below / above the switch to
@pytest.mark.parametrize("quant", ["awq", "bf16"])                                         # large-batch GEMMs, both kinds
def test_extend_matches_torch(T, gemm, quant):
    from sglang_security_amd.prefill_runner import PrefixCacheHarness

    dec = _tiny(quant)
    h = PrefixCacheHarness(dec, 4096, 2048, None, prefill_gemm=gemm)
    ids = torch.randint(0, dec.cfg.vocab, (T,), generator=torch.Generator().manual_seed(T)).tolist()
    tok, pre, req = h.serve_first_token(ids, "u", finish=False)
    assert pre == 0
    got_x, got_res = h.model.hidden[:T], h.model.residual[:T]
    want_x, want_res = _ref_forward(dec, torch.tensor(ids, device=DEV))
    assert _rel(got_res, want_res) < 2e-2
    assert _rel(got_x, want_x) < 3e-2
    # the KV the pool now holds for the request is what the restatement computed (layer 0 keys, rotated)
    assert h.tree.total_size() == 0
    h.finish(req, int(tok.item()))
    assert h.tree.total_size() == T


def test_overlapped_dequantisation_gives_the_same_bits():
    """The library path dequantises projection i + 1 on a second stream under the product of projection i; the
    result is the one of the two in sequence, on the first extend and on a second one that re-uses the buffers."""
    from sglang_security_amd.prefill_runner import PrefixCacheHarness

    dec = _tiny("awq")
    a = PrefixCacheHarness(dec, 4096, 2048, None, overlap_dequant=True)
    b = PrefixCacheHarness(dec, 4096, 2048, None, overlap_dequant=False)
    for T in (300, 517, 256):
        ids = torch.randint(0, dec.cfg.vocab, (T,), generator=torch.Generator().manual_seed(T)).tolist()
        ta, _, _ = a.serve_first_token(ids, None)
        tb, _, _ = b.serve_first_token(ids, None)
        torch.cuda.synchronize()
        assert a.model._ring is not None and b.model._ring is None
        assert torch.equal(a.model.hidden[:T], b.model.hidden[:T])
        assert torch.equal(a.model.residual[:T], b.model.residual[:T])
        assert int(ta.item()) == int(tb.item())
        for h in (a, b):
            h.tree.reset()
            h.alloc.clear()
            h.req_pool.clear()


def test_prefix_hit_equals_recompute():
    """A request whose first 1024 tokens are served from the radix cache ends in the same hidden state (within bf16
    accumulation noise) and the same first token as the same request computed from scratch."""
    from sglang_security_amd.prefill_runner import PrefixCacheHarness

    dec = _tiny("awq")
    g = torch.Generator().manual_seed(5)
    shared = torch.randint(0, dec.cfg.vocab, (1024,), generator=g).tolist()
    a = shared + torch.randint(0, dec.cfg.vocab, (24,), generator=g).tolist()
    b = shared + torch.randint(0, dec.cfg.vocab, (40,), generator=g).tolist()
    h = PrefixCacheHarness(dec, 8192, 2048, None)
    _, pre_a, _ = h.serve_first_token(a, None)
    tok_hit, pre_b, _ = h.serve_first_token(b, None, finish=False)
    assert (pre_a, pre_b) == (0, 1024)
    hit_x = h.model.hidden[:40].clone()
    hit_res = h.model.residual[:40].clone()
    tok_hit = int(tok_hit.item())
    cold = PrefixCacheHarness(dec, 8192, 2048, None)
    tok_cold, pre_c, _ = cold.serve_first_token(b, None, finish=False)
    assert pre_c == 0
    # 40 tokens go through the fused int4 GEMM, 1064 through dequantise + GEMM: the two paths round differently, so
    # the bound is the one of the comparison with the torch restatement
    assert _rel(hit_res, cold.model.residual[1024:1064]) < 2e-2
    assert _rel(hit_x, cold.model.hidden[1024:1064]) < 3e-2
    assert tok_hit == int(tok_cold.item())


def test_safekv_private_prefix_is_owner_only():
    from sglang_security_amd.prefill_runner import PrefixCacheHarness
    from sglang_security_amd.private_service.private_client import PrivateJudgeClient

    dec = _tiny("awq")
    g = torch.Generator().manual_seed(6)
    shared = torch.randint(0, dec.cfg.vocab, (1024,), generator=g).tolist()
    tail = lambda: torch.randint(0, dec.cfg.vocab, (16,), generator=g).tolist()
    for private, want_other in ((True, 0), (False, 1024)):
        judge = PrivateJudgeClient(detector=lambda text, p=private: p)
        h = PrefixCacheHarness(dec, 8192, 2048, judge)
        _, pre, _ = h.serve_first_token(shared + tail(), "victim", "a line\nUser: q")
        assert pre == 0 and judge.drain()
        _, pre_owner, _ = h.serve_first_token(shared + tail(), "victim", "a line\nUser: q")
        assert judge.drain()
        _, pre_other, _ = h.serve_first_token(shared + tail(), "attacker", "a line\nUser: q")
        assert pre_owner == 1024
        assert pre_other == want_other
        judge.close()


def test_graph_replay_equals_eager():
    """The captured single-request extend gives the bits of the eager one, on the capture call and on replays with
    other tokens, another prefix length and the same token count."""
    from sglang_security_amd.prefill_runner import PrefixCacheHarness

    dec = _tiny("awq")
    g = torch.Generator().manual_seed(9)
    rnd = lambda n: torch.randint(0, dec.cfg.vocab, (n,), generator=g).tolist()
    shared = rnd(1024)
    reqs = [shared + rnd(30), shared + rnd(30), shared[:512] + rnd(542), shared + rnd(30), rnd(30)]
    outs = []
    for use_graph in (True, False):
        h = PrefixCacheHarness(dec, 16384, 2048, None, use_graph=use_graph)
        got = []
        for r in reqs:
            tok, pre, _ = h.serve_first_token(r, None)
            ext = len(r) - pre
            got.append((pre, int(tok.item()), h.model.hidden[:ext].clone(), h.model.residual[:ext].clone()))
        outs.append(got)
        if use_graph:
            assert any(k[0] == 30 for k in h.model.graphs)   # requests 2, 4 and 5 extend 30 tokens
    for a, b in zip(*outs):
        assert a[0] == b[0] and a[1] == b[1]
        assert torch.equal(a[2], b[2]) and torch.equal(a[3], b[3])


def test_bench_tiny_line_and_ttft_block():
    """bench.py end to end on the tiny configuration: one JSON line with the contract's keys, and the
    time-to-first-token experiment on the same model (cache hits where expected)."""
    import json
    import os
    import subprocess
    import sys

    from sglang_security_amd.prefill_runner import ttft_experiment

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--tiny", "--steps", "3", "--warmup", "1",
                        "--no-cpu-baseline"], capture_output=True, text=True, timeout=300, cwd=root)
    assert r.returncode == 0, r.stderr[-2000:]
    line = json.loads(r.stdout.strip().splitlines()[-1])
    for key in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
                "vs_baseline", "dtype", "data", "config"):
        assert key in line
    assert line["steps"] == 3 and line["n_gpus"] == 1 and line["value"] > 0 and "workload" in line["config"]
    out = ttft_experiment(_tiny("awq"), 1024, 16, pool_tokens=8192, repeats=1)
    assert out["public"]["cached_prefix_tokens_cold_other_owner"] == [0, 1024, 1024]
    assert out["private"]["cached_prefix_tokens_cold_other_owner"] == [0, 0, 1024]


@pytest.mark.parametrize("counts", [(1,), (5, 0, 300), (128, 128, 128, 2, 2, 70000), (0, 0)])
def test_copy_indices(counts):
    """Vectors of both widths, empty ones and ones longer than a block, and nothing beside them is written."""
    from sglang_security_amd import ops
    from sglang_security_amd._lib import SglkError

    g = torch.Generator().manual_seed(sum(counts))
    kinds = [(torch.int32, torch.int32), (torch.int64, torch.int32), (torch.int32, torch.int64), (torch.int64, torch.int64)]
    src = [torch.randint(-9, 2**31 - 1, (n,), generator=g).to(kinds[i % 4][0]).to(DEV) for i, n in enumerate(counts)]
    whole = [torch.full((n + 2,), -77, dtype=kinds[i % 4][1], device=DEV) for i, n in enumerate(counts)]
    ops.copy_indices([w[1:-1] for w in whole], src)
    for w, s in zip(whole, src):
        assert torch.equal(w[1:-1].long(), s.long()) and w[0] == -77 and w[-1] == -77
    with pytest.raises(SglkError):
        ops.copy_indices([whole[0]], [src[0]])


def test_extend_refuses_more_cached_tokens_than_indices():
    """kv_indptr beyond kv_indices is an error, and the next extend is right."""
    from sglang_security_amd.mem_cache.memory_pool import MHATokenToKVPool
    from sglang_security_amd.prefill_runner import LlamaPrefill

    dec = _tiny()
    c = dec.cfg
    kv = MHATokenToKVPool(128, 1, torch.bfloat16, c.kv_heads, c.head_dim, c.layers, DEV)
    model = LlamaPrefill(dec, kv, 64)
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)
    ids, pos, loc = torch.arange(8, device=DEV), torch.arange(8, device=DEV), torch.arange(1, 9, device=DEV)
    good = (ids, pos, loc, i32(0, 8), i32(0, 0), i32(0), 8)
    want = [t.clone() for t in model.extend(*good)]
    with pytest.raises(RuntimeError):
        model.extend(ids, pos, loc, i32(0, 8), i32(0, 5), i32(20, 21, 22), 8)
    # ... also where a copy of the indices would fit: one that could be spread over all of them, and as many as the buffer holds
    for pre, have in ((5, i32(20)), (65, torch.arange(1, 65, dtype=torch.int32, device=DEV))):
        with pytest.raises(RuntimeError, match="cached tokens"):
            model.extend(ids, pos, loc, i32(0, 8), i32(0, pre), have, 8)
    assert all(torch.equal(a, b) for a, b in zip(model.extend(*good), want))
    # vectors of other widths, and views with gaps, are copied one by one or converted
    got = model.extend(ids.int(), pos.repeat_interleave(2)[::2], loc.int(), i32(0, 8).long(), i32(0, 0), i32(0).long(), 8)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
