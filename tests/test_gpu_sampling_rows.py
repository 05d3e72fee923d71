"""GPU: the sampling filters' radix selection where its shortcuts end: rows of peaked, flat, tied and unnormalised
values, lists that overflow, thresholds below the mean, vocabularies that are no multiple of a load or a chunk, and rows
that are not aligned.  Values are sums of few powers of two, so that every mass is exact and so is the kept set."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rows(kind, n, g):
    e = {"peaked": lambda: torch.randint(-20, 1, (n,), generator=g), "flat": lambda: torch.zeros(n, dtype=torch.long),
         "two": lambda: torch.randint(-1, 1, (n,), generator=g) * 9,
         "steep": lambda: -(torch.arange(n) * 22 // n)[torch.randperm(n, generator=g)]}[kind]()
    x = 2.0 ** e.double()
    if kind == "peaked":
        x = x * (1 + torch.randint(0, 8, (n,), generator=g) / 8)
    return x


def _threshold(x, k, p, joint):
    thr = 0.0
    s = x.sort(descending=True).values
    if 0 < k < len(x):
        thr = s[k - 1].item()
    if p < 1:
        lo = thr if (0 < k < len(x) and not joint) else 0.0
        v = x[x >= lo].sort().values
        target = (1 - p) * v.sum()
        at = torch.nonzero(v.cumsum(0) >= target)
        thr = max(thr, v[at[0, 0]].item() if len(at) else v[-1].item())
    return thr


@pytest.mark.parametrize("kind", ["peaked", "flat", "two", "steep"])
@pytest.mark.parametrize("n", [1, 3, 255, 4099, 40000, 128259])
@pytest.mark.parametrize("scale", [None, 2.0 ** -30, 2.0 ** 12])   # None: a mass between one half and one, as probabilities have
def test_kept_sets(kind, n, scale):
    import sglang_security_amd.sgl_kernel as sk
    from sglang_security_amd import ops

    g = torch.Generator().manual_seed(n)
    x = _rows(kind, n, g)
    x = x * (scale or 2.0 ** -math.ceil(math.log2(x.sum().item())))
    B = 6
    wide = torch.zeros(B, n + 5, device=DEV)
    wide[:, 1: n + 1] = x.float().to(DEV)
    aligned = torch.zeros(B, (n + 3) // 4 * 4, device=DEV)
    aligned[:, :n] = x.float().to(DEV)
    ks = [0, 1, min(50, n), n // 2, n - 1, n]
    ps = [0.75, 0.5, 0.875, 0.0, 1.0, 0.9375]       # exact in fp32
    kt, pt = torch.tensor(ks, dtype=torch.int32, device=DEV), torch.tensor(ps, device=DEV)
    for rows in (wide[:, 1: n + 1], aligned[:, :n]):
        got_p = sk.top_p_renorm_probs(rows, pt).cpu().double()
        got_k = sk.top_k_renorm_probs(rows, kt).cpu().double()
        for b in range(B):
            for got, want in ((got_p, _threshold(x, 0, ps[b], True)), (got_k, _threshold(x, ks[b], 1.0, True))):
                kept = torch.where(x >= want, x, 0.0)
                assert torch.equal(got[b] > 0, kept > 0)
                assert torch.allclose(got[b], kept / kept.sum(), rtol=1e-5, atol=0)
        for joint in (True, False):
            for u in (0.0, 0.3, 0.999999):
                ids = ops.sampling_from_probs(rows, torch.full((B,), u, device=DEV), kt, pt, 0.0, joint).cpu().long()
                for b in range(B):
                    kept = torch.where(x >= _threshold(x, ks[b], ps[b], joint), x, 0.0)
                    cum = kept.cumsum(0) / kept.sum()
                    i = int(ids[b])
                    assert kept[i] > 0
                    # the running sum passes u at the chosen index, up to the rounding of fp32 sums
                    assert cum[i] >= u - 1e-5 and (i == 0 or cum[i - 1] <= u + 1e-5)


@pytest.mark.parametrize("B,n", [(64, 128259), (64, 163843), (100, 128259), (128, 81923), (20, 8195 * 12)])
def test_spread_rows_of_large_batches(B, n):
    """Rows over two, four and twelve blocks with slices of 8192 to 64000 elements, and a row's last three."""
    import sglang_security_amd.sgl_kernel as sk
    from sglang_security_amd import ops

    g = torch.Generator().manual_seed(n + B)
    x = _rows("peaked", n, g)
    x[-2] = 2.0                                     # the last elements are kept ones
    x = x * 2.0 ** -math.ceil(math.log2(x.sum().item()))
    rows = torch.zeros(B, (n + 3) // 4 * 4, device=DEV)[:, :n]
    rows[:] = x.float().to(DEV)
    ps = torch.tensor([0.75, 0.5, 0.875, 0.9375][: 4] * (B // 4 + 1), device=DEV)[:B]
    got = sk.top_p_renorm_probs(rows, ps).cpu().double()
    ids = ops.sampling_from_probs(rows, torch.full((B,), 0.999999, device=DEV), 0, ps, 0.0, True).cpu().long()
    for b in range(4):
        kept = torch.where(x >= _threshold(x, 0, ps[b].item(), True), x, 0.0)
        cum = kept.cumsum(0) / kept.sum()
        for r in range(b, B, 4):
            assert torch.equal(got[r] > 0, kept > 0)
            assert torch.allclose(got[r], kept / kept.sum(), rtol=1e-5, atol=0)
            i = int(ids[r])
            assert kept[i] > 0 and cum[i] >= 0.999999 - 1e-5


@pytest.mark.parametrize("n", [1, 3, 255, 4099, 8192, 8193, 65536, 65537])
@pytest.mark.parametrize("B", [5, 300])
@pytest.mark.parametrize("min_p", [0.0, 0.5])
def test_rows_without_top_k_and_top_p(n, B, min_p):
    """The kernel without a selection, and the spread rows: multiples of 2^-10, so every mass is exact."""
    import sglang_security_amd.sgl_kernel as sk
    from sglang_security_amd import ops

    g = torch.Generator().manual_seed(n + B)
    x = torch.randint(0, 9, (B, n), generator=g).float()
    x[:, n // 2] = 8.0
    u = torch.randint(0, 1024, (B,), generator=g) / 1024
    kept = torch.where(x >= min_p * 8, x, 0.0).double()
    cum = kept.cumsum(1)
    wide = torch.zeros(B, n + 5, device=DEV)
    wide[:, 1: n + 1] = x.to(DEV) / 1024
    aligned = torch.zeros(B, (n + 3) // 4 * 4, device=DEV)
    aligned[:, :n] = x.to(DEV) / 1024
    for rows in (wide[:, 1: n + 1], aligned[:, :n]):
        ids = ops.sampling_from_probs(rows, u.to(DEV), 0, 1.0, min_p).cpu().long()
        target = u.double() * cum[:, -1]                # the product is rounded once to fp32
        assert (kept.gather(1, ids[:, None]) > 0).all()
        at = cum.gather(1, ids[:, None])[:, 0]
        assert (at * (1 + 2.0**-23) >= target).all()
        assert (((at - kept.gather(1, ids[:, None])[:, 0]) * (1 - 2.0**-23)) <= target).all()
        got = sk.top_p_renorm_probs(rows, 1.0).cpu().double()
        assert torch.allclose(got, x.double() / x.double().sum(1, keepdim=True), rtol=1e-6, atol=0)


def test_rows_without_mass():
    """All zeros, and values that are not numbers or negative beside one that is."""
    from sglang_security_amd import ops

    x = torch.zeros(3, 1000, device=DEV)
    x[1, 17] = 0.5
    x[2] = float("nan")
    x[2, ::2] = -1.0
    x[2, 400] = 0.25
    u = torch.full((3,), 0.5, device=DEV)
    k, p = torch.full((3,), 10, dtype=torch.int32, device=DEV), torch.full((3,), 0.9, device=DEV)
    for joint in (True, False):
        ids = ops.sampling_from_probs(x, u, k, p, 0.0, joint).tolist()
        assert ids == [999, 17, 400]


def test_rows_of_infinite_mass():
    """The k largest are found where masses say nothing."""
    import sglang_security_amd.sgl_kernel as sk

    x = (torch.arange(3000, device=DEV) % 997).float()[None] + 1
    x[0, 5] = float("inf")
    got = sk.top_k_renorm_probs(x, 20)
    assert torch.equal(torch.nan_to_num(got, nan=1.0)[0] != 0, x[0] == float("inf"))
    assert got[0].isnan().sum() == 1            # inf / inf; the other kept values over infinity are zeros


def test_one_block_and_several_agree():
    """A row alone (spread over sixteen blocks) and in a batch too large to spread give the same tokens and rows."""
    import sglang_security_amd.sgl_kernel as sk
    from sglang_security_amd import ops

    g = torch.Generator(device=DEV).manual_seed(3)
    x = torch.softmax(3 * torch.randn(1, 50257, device=DEV, generator=g), -1)
    many = x.repeat(600, 1)
    u = torch.rand(600, device=DEV, generator=g)
    for kw in (dict(top_k=40, top_p=0.9), dict(top_p=0.99), dict(top_k=500), dict(min_p=0.1), dict()):
        ids = ops.sampling_from_probs(many, u, **kw)
        assert torch.equal(ids[:50], torch.cat([ops.sampling_from_probs(x, u[i: i + 1], **kw) for i in range(50)]))
    assert torch.equal(sk.top_p_renorm_probs(many, 0.9)[7:8], sk.top_p_renorm_probs(x, 0.9))
    assert torch.equal(sk.top_k_renorm_probs(many, 77)[7:8], sk.top_k_renorm_probs(x, 77))


@pytest.mark.parametrize("B,n", [(6, 40000), (6, 128259), (64, 163843)])
def test_spread_rows_with_all_filters(B, n):
    """Rows of different filters in one call over several slices: none, one, two, with a min-p below and above their cut."""
    from sglang_security_amd import ops

    g = torch.Generator().manual_seed(n)
    x = _rows("peaked", n, g)
    x = x * 2.0 ** -math.ceil(math.log2(x.sum().item()))
    rows = [(0, 1.0, 0.25), (50, 1.0, 0.0), (0, 0.875, 0.0), (50, 0.75, 0.125), (1000, 0.875, 2.0 ** -12), (n, 0.5, 0.0)]
    rows = [rows[b % 6] for b in range(B)]
    kt = torch.tensor([r[0] for r in rows], dtype=torch.int32, device=DEV)
    pt, mt = (torch.tensor([r[i] for r in rows], device=DEV) for i in (1, 2))
    wide = torch.zeros(B, n + 5, device=DEV)
    wide[:, 1: n + 1] = x.float().to(DEV)
    aligned = torch.zeros(B, (n + 3) // 4 * 4, device=DEV)
    aligned[:, :n] = x.float().to(DEV)
    for rows_of in (wide[:, 1: n + 1], aligned[:, :n]):
        for u in (0.0, 0.3, 0.7, 0.999999):
            ids = ops.sampling_from_probs(rows_of, torch.full((B,), u, device=DEV), kt, pt, mt, True).cpu().long()
            again = ops.sampling_from_probs(rows_of, torch.full((B,), u, device=DEV), kt, pt, mt, True).cpu().long()
            assert torch.equal(ids, again)
            for b in range(6):
                k, p, m = rows[b]
                kept = torch.where(x >= max(_threshold(x, k, p, True), m * x.max().item()), x, 0.0)
                cum = kept.cumsum(0) / kept.sum()
                for i in ids[b::6].tolist():
                    assert kept[i] > 0 and cum[i] >= u - 1e-5 and (i == 0 or cum[i - 1] <= u + 1e-5)


@pytest.mark.parametrize("aligned", [True, False])
def test_spread_rows_of_special_values(aligned, monkeypatch):
    """Rows that are not all finite and positive, beside one that is, spread over several blocks and done by one block each."""
    import sglang_security_amd.sgl_kernel as sk
    from sglang_security_amd import ops

    n, inf, nan = 40003, float("inf"), float("nan")
    g = torch.Generator().manual_seed(5)
    x = _rows("peaked", n, g)
    x = x * 2.0 ** -math.ceil(math.log2(x.sum().item()))
    rows = x.float().repeat(10, 1)
    rows[1, ::3] = nan
    rows[2, ::3] = -rows[2, ::3]
    rows[3] = 0.0
    rows[4], rows[4, 31007] = 0.0, 1.0
    rows[5, 7] = inf
    rows[6, 39999:] = inf                       # several of infinite mass, in the last slice
    rows[7, ::2] = -0.0
    rows[8] = nan
    rows[8, 20001], rows[8, 20002] = 0.75, -inf
    rows[9] = rows[9] * 2.0 ** -130             # no mass to speak of: values down to the smallest there are
    B = len(rows)
    wide = torch.full((B, n + 5), nan, device=DEV)
    at = 0 if aligned else 1
    if aligned:
        wide = torch.full((B, (n + 3) // 4 * 4), nan, device=DEV)
    wide[:, at: at + n] = rows.to(DEV)
    rows = wide[:, at: at + n]
    kt = torch.tensor([50, 0, 1000, 7, 2, n, 300, 1, 10, 40], dtype=torch.int32, device=DEV)
    pt = torch.tensor([0.75, 0.875, 1.0, 0.5, 0.875, 0.875, 1.0, 0.9, 0.5, 0.75], device=DEV)
    mt = torch.tensor([0.0, 0.25, 0.0, 0.125, 0.0, 0.5, 0.0, 0.0, 0.25, 0.0], device=DEV)
    assert ops._filter_workspace(rows)[1] > 0

    def everything():
        got = []
        for u in (0.0, 0.4, 0.999):
            u = torch.full((B,), u, device=DEV)
            for kw in (dict(top_k=kt, top_p=pt, min_p=mt), dict(top_k=kt, top_p=pt), dict(top_k=30), dict(top_p=0.75), dict(min_p=0.25)):
                got.append(ops.sampling_from_probs(rows, u, **kw))
        return got + [sk.top_k_renorm_probs(rows, kt), sk.top_p_renorm_probs(rows, pt), sk.top_k_renorm_probs(rows, 30)]

    spread = everything()
    monkeypatch.setattr(ops, "_filter_workspace", lambda *a, **k: (None, 0))
    for got, want in zip(spread, everything()):
        torch.testing.assert_close(got, want, rtol=1e-6 if got.is_floating_point() else 0, atol=0, equal_nan=True)


@pytest.mark.parametrize("B,n", [(1, 32768), (1, 32772), (5, 32773), (3, 151936), (64, 128256)])
def test_spread_draws_without_a_selection(B, n, monkeypatch):
    """Rows just long enough to be spread without a top-k or top-p, with a min-p for none, all and some of them, against one
    block a row; and their renormalisation."""
    import sglang_security_amd.sgl_kernel as sk
    from sglang_security_amd import ops

    g = torch.Generator().manual_seed(n)
    rows = torch.stack([_rows("peaked", n, g) for _ in range(min(B, 3))])
    rows = (rows * 2.0 ** -math.ceil(math.log2(rows.sum(1).max().item()))).float().to(DEV).repeat(-(-B // 3), 1)[:B].contiguous()
    some = torch.tensor([(0.0, 0.25, 0.5)[b % 3] for b in range(B)], device=DEV)

    def everything():
        ids = [ops.sampling_from_probs(rows, torch.full((B,), u, device=DEV), min_p=m) for u in (0.0, 0.37, 0.99999) for m in (0.0, 0.25, some)]
        return ids + [sk.top_p_renorm_probs(rows, 1.0)]

    spread = everything()
    monkeypatch.setattr(ops, "_filter_workspace", lambda *a, **k: (None, 0))
    for got, want in zip(spread, everything()):
        torch.testing.assert_close(got, want, rtol=1e-6 if got.is_floating_point() else 0, atol=0)
