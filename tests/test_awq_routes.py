"""CPU: which int4 products of many rows go where -- the tiles a plan cuts, and the rows that only the library takes."""
from types import SimpleNamespace

import pytest
import torch

from sglang_security_amd import ops
from sglang_security_amd._lib import SglkError
from sglang_security_amd.quantization.awq import AWQLinearMethod


@pytest.mark.parametrize("gated", [False, True])
def test_tiles_cover_a_product_once(gated):
    """Every row and column lies in one tile, and no tile lies outside; strips of 192 columns that do not divide the rest occur."""
    ragged = 0
    for K in (128, 512, 4096):
        for N in (256, 1024, 2560, 4096, 5120, 6144, 6656, 6784, 7168, 8192, 22016, 27648, 28672):
            for M in (1, 63, 64, 129, 300, 627, 819, 1152, 1600, 2112, 3200, 3700):
                rows, row_tiles, whole, tail, narrow = ops.awq_gemm_prefill_tiles(M, N, K, gated)
                assert rows in (128, 192, 256) and (row_tiles - 1) * rows < M <= row_tiles * rows
                rest = N - 256 * whole
                if tail:
                    assert narrow in ((128,) if gated else (128, 192)) and (tail - 1) * narrow < rest <= tail * narrow
                    ragged += rest % narrow != 0
                else:
                    assert -256 < rest <= 0
    assert gated or ragged > 20


def test_rules_of_many_rows_stay_where_they_were_measured():
    """Sizes that were timed with the library ahead by 5 % or more are the library's, and those with this package's product ahead by as much its."""
    library = [(8192, 14336, 4096), (8192, 4096, 28672), (4096, 4096, 28672), (3000, 8192, 10240), (4096, 13824, 5120), (2500, 3072, 8192),
               (500, 14336, 4096), (1152, 8192, 7168), (800, 4096, 6144), (1300, 11008, 4096), (640, 14336, 4096), (100, 8192, 8192),
               (1, 28672, 8192), (64, 8192, 10240)]
    here = [(257, 4096, 28672), (500, 4096, 28672), (1152, 4096, 28672), (257, 2560, 13824), (500, 5120, 15360), (384, 28672, 8192),
            (257, 1024, 8192), (500, 1536, 8960), (500, 8192, 57344), (800, 1024, 8192), (64, 4096, 28672), (200, 2560, 13824)]
    assert not any(ops.awq_prefill_fused(m, n, k) for m, k, n in library)
    assert all(ops.awq_prefill_fused(m, n, k) for m, k, n in here)
    gated = [(257, 4096, 28672), (1700, 4096, 28672), (1300, 5120, 27648), (2048, 8192, 57344)]
    assert all(ops.awq_prefill_fused(m, n, k, True) for m, k, n in gated)
    assert not any(ops.awq_prefill_fused(m, n, k, True) for m, k, n in [(4096, 4096, 28672), (8192, 3072, 16384), (1152, 8192, 7168)])


def test_blocks_of_96_and_128_rows_stay_where_they_were_measured():
    """Sizes that were timed with the wide kernel ahead by 5 % or more are its, whoever forms the block sums (fp16 and up to 64 rows always)."""
    rows = ops.awq_gemm_tall_rows
    wide = [(80, 13824, 5120), (255, 26624, 12160), (128, 4096, 6144), (128, 14336, 4096)]
    here = [(96, 4096, 28672), (128, 4096, 28672), (192, 5120, 15360), (96, 8192, 10240), (192, 28672, 8192), (97, 1536, 16640)]
    for sums in (False, True):
        assert not any(rows(m, n, k, sums=sums) for m, k, n in wide)
        assert all(rows(m, n, k, sums=sums) for m, k, n in here)
    assert not rows(128, 28672, 4096, dtype=torch.float16) and not rows(64, 28672, 4096) and not rows(128, 28672, 4096, group=256)


def _layer(k, n, dtype):
    return SimpleNamespace(sglk_shape=(k, n), scales=torch.ones(k // 128, n, dtype=dtype))


def test_rows_that_start_off_16_bytes_are_the_librarys():
    layer, flat = _layer(256, 128, torch.bfloat16), torch.randn(4 * 256 + 8).to(torch.bfloat16)
    rows = flat[8:].view(4, 256)
    assert AWQLinearMethod._kernel_rows(layer, rows) is rows
    assert AWQLinearMethod._kernel_rows(layer, flat[1: 1 + 4 * 256].view(4, 256)) is None
    copied = AWQLinearMethod._kernel_rows(layer, flat[1: 1 + 4 * 256].view(256, 4).t())   # a copy of its own is in place
    assert copied.is_contiguous() and copied.data_ptr() % 16 == 0
    one = flat[: 2 * 260].as_strided((1, 256), (260 + 1, 1))
    assert one.is_contiguous() and AWQLinearMethod._kernel_rows(layer, one) is None       # a pitch off 16 bytes


def test_rows_of_another_type_or_length_are_the_librarys():
    """(which refuses them)"""
    layer = _layer(256, 128, torch.bfloat16)
    for rows in (torch.randn(4, 256).half(), torch.randn(4, 256), torch.randn(4, 512).to(torch.bfloat16)):
        assert AWQLinearMethod._kernel_rows(layer, rows) is None


def test_rows_that_autograd_or_a_transform_looks_at_are_the_librarys():
    layer, x = _layer(256, 128, torch.float32), torch.randn(4, 256)
    taken = lambda t: AWQLinearMethod._kernel_rows(layer, t) is not None
    assert taken(x)
    with_grad = x.clone().requires_grad_()
    assert not taken(with_grad) and not taken(with_grad * 2)
    with torch.no_grad():
        assert taken(with_grad)
    with torch.autograd.forward_ad.dual_level():
        assert not taken(torch.autograd.forward_ad.make_dual(x, x))
    seen = []
    torch.vmap(lambda t: (seen.append(taken(t)), t)[1])(x[None])
    torch.jit.trace(lambda t: (seen.append(taken(t)), t + 1)[1], x, check_trace=False)
    assert seen and not any(seen)
    assert not taken(x.as_subclass(type("Own", (torch.Tensor,), {})))


def test_a_weight_of_another_type_or_shape_is_refused():
    """The kernel would read scales as the rows' type and words for the rows' length."""
    w = lambda k, n: (torch.zeros(k, n // 8, dtype=torch.int32), torch.ones(k // 128, n, dtype=torch.bfloat16),
                      torch.zeros(k // 128, n // 8, dtype=torch.int32))
    rows = torch.zeros(3, 256, dtype=torch.bfloat16)
    assert ops._packed_weight("product", rows, *w(256, 128)) == (3, 128, 256)
    packed, scales, zeros = w(256, 128)
    for args in ((rows.half(), packed, scales, zeros), (torch.zeros(3, 512, dtype=torch.bfloat16), packed, scales, zeros),
                 (rows, packed[:, :8], scales, zeros), (rows, packed, scales, zeros[:1])):
        with pytest.raises(SglkError):
            ops._packed_weight("product", *args)


@pytest.mark.parametrize("T", [256, 300, 700, 1152, 1600, 1900, 2112, 2500])
def test_dequantisation_pipeline_holds_what_the_layers_ask_of_it(monkeypatch, T):
    """Projections dequantised ahead are those, in that order, that the layers then multiply by the library: where gate_up takes its
    activation along, on the rule of its own, it is not among them."""
    from sglang_security_amd.decode_runner import _AwqLinear
    from sglang_security_amd.prefill_runner import LlamaPrefill

    def weight(K, N):
        w = _AwqLinear.__new__(_AwqLinear)
        w.K, w.N, w.packed, w.scales, w.qzeros = K, N, None, torch.empty(K // 128, 0), None
        return w

    layers = [{"qkv": weight(4096, 6144), "o": weight(4096, 4096), "gate_up": weight(4096, 28672), "down": weight(14336, 4096),
               "gate_up_il": (None, None, None)} for _ in range(2)]
    model = LlamaPrefill.__new__(LlamaPrefill)
    model.prefill_gemm, model.resident_bf16, model.overlap_dequant, model._pipe = "library", False, True, None
    model.cfg = SimpleNamespace(quant="awq")
    model.dec = SimpleNamespace(layers=layers, device=torch.device("cpu"), dtype=torch.bfloat16)
    model._ring, model._side = [], SimpleNamespace(wait_stream=lambda s: None)
    asked = []
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: None)
    monkeypatch.setattr(ops, "awq_gemm_prefill", lambda *a: None)
    monkeypatch.setattr(LlamaPrefill, "_pipe_issue", lambda self, j: None)
    monkeypatch.setattr(LlamaPrefill, "_pipe_matmul", lambda self, w, x, out: asked.append(w))
    monkeypatch.setattr(ops, "awq_dequantize_packed_nk", lambda *a: pytest.fail("dequantised outside the pipeline"))
    model._pipe_begin(T)
    for L in layers:
        for k in ("qkv", "o", "gate_up", "down"):
            if k != "gate_up" or not model._gated(L, T):
                model._linear(L[k], torch.empty(T, L[k].K, device="meta"), None)
    assert model._gated(layers[0], T) == (T <= 2112)
    assert asked and [id(w) for w in asked] == [id(w) for w in model._seq]
