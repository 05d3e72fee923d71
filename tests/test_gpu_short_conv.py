"""GPU: short causal convolutions of many rows against the same rows a few at a time, which carry their state from call to call."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _seqs(lens, starts, slots):
    from sglang_security_amd.ops_hybrid import RowSeqs

    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    row0 = [sum(lens[:i]) for i in range(len(lens))]
    return RowSeqs(i32([s for s, n in enumerate(lens) for _ in range(n)]), i32(row0), i32(lens), i32(starts), i32(slots))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("W,lens,starts", [
    (5120, [1, 1, 1500, 2, 1, 3, 7, 1801], [5, 0, 9, 1, 4, 0, 2, 0]),      # eight rows a thread; ends inside, at and across them
    (5120, [1] * 37 + [1500, 4, 1801], [i % 6 for i in range(40)]),         # single rows, which are no multiple of four
    (65536, [8, 8, 3, 5, 240, 1], [0, 3, 0, 7, 1, 2]),                       # just enough threads, as few rows
    (65528, [1, 255], [1, 1]),                                               # just too few: four rows a thread
    (64, [1, 2, 3, 4, 5, 250], [1, 2, 3, 0, 5, 6]),
    (64, [257], [0]),
])
@pytest.mark.parametrize("act", [0, 3])
def test_many_rows_and_few(dtype, W, lens, starts, act):
    from sglang_security_amd.ops_hybrid import Source, short_conv

    g = torch.Generator(device=DEV).manual_seed(W + len(lens))
    M, n = sum(lens), len(lens)
    src = torch.randn(M, W + 8, device=DEV, generator=g).to(dtype)[:, :W]
    if dtype == torch.float32:
        src = src.unsqueeze(0)      # fp32 rows are split sums of one split
    conv, bias, conv_b = (torch.randn(*s, device=DEV, generator=g) for s in ((4, W), (W,), (W,)))
    state = torch.randn(n, 3, W, device=DEV, generator=g).to(dtype)
    singles = next((i for i, k in enumerate(lens) if k > 1), n)
    got, held = torch.full((M, W), float("nan"), dtype=dtype, device=DEV), state.clone()
    slots = list(range(n))[::-1]
    short_conv(Source(src, dtype == torch.float32), conv, got, held, _seqs(lens, starts, slots), singles, act, bias, conv_b)
    want, carried, at = torch.empty_like(got), state.clone(), 0
    for k, start, slot in zip(lens, starts, slots):
        for lo in range(0, k, 200):
            m = min(200, k - lo)
            u = torch.empty(m, W, dtype=dtype, device=DEV)
            short_conv(Source(src[..., at + lo: at + lo + m, :], dtype == torch.float32), conv, u, carried, _seqs([m], [start + lo], [slot]), 0, act, bias, conv_b)
            want[at + lo: at + lo + m] = u
        at += k
    assert torch.equal(held, carried)
    if dtype == torch.float16 and act == 0:     # the last sum and its conversion may be one instruction: one rounding, or two
        assert ((got - want).abs() <= 2.0 ** -10 * want.abs() + 2.0 ** -24).all()
    else:
        assert torch.equal(got, want)
    # and the arithmetic itself, where a sequence starts: four products and two roundings to the type
    x = (src.reshape(M, W)[-lens[-1]:].float() + bias).to(dtype).double()
    front = torch.zeros(3, W, dtype=torch.double, device=DEV) if starts[-1] == 0 else state[slots[-1]].double()
    x = torch.cat([front, x])
    terms = [x[t: t + lens[-1]] * conv[t].double() for t in range(4)] + [conv_b.double()]
    z, size = sum(terms), sum(t.abs() for t in terms)
    z = torch.nn.functional.silu(z) if act == 3 else z
    # the result's rounding; four roundings of sums in 32 bits, at most `size` each, through a slope of at most 1.1; the exponential's
    eps = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -23}[dtype]
    assert ((got[-lens[-1]:].double() - z).abs() <= eps * z.abs() + 2.0 ** -21 * size + 2.0 ** -24).all()
