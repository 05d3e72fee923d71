"""Which fp8 weights get a second copy in the streaming layout: one rule, for the linear method and the decode runner."""
import pytest
import torch

from sglang_security_amd import ops

F8 = torch.float8_e4m3fn


@pytest.fixture
def repacked(monkeypatch):
    made = []
    monkeypatch.setattr(ops, "fp8_repack", lambda w: made.append(w) or w)
    return made


@pytest.mark.parametrize("K", [256, 384, 512, 3584, 4096])
@pytest.mark.parametrize("N", [16, 24])
def test_linear_method_and_runner_agree(repacked, K, N):
    from sglang_security_amd.decode_runner import _Fp8Linear
    from sglang_security_amd.quantization import W8A8Fp8Config, W8A8Fp8LinearMethod

    def layer_of(**kw):
        method = W8A8Fp8LinearMethod(W8A8Fp8Config(is_checkpoint_fp8_serialized=True), **kw)
        layer = torch.nn.Module()
        method.create_weights(layer, K, [N], K, N, torch.bfloat16)
        method.process_weights_after_loading(layer)
        return layer

    for rows in (1, 64, 65, None):
        streams = N % 16 == 0 and K >= (512 if rows in (1, 64) else 4096)
        assert ops.fp8_streams(N, K, rows) == streams
        layer = layer_of()
        held = layer.sglk_packed if rows not in (1, 64) or layer.sglk_packed is not None else layer.sglk_packed_short
        assert (held is not None) == streams
    # the decode runner: none for short inner dimensions, whatever its batch
    lin = _Fp8Linear(K, N, torch.bfloat16, "cpu", torch.Generator().manual_seed(0)).pack()
    assert (lin.wpacked is not None) == ops.fp8_streams(N, K)
    # a caller that would rather have the memory: no copy below 4096, the others as before
    repacked.clear()
    layer = layer_of(streaming_short_k=False)
    assert layer.sglk_packed_short is None and len(repacked) == int(ops.fp8_streams(N, K))
