"""MDY_FP8_CHECK_WEIGHT_CACHE: a kept weight that changed through .data is found out, on the layer alone and inside an MLP; "0" and nothing are off."""
import pytest
import torch

import mdy_triton_amd as m

pytestmark = pytest.mark.gpu
NAME = "MDY_FP8_CHECK_WEIGHT_CACHE"


def _layers():
    """(what is called, the layer whose weight changes)"""
    lin = m.DeepLinear(256, 128, bias=False, dtype=torch.bfloat16, device="cuda")
    up, down = (m.Fp8MLP(256, 256, device="cuda", dialect="deeplinear", fp8_dtype=torch.float8_e4m3fn) for _ in range(2))
    for layer in (lin, up.up_gate_proj, up.down_proj, down.up_gate_proj, down.down_proj):
        layer.cache_weight = True
    return (lin, lin), (up, up.up_gate_proj), (down, down.down_proj)


@pytest.mark.parametrize("value,on", [("1", True), ("yes", True), ("00", True), ("0", False), ("", False), (None, False)])
@pytest.mark.parametrize("grad", [False, True])
def test_environment_asks_for_the_check(monkeypatch, value, on, grad):
    x = torch.randn(8, 256, device="cuda").bfloat16().requires_grad_(grad)
    monkeypatch.delenv(NAME, raising=False) if value is None else monkeypatch.setenv(NAME, value)
    with torch.set_grad_enabled(grad):
        for layer, owner in _layers():
            y = layer(x)
            assert torch.equal(layer(x), y)
            owner.weight.data.mul_(2)
            if on:
                with pytest.raises(RuntimeError, match="invalidate_weight_cache"):
                    layer(x)
            else:
                assert torch.equal(layer(x), y)      # the kept copy, as documented


def test_the_check_can_be_switched_while_a_weight_is_kept(monkeypatch):
    x = torch.randn(8, 256, device="cuda").bfloat16()
    with torch.no_grad():
        for layer, owner in _layers():
            monkeypatch.setenv(NAME, "1")
            y = layer(x)
            owner.weight.data.mul_(2)
            for off in ("0", ""):
                monkeypatch.setenv(NAME, off)
                assert torch.equal(layer(x), y)
                monkeypatch.setenv(NAME, "1")
                with pytest.raises(RuntimeError, match="invalidate_weight_cache"):
                    layer(x)
