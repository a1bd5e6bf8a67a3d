"""Calls that something watches - a trace, a function transform, a forward-mode tangent, autograd's version check - go through
the operators' autograd functions, not past them."""
import warnings

import pytest
import torch

import mdy_triton_amd as m

pytestmark = pytest.mark.gpu


def _layer(kind):
    torch.manual_seed(0)
    if kind == "deep":
        return m.DeepLinear(256, 256, bias=True, device="cuda", dtype=torch.bfloat16)
    if kind == "fp8":
        return m.Fp8Linear(256, 256, bias=True, device="cuda", dtype=torch.bfloat16)
    return m.Fp8MLP(256, 256, device="cuda", dtype=torch.bfloat16, dialect=kind[4:], fp8_dtype=torch.float8_e4m3fn)


KINDS = ["deep", "fp8", "mlp_official", "mlp_deeplinear"]


@pytest.mark.parametrize("kind", KINDS)
def test_transforms_are_refused(kind):
    lin = _layer(kind)
    x = torch.randn(2, 16, 256, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        with pytest.raises(RuntimeError):
            torch.vmap(lin)(x)
        with torch.autograd.forward_ad.dual_level():
            with pytest.raises((RuntimeError, NotImplementedError)):
                lin(torch.autograd.forward_ad.make_dual(x[0], x[1]))


@pytest.mark.parametrize("kind", ["deep", "mlp_official", "mlp_deeplinear"])
def test_trace_keeps_the_call(kind):
    lin = _layer(kind)
    x, x2 = torch.randn(2, 16, 256, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad(), warnings.catch_warnings():
        warnings.simplefilter("ignore")
        traced = torch.jit.trace(lin, (x,), check_trace=False)
        assert any(n.kind() == "prim::PythonOp" for n in traced.inlined_graph.nodes())
        assert torch.equal(traced(x2), lin(x2))


@pytest.mark.parametrize("strided", [False, True])
@pytest.mark.parametrize("which", ["x", "w"])
def test_in_place_change_before_backward_is_refused(which, strided):
    lin = _layer("fp8")
    x = torch.randn(256, 32, device="cuda", dtype=torch.bfloat16).t() if strided else torch.randn(32, 256, device="cuda", dtype=torch.bfloat16)
    leaf = x.requires_grad_(True)
    y = leaf * 1
    out = lin(y)
    with torch.no_grad():
        (y if which == "x" else lin.weight).mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()
    out = lin(leaf * 1)
    out.sum().backward()
    assert leaf.grad is not None and lin.weight.grad is not None


def test_inference_tensor_is_refused_in_training():
    lin = _layer("fp8")
    with torch.inference_mode():
        x = torch.randn(32, 256, device="cuda", dtype=torch.bfloat16)
        assert lin(x).shape == (32, 256)
    with pytest.raises(RuntimeError, match="[Ii]nference"):
        lin(x)
