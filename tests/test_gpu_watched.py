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


def _beyond(kind):
    """A composite native call one of whose products is beyond the sizes the GEMMs take, as a function."""
    from mdy_triton_amd._torch_glue import host
    fp8 = lambda *s: torch.zeros(s, device="cuda", dtype=torch.uint8).view(torch.float8_e4m3fn)
    f32, bf = lambda *s: torch.zeros(s, device="cuda"), lambda *s: torch.zeros(s, device="cuda", dtype=torch.bfloat16)
    h = host()
    if kind == "deep_backward":             # 65792 padded tokens: the weight gradient's contraction
        args = (bf(65537, 256), fp8(256, 65792), f32(2, 514), fp8(256, 256), f32(2, 2), 256, True, True, True)
        return lambda: h.deep_backward(*args)
    if kind == "official_backward":         # more than 2^20 tokens
        args = (bf(2 ** 20 + 1, 128), fp8(128, 2 ** 20 + 128), f32(128, 8193), fp8(128, 128), f32(1, 1), 0, True, True, True, None)
        return lambda: h.official_backward(*args)
    if kind == "deep_forward":              # more than 65536 input features
        args = (bf(8, 65792), bf(128, 65792), None, None, 0, True, True)
        return lambda: h.deep_forward(*args)
    args = (bf(8, 65664), bf(128, 65664), None, 0, True, True, True)
    return lambda: h.official_forward(*args)


@pytest.mark.parametrize("kind", ["deep_backward", "official_backward", "deep_forward", "official_forward"])
def test_native_call_that_is_left_to_the_wrapper_has_done_nothing(kind):
    call = _beyond(kind)
    count = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]
    before = count()
    assert call() is None
    assert count() == before
