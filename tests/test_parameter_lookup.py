"""The layers compute with module.weight and module.bias, whatever these mean: a parameter, a subclass's property over it, an attribute of the instance,
a lookup of the class's own, a parametrization - also where that changes between two calls."""
import pytest
import torch

import mdy_triton_amd as m
from mdy_triton_amd import _torch_glue
from mdy_triton_amd._torch_glue import parameter_of


class Masked(m.DeepLinear):
    """The registered parameter under a mask."""

    @property
    def weight(self):
        return self._parameters["weight"] * self.mask


class Looked(m.DeepLinear):
    def __getattr__(self, name):
        return super().__getattr__("_other" if name == "weight" else name)


class Watched(m.DeepLinear):
    def __getattribute__(self, name):
        return super().__getattribute__("_parameters")["_other"] if name == "weight" else super().__getattribute__(name)


def _own(layer):
    return layer


def _masked(layer):
    layer.mask = torch.zeros((), device=layer.weight.device, dtype=layer.weight.dtype)
    layer.__class__ = Masked
    return layer


def _in_the_instance(layer):
    object.__setattr__(layer, "weight", torch.zeros_like(layer.weight))
    return layer


def _lookup_of_the_class(layer, cls=Looked):
    layer.register_parameter("_other", torch.nn.Parameter(torch.zeros_like(layer.weight)))
    layer.__class__ = cls
    return layer


def _parametrized(layer):
    class Zero(torch.nn.Module):
        def forward(self, w):
            return w * 0

    torch.nn.utils.parametrize.register_parametrization(layer, "weight", Zero())
    return layer


def _deleted(layer):
    value = torch.zeros_like(layer.weight)
    del layer.weight
    layer.weight = value
    return layer


FORMS = [_own, _masked, _in_the_instance, _lookup_of_the_class, lambda l: _lookup_of_the_class(l, Watched), _parametrized, _deleted]
IDS = ["own", "property", "instance", "__getattr__", "__getattribute__", "parametrization", "plain tensor"]


class Ordered(dict):
    def __getitem__(self, name):
        return "gathered " + name


@pytest.mark.parametrize("built", [True, False])
@pytest.mark.parametrize("form", FORMS, ids=IDS)
def test_is_the_attribute(form, built, monkeypatch):
    if not built:
        monkeypatch.setattr(_torch_glue, "_host", _torch_glue._NoHost())
    layer = m.DeepLinear(8, 4, bias=False)
    assert parameter_of(layer, "weight") is layer.weight and parameter_of(layer, "bias") is None
    layer = form(layer)
    assert torch.equal(parameter_of(layer, "weight"), layer.weight) and (form is _own or not layer.weight.any())
    assert parameter_of(layer, "bias") is None
    with pytest.raises(AttributeError, match="nothing"):
        parameter_of(layer, "nothing")


def test_is_the_attribute_when_the_class_changes():
    class Later(m.DeepLinear):
        pass

    layer = Later(8, 4)
    assert parameter_of(layer, "weight") is layer._parameters["weight"]
    Later.weight = property(lambda self: "a property")
    assert parameter_of(layer, "weight") == "a property"
    del Later.weight
    assert parameter_of(layer, "weight") is layer._parameters["weight"]
    layer._parameters = Ordered(layer._parameters)
    assert parameter_of(layer, "weight") == layer.weight == "gathered weight"


@pytest.mark.gpu
@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("form", FORMS, ids=IDS)
def test_layers_multiply_by_it(form, grad):
    x = torch.randn(4, 256, device="cuda").bfloat16()
    layer = m.DeepLinear(256, 256, bias=False, device="cuda", dtype=torch.bfloat16)
    with torch.set_grad_enabled(grad):
        layer(x)
        assert bool(form(layer)(x).any()) == (form is _own)
        for name in ("up_gate_proj", "down_proj"):
            mlp = m.Fp8MLP(256, 256, device="cuda", dialect="deeplinear", fp8_dtype=torch.float8_e4m3fn)
            mlp(x)
            form(getattr(mlp, name))
            assert bool(mlp(x).any()) == (form is _own)
