"""Int8Linear's host side, as far as it needs no GPU."""
import pytest
import torch

import triton_int8_amd as T
from triton_int8_amd import linear


@pytest.fixture
def used(monkeypatch):
    """The weight and the bias that a forward hands to the autograd function."""
    seen = []
    monkeypatch.setattr(linear.Int8LinearFunction, "apply", lambda x, weight, bias, *_: seen.append((weight, bias)))
    return seen


def test_parameters_that_something_stands_in_front_of(used):
    class Scaled(T.Int8Linear):
        scale = None
        weight = property(lambda self: self._parameters["weight"] * self.scale if self.scale else self.__getattr__("weight"))

    x = torch.zeros(2, 128)
    layer = T.Int8Linear(128, 128, bias=True)
    layer(x)
    assert used[-1][0] is layer._parameters["weight"] and used[-1][1] is layer._parameters["bias"]
    for name in ("weight", "bias"):
        other = torch.ones_like(layer._parameters[name], requires_grad=True)
        layer.__dict__[name] = other
        layer(x)
        assert used[-1][name == "bias"] is other
    derived = Scaled(128, 128)
    derived.scale = 3
    derived(x)
    assert torch.equal(used[-1][0], derived._parameters["weight"] * 3)
    held = T.Int8Linear(128, 128)
    weight = held._parameters.pop("weight")
    held.weight_orig, held.weight = weight, weight * 2
    held(x)
    assert used[-1][0] is held.__dict__["weight"]


def test_functional_call(used):
    layer = T.Int8Linear(128, 128, bias=True)
    given = {"weight": torch.ones(128, 128, requires_grad=True), "bias": torch.ones(128)}
    torch.func.functional_call(layer, given, torch.zeros(2, 128))
    assert used[-1][0] is given["weight"] and used[-1][1] is given["bias"]
