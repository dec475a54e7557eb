"""`Linear` multiplies with the weight and scale that its attributes name, however a program has come to name them (no GPU needed)."""
import pytest
import torch

import modular_amd as mx
from modular_amd import linear as linear_module


@pytest.fixture
def operands(monkeypatch):
    """what a forward pass hands to the matmul"""
    seen = {}

    def record(x, weight, weight_scale, input_scale, config):
        seen.update(weight=weight, weight_scale=weight_scale)
        return torch.zeros((x.shape[0], weight.shape[0]), dtype=torch.bfloat16)
    monkeypatch.setattr(linear_module, "quantized_matmul", record)
    return seen


def build(cls=mx.Linear):
    return cls(256, 128, mx.blockwise_fp8_config(), device="cpu")


def check(layer, operands):
    layer(torch.zeros((3, 256), dtype=torch.bfloat16))
    assert operands["weight"] is layer.weight and operands["weight_scale"] is layer.weight_scale


def test_the_buffers_as_built_and_replaced(operands):
    layer = build()
    check(layer, operands)
    layer.weight = torch.zeros((128, 256), dtype=torch.uint8).view(torch.float8_e4m3fn)
    check(layer, operands)
    del layer.weight_scale
    layer.weight_scale = torch.nn.Parameter(torch.ones(1, 2))
    check(layer, operands)


def test_an_attribute_of_the_object_hides_the_buffer(operands):
    layer = build()
    for name in ("weight", "weight_scale"):
        object.__setattr__(layer, name, layer._buffers[name].clone())
    assert layer.weight is not layer._buffers["weight"]
    check(layer, operands)


def test_a_subclass_with_a_property_or_a_look_up_of_its_own(operands):
    other = torch.zeros((128, 256), dtype=torch.uint8).view(torch.float8_e4m3fn)

    class Property(mx.Linear):
        @property
        def weight(self):
            return other

    class LookUp(mx.Linear):
        def __getattr__(self, name):
            return other if name == "weight" else super().__getattr__(name)

    for cls in (Property, LookUp):
        layer = build(mx.Linear)
        layer.__class__ = cls  # (built with the buffers in place, as torch's own parametrisation leaves a module)
        check(layer, operands)
        assert operands["weight"] is other
