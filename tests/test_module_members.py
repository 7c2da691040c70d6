"""How the fused operators look up a projection's members: what getattr gives, whatever holds them."""
from collections import OrderedDict

import pytest
import torch

from fms_acceleration_foak.fused_ops.unsloth_lora.utils import get_lora_parameters, member
from fms_acceleration_peft import LoraLinear


class _GathersOnAccess(OrderedDict):
    """A parameter dictionary that brings a partitioned parameter in when it is asked for by subscript."""

    def __getitem__(self, name):
        param = super().__getitem__(name)
        if getattr(param, "whole", None) is not None:
            param.data = param.whole
        return param


def _partition(module):
    gathers = _GathersOnAccess(module._parameters)
    module._parameters = gathers
    for param in filter(lambda p: p is not None, OrderedDict.values(gathers)):
        param.whole, param.data = param.data, torch.empty(0)


def test_partitioned_parameters_are_gathered():
    lin = LoraLinear(torch.nn.Linear(16, 24, bias=False), 8, 16.0)
    A, B = lin.lora_A["default"].weight.data.clone(), lin.lora_B["default"].weight.data.clone()
    for module in (lin.base_layer, lin.lora_A["default"], lin.lora_B["default"]):
        _partition(module)
    W, _, _, A_now, B_now, _, _ = get_lora_parameters(lin)
    assert W.shape == (24, 16) and torch.equal(A_now, A) and torch.equal(B_now, B)


@pytest.mark.parametrize("where", ["parameter", "buffer", "none", "attribute", "property", "missing"])
def test_member_is_getattr(where):
    class M(torch.nn.Module):
        if where == "property":
            weight = property(lambda self: 5)

    m = M()
    if where == "parameter":
        m.weight = torch.nn.Parameter(torch.ones(2))
    elif where == "buffer":
        m.register_buffer("weight", torch.ones(2))
    elif where == "none":
        m.register_parameter("weight", None)
    elif where == "attribute":  # set beside a parameter of the name, as wrappers that hand out views of flat storage do
        m.weight = torch.nn.Parameter(torch.ones(2))
        object.__setattr__(m, "weight", torch.zeros(2))
    if where == "missing":
        assert member(m, "_parameters", "weight", None) is None
        with pytest.raises(AttributeError):
            member(m, "_parameters", "weight")
        return
    for kind in ("_parameters", "_buffers", "_modules"):
        assert member(m, kind, "weight") is getattr(m, "weight")
