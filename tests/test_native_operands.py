"""What native code reads of an adapted projection: what the Python look-ups give, or None where the projection is no ordinary one."""
import pytest
import torch

import fmsa_hip
from fms_acceleration_foak.fused_ops.unsloth_lora.gptq import fast_lora
from fms_acceleration_peft import LoraLinear
from tests.model_utils import make_lora_gptq_linear
from tests.test_module_members import _partition


def _python(lin):
    qstate, bias, *adapter = fast_lora.get_lora_parameters(lin)
    return (*fast_lora.unpack_gptqstate(qstate), bias, *adapter)


def _same(a, b):
    return len(a) == len(b) and all(x is y or (not isinstance(x, torch.Tensor) and x == y) for x, y in zip(a, b))


class _Peft(torch.nn.Module):
    """A layer with attributes only: one active adapter of two."""

    def __init__(self, lin):
        super().__init__()
        self.base_layer, self.merged, self.disable_adapters, self.active_adapter = lin.base_layer, False, False, "b"
        self.lora_A = torch.nn.ModuleDict({"a": torch.nn.Linear(256, 8, bias=False), "b": torch.nn.Linear(256, 16, bias=False)})
        self.lora_B = torch.nn.ModuleDict({"a": torch.nn.Linear(8, 128, bias=False), "b": torch.nn.Linear(16, 128, bias=False)})
        self.scaling = {"a": 1, "b": 3}
        self.lora_dropout = torch.nn.ModuleDict({"a": torch.nn.Identity(), "b": torch.nn.Identity()})


@pytest.mark.parametrize("form", ["plain", "bias", "zero_bias", "dropout", "peft", "partitioned", "wrapped"])
def test_operands_are_those_of_the_python_look_ups(form):
    lin = make_lora_gptq_linear(256, 128, 8, 16.0, seed=1, bias="bias" in form, dropout=torch.nn.Dropout(0.1) if form == "dropout" else None)[0]
    if form == "zero_bias":
        lin.base_layer.bias.zero_()
    if form == "peft":
        lin = _Peft(lin)
    if form == "partitioned":
        for module in (lin.lora_A["default"], lin.lora_B["default"]):
            _partition(module)
    if form == "wrapped":  # a base layer of a base layer
        lin = LoraLinear(lin.base_layer, 8, 16.0)
        lin.base_layer = torch.nn.ModuleDict({"base_layer": lin.base_layer})
        lin.base_layer.base_layer = lin.base_layer["base_layer"]
    expected = _python(lin)  # (and whether the bias is zero is known now)
    assert _same(fmsa_hip.native().gptq_operands(lin), expected) and _same(fast_lora._operands(lin), expected)


@pytest.mark.parametrize("form", ["disabled", "merged", "bare", "new_bias", "auto_gptq"])
def test_other_projections_are_left_to_them(form):
    lin = make_lora_gptq_linear(256, 128, 8, 16.0, seed=1, bias=form == "new_bias")[0]
    if form == "disabled":
        lin.enable_adapters(False)
    if form == "merged":
        lin.merged_adapters.append("default")
    if form == "bare":
        lin = lin.base_layer
    if form == "auto_gptq":
        lin.base_layer.__class__ = type("QuantLinear", (type(lin.base_layer),), {"__module__": "auto_gptq.nn_modules"})
    if form == "new_bias":
        _python(lin)
        lin.base_layer.bias.mul_(0)  # a version that nobody has looked at
    assert fmsa_hip.native().gptq_operands(lin) is None
    assert _same(fast_lora._operands(lin), _python(lin))
    if form == "auto_gptq":
        assert lin.base_layer.qzeros.offset == 1


def test_a_prepared_weight_is_known_by_its_key():
    lin = make_lora_gptq_linear(256, 128, 8, 16.0, seed=1)[0].base_layer
    parts = lin.qweight, lin.scales, lin.qzeros, lin.g_idx
    known = lambda: fmsa_hip.native().gptq_prepared(*parts)

    def key():
        q, s, z, g = parts
        return (q.data_ptr(), s.data_ptr(), z.data_ptr(), g.data_ptr(), g._version, q._version, s._version, z._version,
                int(getattr(z, "offset", 0) or 0))

    assert known() is None
    for change in (lambda: None, lambda: lin.scales.mul_(2), lambda: setattr(lin.qzeros, "offset", 1), lambda: lin.g_idx.add_(0)):
        change()
        assert known() is None
        lin.qweight._fmsa_prepared = (key(), marker := object())
        assert known() is marker
    parts = lin.qweight, lin.scales.clone(), lin.qzeros, lin.g_idx
    assert known() is None
