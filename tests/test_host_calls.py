"""What the tensor-level calls refuse before they look for a GPU: operands that are not what the kernels would read them as."""
import pytest
import torch

import fmsa_hip


def _t(*shape):
    return torch.zeros(shape, dtype=torch.bfloat16)


def _pack(A):
    return fmsa_hip.lora_pack_batch([(A, _t(32, 16), None)], torch.bfloat16)


def _grad(Wt, T):
    return fmsa_hip.lora_grad_batch([(_t(4, 16), _t(4, 64), 1.0, False, torch.float32, Wt, T)])


@pytest.mark.parametrize("call", [
    lambda: fmsa_hip.lora_down(_t(4, 64, 1).as_strided((4, 64, 2), (64, 1, 0)), _t(16, 64)),
    lambda: fmsa_hip.lora_down_batch([(_t(4, 64, 1).as_strided((4, 64, 2), (64, 1, 0)), _t(16, 64), None)] * 2),
    lambda: fmsa_hip.lora_down_batch([(_t(4, 64), _t(16, 64, 2), None)] * 2),
    lambda: _pack(_t(16, 64, 2)),
    lambda: _grad(_t(16, 64, 1), _t(4, 16)),
    lambda: _grad(_t(16, 64), _t(4, 16, 1).as_strided((4, 16, 2), (16, 1, 0))),
], ids=["down, x", "down batch, x", "down batch, Wd", "pack, A", "gradient, Wt", "gradient, T"])
def test_operands_that_are_no_matrices(call):
    with pytest.raises(AssertionError):
        call()
