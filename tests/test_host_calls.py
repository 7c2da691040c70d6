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


def _few(x=None, A=None, B=None, bias=None, K=4096, N=4096):
    """lora_few on a weight that is described only: nothing is read before the refusal."""
    w = fmsa_hip.GptqWeight(0x1000, 0x1000, 0x1000, None, K, N, 128, 0, fmsa_hip.WEIGHT_AFFINE, 0, None, None)
    x = _t(4, K) if x is None else x
    A, B = torch.zeros(16, K) if A is None else A, torch.zeros(N, 16) if B is None else B
    return fmsa_hip.lora_few(x, [(w, A, B, bias, 2.0)])


@pytest.mark.parametrize("kw", [
    {"x": _t(4, 2048)}, {"x": _t(4, 8192)[:, ::2]},
    {"A": torch.zeros(16, 4096, dtype=torch.bfloat16)}, {"B": torch.zeros(4096, 16, dtype=torch.bfloat16)},
    {"A": torch.zeros(4096, 16).t()}, {"B": torch.zeros(16, 4096).t()}, {"A": torch.zeros(16, 4096, 1)}, {"B": torch.zeros(4096, 16, 1)},
    {"bias": torch.zeros(4096)}, {"bias": _t(4095)}, {"bias": _t(8192)[::2]},
], ids=["columns of x", "stride of x", "type of A", "type of B", "order of A", "order of B", "A", "B", "type of bias", "length of bias",
        "stride of bias"])
def test_lora_few_takes_what_its_kernels_read(kw):
    with pytest.raises(AssertionError):
        _few(**kw)


def test_lora_few_gets_as_far_as_the_gpu():
    with pytest.raises(RuntimeError, match="GPU"):
        _few(bias=_t(4096))
