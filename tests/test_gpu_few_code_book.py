"""The kernel for few tokens on code-book weights, entry by entry: rows of the unit matrix bring out every weight as it was rounded, from
one book and from two in a launch, in each of the kernel's shapes."""
import pytest
import torch

from tests.test_gpu_few_tokens import _packed
from tests.test_gpu_nf4 import _prepared

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize("two_books", [False, True])
@pytest.mark.parametrize("M", [1, 16, 17, 33, 64, 65, 200])
def test_every_entry(M, two_books, swiglu, dtype):
    import fmsa_hip

    K, Ns = 576, (96, 96) if swiglu else (96, 32, 64)  # nine chunks for eight waves
    projs, dense, keep = [], [], []
    for i, N in enumerate(Ns):
        _, (words, scales, code), _ = _prepared(N, K, 40 + i, 64)
        if two_books and i == 1:
            code = (0.75 * code.flip(0)).contiguous()
        elif keep:
            code = keep[0][2]
        w = fmsa_hip.make_codebook_weight(words, code, scales, 64)
        keep.append((words, scales, code))
        projs.append({"w": w, "U": None, "B": None, "bias": None, "r": 0, "s": 0.0})
        dense.append(fmsa_hip.weight_dequant(w, torch.device("cuda"), dtype))  # [K, N], each weight rounded once
    mode = fmsa_hip.FWD_SWIGLU if swiglu else fmsa_hip.FWD_LINEAR
    for k0 in range(0, K, max(M, 64)):
        rows = (k0 + torch.arange(M, device="cuda")) % K
        x = torch.nn.functional.one_hot(rows, K).to(dtype)
        for y, W in zip(_packed(x, projs, mode), dense):
            assert torch.equal(y, W[rows])
