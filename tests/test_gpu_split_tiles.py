"""The contraction split of launches whose tiles do not fill the chip: against the fp32 product, next to the same call
without the split.  Only the order of the fp32 sums differs, so the distance from the reference must not grow beyond what a
handful of other roundings can do (2 %), and the ranges are added in a fixed order, so every run gives the same bits."""
import pytest
import torch

from oracle import lora as olora
from tests.helpers import make_gptq, randn
from tests.test_gpu_kernels import _proj_bwd, dev, gweight

pytestmark = pytest.mark.gpu


def _no_further(split, whole, ref):
    err, base = (split.float() - ref).norm(), (whole.float() - ref).norm()
    assert err <= 1.02 * base, (float(err), float(base))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,Ns,swiglu,interleaved", [
    (1, 4096, [1024], False, False),           # one token, one tile row
    (300, 2080, [2048, 512, 288], False, False),  # three projections, ragged last tile, K ends in half a stage
    (257, 2048, [512], False, True),
    (520, 2048, [14336, 14336], True, False),  # 336 tiles: one whole round, 80 cut
    (64, 1280, [256, 256], True, True),
])
def test_forward(M, K, Ns, swiglu, interleaved, dtype):
    import fmsa_hip

    if interleaved and dtype != torch.float16:
        pytest.skip("the interleaved copy is read for fp16 activations")
    gs, r, s = 128, 16, 2.0  # (a group may be cut short by the end of K)
    x = dev(randn((M, K), 1, dtype))
    projs, refs, keep = [], [], []
    for i, N in enumerate(Ns):
        w = make_gptq(K, N, gs, seed=40 + i)
        A, B = (dev(t.to(dtype)) for t in olora.make_lora(K, N, r, 50 + i))
        U = fmsa_hip.lora_down(x, A)
        keep.append((w, A, B))
        projs.append({"w": gweight(w, interleaved=interleaved), "U": U, "B": B, "bias": None, "r": r, "s": s})
        refs.append(x.float() @ dev(w["dense"]).float() + s * (U.float() @ B.float().t()))
    mode = fmsa_hip.FWD_SWIGLU if swiglu else fmsa_hip.FWD_LINEAR
    whole = fmsa_hip.gptq_lora_fwd(x, projs, mode)
    split = fmsa_hip.gptq_lora_fwd(x, projs, mode, split=True)
    again = fmsa_hip.gptq_lora_fwd(x, projs, mode, split=True)
    if swiglu:
        refs.append(torch.nn.functional.silu(refs[0]) * refs[1])
    for a, b, c, ref in zip(split, whole, again, refs):
        _no_further(a, b, ref)
        assert torch.equal(a, c)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,Ns", [
    (1, 256, [2048]),
    (300, 1152, [1024, 256, 1056]),  # ranges that begin and end inside a projection; N ends in half a stage
    (513, 14336, [2048]),            # 168 tiles: too many to cut
    (1030, 14336, [2048]),           # 280 tiles: one whole round, 24 cut
])
def test_input_gradient(M, K, Ns, dtype):
    import fmsa_hip

    r, s = 24, 0.5
    x = dev(randn((M, K), 2, dtype))
    x[::3, ::5] = 0
    projs, ref, keep = [], 0.0, []
    for i, N in enumerate(Ns):
        w = make_gptq(K, N, 64, seed=60 + i)
        keep.append(w)
        A, B = olora.make_lora(K, N, r, 70 + i)
        dy = dev(randn((M, N), 80 + i, dtype))
        p = _proj_bwd(w, dy, A, B, s, dtype, mask_src=x, twin=True)
        projs.append(p)
        ref = ref + dy.float() @ dev(w["dense"]).float().t() + (x != 0) * (s * (p["T"].float() @ dev(A.to(dtype)).float()))
    whole = fmsa_hip.gptq_lora_bwd_dx(projs, M, K)
    split = fmsa_hip.gptq_lora_bwd_dx(projs, M, K, split=True)
    _no_further(split, whole, ref)
    assert torch.equal(split, fmsa_hip.gptq_lora_bwd_dx(projs, M, K, split=True))
