"""Tiles of 128, 160, 192 and 224 tokens: the rows of a launch that takes them have the bits the same rows have in a batch whose
tiles hold 256 (a height changes no sum), with the last tile full, one row over, one short, and holding a single row; cut along the
contraction they stay as close to the fp32 product as whole ones."""
import pytest
import torch

from oracle import lora as olora
from oracle import nf4 as onf4
from tests.helpers import make_gptq, randn
from tests.test_gpu_kernels import dev, gweight
from tests.test_gpu_nf4 import _prepared
from tests.test_gpu_split_tiles import _bwd_projs, _no_further

pytestmark = pytest.mark.gpu

HEIGHTS = (128, 160, 192, 224)


def _rows(tile_of, height, limit=4096):
    """Token counts that take tiles of `height`: around its first full tiles, and the largest below a batch of 256-token ones."""
    takes = [M for M in range(1, limit) if tile_of(M) == height]
    edges = [M for M in takes if M % height in (0, 1, height - 1)]
    return sorted({*takes[:1], *edges[:3], *edges[-2:], takes[-1]}) if takes else []


def _fwd_arr(projs):
    import fmsa_hip

    arr = (fmsa_hip.FwdProj * len(projs))()
    for q, p in zip(arr, projs):
        q.w = p["w"]
    return arr


def _fwd_projs(x, Ns, base, r, bias):
    import fmsa_hip

    M, K = x.shape
    projs, refs, keep, code = [], [], [], None
    for i, N in enumerate(Ns):
        if base == "nf4":
            _, parts, q = _prepared(N, K, 90 + i, 64)
            code = parts[2] if code is None else code
            w, dense = fmsa_hip.make_codebook_weight(parts[0], code, parts[1], 64), dev(onf4.dequant(q, "fp32").t().contiguous())
            keep.append(parts)
        else:
            parts = make_gptq(K, N, 64, seed=40 + i)
            w, dense = gweight(parts, interleaved=base == "interleaved"), dev(parts["dense"]).float()
            keep.append(parts)
        A, B = (dev(t.to(x.dtype)) for t in olora.make_lora(K, N, r, 50 + i))
        U = fmsa_hip.lora_down(x, A)
        b = dev(randn((N,), 60 + i, x.dtype, 0.1)) if bias else None
        projs.append({"w": w, "U": U, "B": B, "bias": b, "r": r, "s": 2.0})
        ref = x.float() @ dense + 2.0 * (U.float() @ B.float().t())
        refs.append(ref if b is None else ref + b.float())
    return projs, refs, keep


@pytest.mark.parametrize("base,dtype", [("gptq", torch.bfloat16), ("gptq", torch.float16), ("interleaved", torch.float16),
                                        ("nf4", torch.bfloat16), ("nf4", torch.float16)])
@pytest.mark.parametrize("Ns,swiglu,K,r,bias", [([3040, 512, 512], False, 320, 24, True), ([2016, 2016], True, 256, 16, False)])
def test_forward(Ns, swiglu, K, r, bias, base, dtype):
    import fmsa_hip

    mode = fmsa_hip.FWD_SWIGLU if swiglu else fmsa_hip.FWD_LINEAR
    x = dev(randn((4096, K), 1, dtype))
    projs, refs, keep = _fwd_projs(x, Ns, base, r, bias)
    arr = _fwd_arr(projs)
    tile_of = lambda M: fmsa_hip.lib().fmsa_gptq_lora_fwd_tile(arr, len(projs), M, mode)
    assert tile_of(4096) == 256
    full = fmsa_hip.gptq_lora_fwd(x, projs, mode)
    if swiglu:
        refs = refs + [torch.nn.functional.silu(refs[0]) * refs[1]]
    seen = set()
    for height in HEIGHTS:
        for M in _rows(tile_of, height):
            part = [dict(p, U=p["U"][:M]) for p in projs]
            whole = fmsa_hip.gptq_lora_fwd(x[:M], part, mode)
            assert all(torch.equal(a, b[:M]) for a, b in zip(whole, full)), (height, M)
            if M > 768:  # (below, the kernel for few tokens may be taken)
                for a, b, ref in zip(fmsa_hip.gptq_lora_fwd(x[:M], part, mode, split=True), whole, refs):
                    _no_further(a, b, ref[:M])
            seen.add(height)
    assert len(seen) >= 3, seen


@pytest.mark.parametrize("base", ["gptq", "nf4"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("swiglu,K,Ns,r", [(False, 4032, [256, 64], 24), (True, 4032, [320], 16)])
def test_input_gradient(swiglu, K, Ns, r, dtype, base):
    import fmsa_hip

    mode = fmsa_hip.BWD_SWIGLU if swiglu else fmsa_hip.BWD_LINEAR
    M_full = 4096
    mask = dev(randn((M_full, K), 9, dtype))
    mask[::5, ::3] = 0
    projs, ref, lora, keep = _bwd_projs(M_full, K, Ns, r, 0.5, dtype, mask, base)
    ref = ref + (mask != 0) * lora
    e, g = dev(randn((M_full, K), 7, dtype)), dev(randn((M_full, K), 8, dtype))
    arr = (fmsa_hip.BwdProj * len(projs))()
    for q, p in zip(arr, projs):
        q.w = p["w"]
        for name in ("nsz", "qweight_t", "scale_f32", "negzp_f16"):
            setattr(q, name, None if p.get(name) is None else p[name].data_ptr())
    tile_of = lambda M: fmsa_hip.lib().fmsa_gptq_lora_bwd_dx_tile(arr, len(projs), M, mode, fmsa_hip.act_enum(dtype))
    assert tile_of(M_full) == 256

    def run(M, split):
        part = [dict(p, dY=p["dY"][:M], T=p["T"][:M], mask_src=mask[:M]) for p in projs]
        if not swiglu:
            return [fmsa_hip.gptq_lora_bwd_dx(part, M, K, split=split)]
        eg = e[:M].clone(), g[:M].clone()
        return [fmsa_hip.gptq_lora_bwd_dx(part, M, K, mode, e=eg[0], g=eg[1], split=split), *eg]

    full = run(M_full, False)
    seen = set()
    for height in HEIGHTS:
        for M in _rows(tile_of, height):
            whole = run(M, False)
            assert all(torch.equal(a, b[:M]) for a, b in zip(whole, full)), (height, M)
            split = run(M, True)
            if not swiglu:
                _no_further(split[0], whole[0], ref[:M])
            else:
                assert torch.equal(split[0], whole[0])
            seen.add(height)
    assert len(seen) >= 3, seen
