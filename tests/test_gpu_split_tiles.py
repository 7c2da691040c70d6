"""The contraction split of launches whose tiles do not fill the chip: against the fp32 product, next to the same call
without the split.  Only the order of the fp32 sums differs, so the distance from the reference must not grow beyond what a
handful of other roundings can do (2 %), and the ranges are added in a fixed order, so every run gives the same bits.
Every case says whether it is cut, and the rule is asked."""
import pytest
import torch

from oracle import lora as olora
from oracle import nf4 as onf4
from tests.helpers import make_gptq, randn
from tests.test_gpu_kernels import _proj_bwd, dev, gweight
from tests.test_gpu_nf4 import _prepared

pytestmark = pytest.mark.gpu


def _no_further(split, whole, ref):
    err, base = (split.float() - ref).norm(), (whole.float() - ref).norm()
    assert err <= 1.02 * base, (float(err), float(base))


def _fwd_cut(projs, M, mode):
    import fmsa_hip

    arr = (fmsa_hip.FwdProj * len(projs))()
    for i, p in enumerate(projs):
        arr[i].w = p["w"]
    return fmsa_hip.lib().fmsa_gptq_lora_fwd_workspace(arr, len(projs), M, mode) > 0


def _bwd_cut(projs, M, dtype):
    """(The larger of the two modes' needs.)"""
    import fmsa_hip

    arr = (fmsa_hip.BwdProj * len(projs))()
    for i, p in enumerate(projs):
        arr[i].w = p["w"]
        for name in ("nsz", "qweight_t", "scale_f32", "negzp_f16"):
            setattr(arr[i], name, None if p.get(name) is None else p[name].data_ptr())
    return fmsa_hip.lib().fmsa_gptq_lora_bwd_dx_workspace(arr, len(projs), M, fmsa_hip.act_enum(dtype)) > 0


def _adapter(K, N, r, seed, dtype):
    if r == 0:
        return None, None
    return tuple(dev(t.to(dtype)) for t in olora.make_lora(K, N, r, seed))


def _fwd_and_check(x, projs, refs, swiglu, cut):
    import fmsa_hip

    mode = fmsa_hip.FWD_SWIGLU if swiglu else fmsa_hip.FWD_LINEAR
    assert _fwd_cut(projs, x.shape[0], mode) == cut
    whole = fmsa_hip.gptq_lora_fwd(x, projs, mode)
    split = fmsa_hip.gptq_lora_fwd(x, projs, mode, split=True)
    again = fmsa_hip.gptq_lora_fwd(x, projs, mode, split=True)
    if swiglu:
        refs = refs + [torch.nn.functional.silu(refs[0]) * refs[1]]
    for a, b, c, ref in zip(split, whole, again, refs):
        _no_further(a, b, ref)
        assert torch.equal(a, c) and (cut or torch.equal(a, b))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,Ns,swiglu,interleaved,bias,r,cut", [
    (1, 4096, [1024], False, False, False, 16, True),           # one token, one tile row
    (300, 2080, [2048, 512, 288], False, False, False, 16, True),  # three projections, ragged last tile, K ends in half a stage
    (300, 2080, [2048, 512, 288], False, False, True, 0, True),    # biases, no adapters
    (257, 2048, [512], False, True, True, 64, True),
    (520, 2048, [14336, 14336], True, False, False, 16, False),  # 336 tiles: the 80 behind the whole round are not worth it
    (8300, 2048, [2048], False, False, True, 16, True),         # 264 tiles: one whole round, 8 cut
    (4200, 2048, [2048, 2048], True, False, True, 16, True),    # 272 tiles: one whole round, 16 cut
    (64, 1280, [256, 256], True, True, False, 16, True),
    (64, 1280, [256, 256], True, False, True, 16, True),
    (33, 1312, [288, 288], True, False, False, 0, True),
])
def test_forward(M, K, Ns, swiglu, interleaved, bias, r, cut, dtype):
    import fmsa_hip

    if interleaved and dtype != torch.float16:
        pytest.skip("the interleaved copy is read for fp16 activations")
    gs, s = 128, 2.0  # (a group may be cut short by the end of K)
    x = dev(randn((M, K), 1, dtype))
    projs, refs, keep = [], [], []
    for i, N in enumerate(Ns):
        w = make_gptq(K, N, gs, seed=40 + i)
        A, B = _adapter(K, N, r, 50 + i, dtype)
        U = fmsa_hip.lora_down(x, A) if r else None
        b = dev(randn((N,), 60 + i, dtype, 0.1)) if bias else None
        keep.append((w, A, B))
        projs.append({"w": gweight(w, interleaved=interleaved), "U": U, "B": B, "bias": b, "r": r, "s": s})
        ref = x.float() @ dev(w["dense"]).float()
        if r:
            ref = ref + s * (U.float() @ B.float().t())
        refs.append(ref if b is None else ref + b.float())
    _fwd_and_check(x, projs, refs, swiglu, cut)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,Ns,swiglu,blocksize,bias,r", [
    (300, 2176, [512], False, 64, True, 16),       # ranges of three and four stages
    (300, 2176, [512, 288], False, 128, False, 24),  # ranges that begin inside a block
    (40, 2176, [320, 320], True, 128, True, 8),
    (8300, 2048, [2048], False, 64, False, 16),    # one whole round, 8 tiles cut
])
def test_forward_code_book(M, K, Ns, swiglu, blocksize, bias, r, dtype):
    import fmsa_hip

    s = 2.0
    x = dev(randn((M, K), 3, dtype))
    projs, refs, keep = [], [], []
    code = None
    for i, N in enumerate(Ns):
        w, parts, q = _prepared(N, K, 90 + i, blocksize)
        code = parts[2] if code is None else code  # one code book for the launch
        w = fmsa_hip.make_codebook_weight(parts[0], code, parts[1], blocksize)
        A, B = _adapter(K, N, r, 50 + i, dtype)
        U = fmsa_hip.lora_down(x, A)
        b = dev(randn((N,), 60 + i, dtype, 0.1)) if bias else None
        keep.append((parts, A, B))
        projs.append({"w": w, "U": U, "B": B, "bias": b, "r": r, "s": s})
        ref = x.float() @ dev(onf4.dequant(q, "fp32").t().contiguous()) + s * (U.float() @ B.float().t())
        refs.append(ref if b is None else ref + b.float())
    _fwd_and_check(x, projs, refs, swiglu, True)


def _bwd_projs(M, K, Ns, r, s, dtype, mask, base, blocksize=64):
    """(operands on the twin, dX before the mask's part as fp32: base product and adapter product)"""
    import fmsa_hip

    projs, ref, lora, keep = [], 0.0, 0.0, []
    code = None
    for i, N in enumerate(Ns):
        dy = dev(randn((M, N), 80 + i, dtype))
        A, B = olora.make_lora(K, N, r or 8, 70 + i)
        if base == "gptq":
            w = make_gptq(K, N, 64, seed=60 + i)
            p = _proj_bwd(w, dy, A, B, s, dtype, mask_src=mask, twin=True)
            dense = dev(w["dense"]).float()
            keep.append(w)
        else:
            _, parts, q = _prepared(N, K, 30 + i, blocksize)
            code = parts[2] if code is None else code
            p = {"w": fmsa_hip.make_codebook_weight(parts[0], code, parts[1], blocksize), "nsz": None, "dY": dy, "r": r, "s": s,
                 "mask_src": mask, "qweight_t": fmsa_hip.gptq_transpose(parts[0]), "T": fmsa_hip.lora_down(dy, dev(B.to(dtype).t().contiguous())),
                 "At": dev(A.to(dtype).t().contiguous())}
            dense = dev(onf4.dequant(q, "fp32").t().contiguous())
            keep.append(parts)
        if r:
            lora = lora + s * (p["T"].float() @ dev(A.to(dtype)).float())
        else:
            p.update(r=0, T=None, At=None, mask_src=None)
        projs.append(p)
        ref = ref + dy.float() @ dense.t()
    return projs, ref, lora, keep


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,Ns,r,masked,cut", [
    (1, 256, [2048], 24, True, True),
    (300, 1152, [1024, 256, 1056], 24, True, True),  # ranges that begin and end inside a projection; N ends in half a stage
    (300, 1152, [1024, 256, 1056], 64, False, True),
    (65, 288, [2048], 0, False, True),               # no adapter
    (2000, 2016, [2048, 512, 288], 64, True, True),  # 64 cut tiles and 192 ranks, 104 and 128: both column tiles in a workgroup
    (2000, 3296, [4096], 128, False, True),          # of the second launch
    (513, 14336, [2048], 24, True, False),           # 168 tiles: too many to cut
    (1030, 14336, [2048], 24, True, False),          # 280 tiles: the whole round would cost more than the 24 give
    (8300, 2048, [2048], 24, True, True),            # 264 tiles: one whole round, 8 cut
])
def test_input_gradient(M, K, Ns, r, masked, cut, dtype):
    import fmsa_hip

    x = dev(randn((M, K), 2, dtype))
    x[::3, ::5] = 0
    projs, ref, lora, keep = _bwd_projs(M, K, Ns, r, 0.5, dtype, x if masked else None, "gptq")
    ref = ref + ((x != 0) * lora if masked else lora)
    assert _bwd_cut(projs, M, dtype) == cut
    whole = fmsa_hip.gptq_lora_bwd_dx(projs, M, K)
    split = fmsa_hip.gptq_lora_bwd_dx(projs, M, K, split=True)
    _no_further(split, whole, ref)
    assert torch.equal(split, fmsa_hip.gptq_lora_bwd_dx(projs, M, K, split=True)) and (cut or torch.equal(split, whole))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,Ns,r,masked,blocksize", [
    (300, 1152, [1088, 288], 24, True, 64),
    (300, 1152, [2048], 16, False, 128),
    (8300, 2048, [2048], 8, True, 64),  # one whole round, 8 tiles cut
])
def test_input_gradient_code_book(M, K, Ns, r, masked, blocksize, dtype):
    import fmsa_hip

    x = dev(randn((M, K), 2, dtype))
    x[::3, ::5] = 0
    projs, ref, lora, keep = _bwd_projs(M, K, Ns, r, 0.5, dtype, x if masked else None, "nf4", blocksize)
    ref = ref + ((x != 0) * lora if masked else lora)
    assert _bwd_cut(projs, M, dtype)
    split = fmsa_hip.gptq_lora_bwd_dx(projs, M, K, split=True)
    _no_further(split, fmsa_hip.gptq_lora_bwd_dx(projs, M, K), ref)
    assert torch.equal(split, fmsa_hip.gptq_lora_bwd_dx(projs, M, K, split=True))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("base", ["gptq", "nf4"])
@pytest.mark.parametrize("M,I,H,r,masked", [
    (300, 1152, 2048, 24, False),
    (300, 1152, 2048, 64, True),
    (77, 320, 2080, 0, False),
    (8300, 2048, 2048, 16, True),  # one whole round, 8 tiles cut
])
def test_swiglu_backward(M, I, H, r, masked, base, dtype):
    """e and g are overwritten by d_g and d_e in whole and in cut tiles alike; h does not depend on the product."""
    import fmsa_hip

    e, g = dev(randn((M, I), 7, dtype)), dev(randn((M, I), 8, dtype))
    e[::9, ::4] = 0  # h = 0 there: without a mask source h itself masks the adapter's part
    mask = None
    if masked:
        mask = dev(randn((M, I), 9, dtype))
        mask[::5, ::3] = 0
    projs, dh, lora, keep = _bwd_projs(M, I, [H], r, 0.5, dtype, mask, base)
    se = torch.sigmoid(e.float())
    h = se * e.float() * g.float()
    dh = dh + ((h if mask is None else mask) != 0) * lora
    refs = [dh * se * e.float(), dh * g.float() * se * (1.0 + e.float() * (1.0 - se))]
    assert _bwd_cut(projs, M, dtype)
    results = []
    for split in (False, True, True):
        eg = e.clone(), g.clone()
        h_out = fmsa_hip.gptq_lora_bwd_dx(projs, M, I, fmsa_hip.BWD_SWIGLU, e=eg[0], g=eg[1], split=split)
        results.append((h_out,) + eg)
    whole, split, again = results
    assert all(torch.equal(a, b) for a, b in zip(split, again)) and torch.equal(whole[0], split[0])
    assert not torch.equal(whole[1], split[1])  # it was cut: some sums round differently
    for a, b, ref in zip(split[1:], whole[1:], refs):
        _no_further(a, b, ref)
