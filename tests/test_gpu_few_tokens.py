"""The forward kernel for few tokens: against the fp32 product, next to the whole-tile kernel on the same operands (another
order of the fp32 sums, so the distance from the reference must not grow beyond what a handful of other roundings can do), and
straight from the adapters' parameters next to packed ones."""
import pytest
import torch

from oracle import lora as olora
from oracle import nf4 as onf4
from tests.helpers import make_gptq, randn
from tests.test_gpu_kernels import dev, gweight
from tests.test_gpu_nf4 import _prepared

pytestmark = pytest.mark.gpu


def _no_further(few, whole, ref):
    err, base = (few.float() - ref).norm(), (whole.float() - ref).norm()
    assert err <= 1.02 * base, (float(err), float(base))


def _packed(x, projs, mode):
    """What gptq_lora_fwd returns, on the kernel for few tokens whatever the rule says of the shape."""
    import fmsa_hip

    arr, outs = (fmsa_hip.FwdProj * len(projs))(), []
    for q, p in zip(arr, projs):
        y = x.new_empty((x.shape[0], p["w"].N))
        outs.append(y)
        q.w, q.Y, q.ldy, q.bias = p["w"], y.data_ptr(), y.stride(0), None if p["bias"] is None else p["bias"].data_ptr()
        if p["r"]:
            q.U, q.ldu, q.B, q.r, q.s = p["U"].data_ptr(), p["U"].stride(0), p["B"].data_ptr(), p["r"], p["s"]
    h = torch.empty_like(outs[0]) if mode == fmsa_hip.FWD_SWIGLU else None
    rc = fmsa_hip.lib().fmsa_gptq_lora_fwd_few(arr, len(projs), x.data_ptr(), x.stride(0), x.shape[0], mode,
                                               None if h is None else h.data_ptr(), 0 if h is None else h.stride(0),
                                               fmsa_hip.act_enum(x.dtype), torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    return outs if h is None else [*outs, h]


def _direct(x, few, mode):
    """lora_few, whatever the rule says of the shape."""
    import fmsa_hip

    L, arr, outs = fmsa_hip.lib(), (fmsa_hip.FewProj * len(few))(), []
    for q, (w, A, B, bias, s) in zip(arr, few):
        y = x.new_empty((x.shape[0], w.N))
        outs.append(y)
        q.w, q.Y, q.ldy, q.bias = w, y.data_ptr(), y.stride(0), None if bias is None else bias.data_ptr()
        if A is not None:
            q.A, q.B, q.r, q.s, q.param_dtype = A.data_ptr(), B.data_ptr(), A.shape[0], s, fmsa_hip.F32
    h = torch.empty_like(outs[0]) if mode == fmsa_hip.FWD_SWIGLU else None
    ws = torch.empty(max(16, L.fmsa_lora_few_workspace(arr, len(few), x.shape[0])), dtype=torch.uint8, device="cuda")
    rc = L.fmsa_lora_few_fwd(arr, len(few), x.data_ptr(), x.stride(0), x.shape[0], mode, None if h is None else h.data_ptr(),
                             0 if h is None else h.stride(0), fmsa_hip.act_enum(x.dtype), ws.data_ptr(), ws.numel(),
                             torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    return outs if h is None else h


def _weights(K, Ns, fmt, gs):
    ws, dense, keep, code = [], [], [], None
    for i, N in enumerate(Ns):
        if fmt == "nf4":
            _, parts, q = _prepared(N, K, 90 + i, gs)
            import fmsa_hip

            code = parts[2] if code is None else code
            ws.append(fmsa_hip.make_codebook_weight(parts[0], code, parts[1], gs))
            dense.append(dev(onf4.dequant(q, "fp32").t().contiguous()).float())
            keep.append(parts)
        else:
            w = make_gptq(K, N, gs, seed=40 + i)
            ws.append(gweight(w, interleaved=fmt == "interleaved"))
            dense.append(dev(w["dense"]).float())
            keep.append(w)
    return ws, dense, keep


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,Ns,swiglu,fmt,gs,bias,r", [
    (1, 4096, [1024], False, "gptq", 128, False, 16),
    (16, 512, [256, 96, 32], False, "gptq", 64, True, 8),         # eight chunks: one per wave
    (17, 1312, [288, 64], False, "gptq", 128, False, 24),         # K ends in half a chunk, second token tile of one token
    (33, 1312, [288, 288], True, "gptq", 128, True, 40),
    (64, 96, [64], False, "gptq", 192, True, 128),                # fewer chunks than waves, a group of three chunks
    (64, 2048, [512, 512], True, "interleaved", 128, False, 16),
    (5, 2080, [64, 32], False, "interleaved", 64, False, 0),
    (48, 640, [96], False, "nf4", 64, True, 64),
    (12, 2048, [320, 320], True, "nf4", 128, False, 8),
    (3, 576, [64, 32, 32], False, "nf4", 64, False, 16),
    (257, 512, [192, 64], False, "gptq", 128, False, 16),         # five token blocks, the last of one token
    (130, 544, [96, 96], True, "gptq", 64, True, 72),
    (200, 1024, [64], False, "nf4", 64, False, 16),
])
def test_few_tokens(M, K, Ns, swiglu, fmt, gs, bias, r, dtype):
    import fmsa_hip

    if fmt == "interleaved" and dtype != torch.float16:
        pytest.skip("the interleaved copy is read for fp16 activations")
    s, mode = 2.0, fmsa_hip.FWD_SWIGLU if swiglu else fmsa_hip.FWD_LINEAR
    x = dev(randn((M, K), 1, dtype))
    ws, dense, keep = _weights(K, Ns, fmt, gs)
    projs, few, refs = [], [], []
    for i, (w, W) in enumerate(zip(ws, dense)):
        A = B = U = None
        if r:
            A, B = (dev(t) for t in olora.make_lora(K, w.N, r, 50 + i))  # fp32, as parameters are kept
            U = fmsa_hip.lora_down(x, A.to(dtype))
        b = dev(randn((w.N,), 60 + i, dtype, 0.1)) if bias else None
        projs.append({"w": w, "U": U, "B": None if B is None else B.to(dtype), "bias": b, "r": r, "s": s})
        assert fmsa_hip.lora_few_ok(x, w, A, B) or M > fmsa_hip.FEW_TOKENS
        few.append((w, A, B, b, s))
        ref = x.float() @ W
        if r:
            ref = ref + s * (x.float() @ A.to(dtype).float().t()) @ B.to(dtype).float().t()
        refs.append(ref if b is None else ref + b.float())
    whole = fmsa_hip.gptq_lora_fwd(x, projs, mode)
    packed = _packed(x, projs, mode)
    direct = _direct(x, few, mode)
    if swiglu:
        refs = refs + [torch.nn.functional.silu(refs[0]) * refs[1]]
    for a, b, ref in zip(packed, whole, refs):
        _no_further(a, b, ref)
    for a, b in zip(packed, _packed(x, projs, mode)):
        assert torch.equal(a, b)
    # U of one projection is one lora_down; of several, what their stacked adapters give, whose ranges may be others
    for a, b, ref in zip([direct] if swiglu else direct, packed[2:] if swiglu else packed, refs[2:] if swiglu else refs):
        if len(ws) == 1:
            assert torch.equal(a, b)
        else:
            _no_further(a, b, ref)


@pytest.mark.parametrize("M", [1, 20, 64, 65])
def test_operators_without_a_graph(M):
    """The patched operators with gradients switched off (parameters read as they are, no autograd node) and on."""
    from fms_acceleration_foak.models.utils import FUSED_OPS
    from tests.model_utils import make_lora_gptq_linear

    H, I, r, dtype = 1536, 4608, 24, torch.bfloat16  # (the columns of the rank-r products are split)
    mod = torch.nn.Module()
    for i, (name, K, N) in enumerate((("q_proj", H, H), ("k_proj", H, 64), ("v_proj", H, 64), ("gate_proj", H, I), ("up_proj", H, I),
                                      ("down_proj", I, 128))):
        setattr(mod, name, make_lora_gptq_linear(K, N, r, 16.0, seed=70 + i, device="cuda:0")[0])
    ops = FUSED_OPS["auto_gptq"]
    x = dev(randn((1, M, H), 5, dtype))
    with_graph = list(ops["qkv"](mod, x)) + [ops["mlp"](mod, x), ops["o"](mod.q_proj, x)]
    with torch.no_grad():
        without = list(ops["qkv"](mod, x)) + [ops["mlp"](mod, x), ops["o"](mod.q_proj, x)]
    for a, b in zip(with_graph, without):
        assert a.requires_grad and not b.requires_grad and torch.equal(a, b)
