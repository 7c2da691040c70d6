"""Few tokens without a graph: the calls whose look-ups run in native code give the bits of the general way, and leave to it what it
alone takes."""
import pytest
import torch

from fms_acceleration_foak.fused_ops.unsloth_lora import fused_core as core
from fms_acceleration_foak.kernels.unsloth import fast_rms_layernorm, rms_layernorm
from fms_acceleration_foak.models.utils import FUSED_OPS
from tests.model_utils import MaskDropout, make_lora_gptq_linear, make_lora_nf4_linear

pytestmark = pytest.mark.gpu


def _module(base, names, K, N, **kw):
    module = torch.nn.Module()
    for i, name in enumerate(names):
        k, n = (N, K) if name == "down_proj" else (K, N)
        make = make_lora_nf4_linear if base == "bitsandbytes" else make_lora_gptq_linear
        setattr(module, name, make(k, n, 16, 32.0, seed=20 + i, device="cuda", **kw)[0])
    return module


def _ways(monkeypatch, call):
    """(result of the call, result of the general way, whether native code made the call)"""
    taken = []
    for name in ("few_linear", "few_mlp"):
        f = getattr(core, name)
        monkeypatch.setattr(core, name, lambda *a, f=f: taken.append(f(*a)) or taken[-1])
    with torch.no_grad():
        call()  # weights are prepared
        taken.clear()
        native = call()
    made = taken[0] is not None
    for name in ("few_linear", "few_mlp"):
        monkeypatch.setattr(core, name, lambda *a: None)
    with torch.no_grad():
        general = call()
    monkeypatch.undo()
    return native, general, made


def _equal(a, b):
    a, b = (t if isinstance(t, tuple) else (t,) for t in (a, b))
    return len(a) == len(b) and all(x.shape == y.shape and x.dtype == y.dtype and torch.equal(x, y) for x, y in zip(a, b))


CALLS = {"qkv": ("q_proj", "k_proj", "v_proj"), "mlp": ("gate_proj", "up_proj", "down_proj"), "o": ("o_proj",)}


@pytest.mark.parametrize("base,dtype", [("auto_gptq", torch.bfloat16), ("auto_gptq", torch.float16), ("bitsandbytes", torch.bfloat16)])
@pytest.mark.parametrize("op", CALLS)
@pytest.mark.parametrize("shape,made", [((1, 1), True), ((3, 5), True), ((64,), True), ((65,), False)])
def test_bits(monkeypatch, op, base, dtype, shape, made):
    module = _module(base, CALLS[op], 2048, 1024)
    x = torch.randn(*shape, 2048, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3)).to(dtype)
    arg = module.o_proj if op == "o" else module
    native, general, was = _ways(monkeypatch, lambda: FUSED_OPS[base][op](arg, x))
    assert was == made and _equal(native, general)


@pytest.mark.parametrize("form,made", [("bias", False), ("bias_of_the_type", True), ("strided", False), ("disabled", False), ("dropout", False),
                                       ("act_order", False), ("half_adapter", True), ("scaled_in_place", False)])
def test_forms(monkeypatch, form, made):
    kw = {"bias": {"bias": True}, "bias_of_the_type": {"bias": True}, "act_order": {"act_order": True},
          "half_adapter": {"lora_dtype": torch.bfloat16}}.get(form, {})
    dtype = torch.float16 if form == "bias_of_the_type" else torch.bfloat16
    module = _module("auto_gptq", CALLS["qkv"], 2048, 1024, **kw)
    x = torch.randn(6, 2048, device="cuda").to(dtype)
    if form == "strided":
        x = torch.randn(6, 4096, device="cuda").to(dtype)[:, ::2]
    if form == "disabled":
        module.k_proj.enable_adapters(False)
    if form == "dropout":
        module.v_proj.lora_dropout["default"] = MaskDropout(0.5, (6, 2048)).cuda()
    call = lambda: FUSED_OPS["auto_gptq"]["qkv"](module, x)
    native, general, was = _ways(monkeypatch, call)
    assert was == (made or form == "scaled_in_place") and _equal(native, general)
    if form == "scaled_in_place":  # the prepared weight is another one from here on
        module.q_proj.base_layer.scales.mul_(2)
        with torch.no_grad():
            changed = call()
        assert not torch.equal(changed[0], native[0]) and torch.equal(changed[1], native[1])


def test_a_graph_is_built_where_one_is_asked_for():
    module = _module("auto_gptq", CALLS["qkv"], 2048, 1024)
    x = torch.randn(6, 2048, device="cuda").bfloat16()
    assert all(y.requires_grad for y in FUSED_OPS["auto_gptq"]["qkv"](module, x))


@pytest.mark.parametrize("dtype,wtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("shape", [(1, 1, 512), (7, 2048), (64,), (3, 5, 4096)])
@pytest.mark.parametrize("gemma", [False, True])
def test_rms_layernorm(monkeypatch, shape, dtype, wtype, gemma):
    norm = torch.nn.Module()
    norm.weight, norm.variance_epsilon = torch.nn.Parameter(torch.randn(shape[-1], device="cuda").to(wtype)), 1e-5
    x = torch.randn(shape, device="cuda").to(dtype)
    with torch.no_grad():
        native, strided = fast_rms_layernorm(norm, x, gemma), fast_rms_layernorm(norm, x.repeat_interleave(2, -1)[..., ::2], gemma)
        monkeypatch.setattr(rms_layernorm, "no_graph", lambda: False)
        general = fast_rms_layernorm(norm, x, gemma)
    assert _equal(native, general) and _equal(strided, general)


@pytest.mark.parametrize("C", [8, 504, 4096])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rms_layernorm_asks_for_the_weight_early_up_to_64_rows(C, dtype):
    import fmsa_hip

    x, w = torch.randn(65, C, device="cuda").to(dtype), torch.randn(C, device="cuda").to(dtype)
    y, r = fmsa_hip.rms_layernorm_fwd(x, w, 1e-5, False)
    for M in (1, 63, 64):
        y_few, r_few = fmsa_hip.rms_layernorm_fwd(x[:M], w, 1e-5, False)
        assert torch.equal(y_few, y[:M]) and torch.equal(r_few, r[:M])
