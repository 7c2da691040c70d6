"""bitsandbytes-flavoured helpers of the fused operators (reference:
fused_ops/unsloth_lora/utils.py:53-141, 250-283): quant-state lookup, parameter scrape, and
`fast_dequantize`, which here is one launch of libfmsa_hip's NF4 kernel instead of two ctypes calls
into libbitsandbytes."""
from __future__ import annotations

import torch

import fmsa_hip


def QUANT_STATE(W, base_layer):
    """The quant state normally rides on the weight; fall back to the layer (FSDP re-creates the
    parameter and drops python attributes)."""
    if hasattr(W, "quant_state"):
        return W.quant_state
    return getattr(base_layer, "quant_state", None)


_RAISE = object()


def member(module, kind, name, default=_RAISE):
    """getattr(module, name) for what a module keeps in its `kind` dictionary (_modules, _buffers, _parameters), asked for
    there first: nn.Module.__getattr__ runs after a failed lookup and searches all three, which a layer pass of seven
    adapted projections pays for a hundred times.  Anything kept elsewhere (a property, a plain attribute) is found as
    getattr finds it, and a plain attribute goes first, as there.  The dictionary is asked by subscript, as
    nn.Module.__getattr__ does: one that gathers a partitioned parameter on access does it there, and not in get()."""
    own = module.__dict__
    found = own.get(kind)
    if found is not None and name in found and name not in own:
        return found[name]
    return getattr(module, name) if default is _RAISE else getattr(module, name, default)


def active_adapter_parts(proj):
    """(A, B, scaling, dropout) of the active adapter of a LoRA layer."""
    active = proj.active_adapters[0] if hasattr(proj, "active_adapters") else proj.active_adapter
    A = member(member(proj, "_modules", "lora_A")[active], "_parameters", "weight")
    B = member(member(proj, "_modules", "lora_B")[active], "_parameters", "weight")
    dropout = member(proj, "_modules", "lora_dropout", None)
    return A, B, proj.scaling[active], None if dropout is None else dropout[active]


def get_lora_parameters(proj):
    base_layer = member(proj, "_modules", "base_layer", proj)
    W = member(base_layer, "_parameters", "weight")
    bias = getattr(base_layer, "bias", None)
    if not hasattr(proj, "disable_adapters") or proj.disable_adapters or proj.merged:
        return W, QUANT_STATE(W, base_layer), bias, None, None, None, None
    return (W, QUANT_STATE(W, base_layer), bias) + active_adapter_parts(proj)


def fast_dequantize(W, quant_state=None, out_dtype=None):
    """Dense weight of an NF4 tensor with double-quantised absmax, as [N, K] row-major (callers
    transpose the view when they need [K, N]).  Without a quant state W is returned as is."""
    if quant_state is None:
        return W
    from fmsa_hip.nf4_prepared import normalize_quant_state  # the older list form is accepted too (:100-105)

    quant_state = normalize_quant_state(quant_state)
    state2 = quant_state.state2
    if state2 is None or quant_state.absmax.dtype != torch.uint8:
        raise NotImplementedError("only double-quantised NF4 weights (compress_statistics=True) are supported")
    data = W.data if isinstance(W, torch.nn.Parameter) else W
    return fmsa_hip.nf4_dequant(data.reshape(-1), quant_state.absmax, state2.absmax, state2.code, quant_state.code,
                                float(quant_state.offset), tuple(quant_state.shape), quant_state.blocksize,
                                state2.blocksize, out_dtype or quant_state.dtype)
