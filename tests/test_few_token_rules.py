"""Which launches the rank-r products and adapter gradients of few tokens take: host-side rules, asked without a GPU."""
import pytest
import torch

import fmsa_hip
from fms_acceleration_foak.fused_ops.unsloth_lora import fused_core as core


class _Weight:
    perm = perm_key = None

    def __init__(self, K, N):
        self.K, self.N = K, N


def _projs(K, Ns, r):
    projs = []
    for N in Ns:
        p = core._Proj(_Weight(K, N), None, torch.empty(r, K, device="meta"), torch.empty(N, r, device="meta"), 2.0, torch.bfloat16)
        p.Bt = torch.empty(r, N, device="meta", dtype=torch.bfloat16)
        projs.append(p)
    return projs


def _meta(*shape):
    return torch.empty(*shape, device="meta", dtype=torch.bfloat16)


@pytest.mark.parametrize("M", [1, 300, 512, 513])
def test_t_has_its_own_launch_for_few_tokens(M):
    """T out of the gradient launch pays from 96 MB of dY on, however many projections share the launch."""
    projs = _projs(4096, (4096, 1024, 1024), 16)
    assert not core._fuse_t(projs, [_meta(M, p.w.N) for p in projs])
    wide = _projs(8192, (28672, 28672), 16)
    assert core._fuse_t(wide, [_meta(1024, p.w.N) for p in wide])


@pytest.mark.parametrize("M,N,r,batched", [(2047, 28672, 16, False), (2047, 28672, 8, False), (2047, 28672, 32, True), (1536, 28672, 16, True),
                                           (2047, 14336, 16, True)])
def test_unstacked_projections_keep_t_in_the_gradient_launch_where_it_pays(monkeypatch, M, N, r, batched):
    calls = []
    monkeypatch.setattr(fmsa_hip, "lora_down_batch", lambda jobs: calls.append("down_batch") or [_meta(M, r) for _ in jobs])
    monkeypatch.setattr(fmsa_hip, "lora_down", lambda *a, **k: calls.append("down") or _meta(M, r))
    monkeypatch.setattr(fmsa_hip, "lora_grad_batch", lambda jobs: calls.append("grad") or [_meta(1, 1) for _ in jobs])
    projs = _projs(8192, (N, N), r)
    Ts, grads = core._adapter_grads(projs, [_meta(M, N)] * 2, [_meta(M, 8192)] * 2, [_meta(M, r)] * 2, None)
    assert len(Ts) == len(grads) == 2
    assert calls == (["down_batch", "grad"] if batched else ["grad"] * 4)


@pytest.mark.parametrize("M,C,r,split", [(300, 1024, 16, False), (1, 1024, 32, False), (300, 1024, 64, True), (300, 1024, 128, True),
                                         (1, 2048, 16, False), (300, 2048, 24, True), (1, 4096, 8, True), (2047, 4096, 8, True),
                                         (2048, 1024, 128, False), (3000, 1536, 64, False), (2048, 2048, 64, True)])
def test_columns_are_split_where_the_second_launch_pays(M, C, r, split):
    assert (fmsa_hip.lib().fmsa_lora_down_split_workspace(M, C, r) > 0) == split


@pytest.mark.parametrize("M,C,r,ranges", [(3217, 14336, 16, 10), (4095, 14336, 16, 4), (2048, 8192, 8, 8), (2100, 28672, 16, 15),
                                          (1100, 8192, 8, 7), (1100, 14336, 8, 28)])
def test_which_products_64_token_workgroups_take(M, C, r, ranges):
    """By the ranges of their buffer: theirs where the staged kernels need a second round of workgroups or the fragment kernel
    is bound by its loads (26 / 20, 23 / 28, 10.6 / 11.4, 24 / 17, 10.1 / 11.4, 14.6 / 11 us without / with)."""
    assert fmsa_hip.lib().fmsa_lora_down_split_workspace(M, C, r) == ranges * M * r * 4


def _struct(K, N, codebook=False, group=128):
    return fmsa_hip.GptqWeight(0x1000, None if codebook else 0x2000, None if codebook else 0x3000, None, K, N, 64 if codebook else group, 0,
                               fmsa_hip.WEIGHT_CODEBOOK if codebook else fmsa_hip.WEIGHT_AFFINE, 0, 0x7000 if codebook else None,
                               0x8000 if codebook else None)


def _cut_fwd(M, K, Ns, swiglu=False, **kw):
    arr = (fmsa_hip.FwdProj * len(Ns))()
    for i, N in enumerate(Ns):
        arr[i].w = _struct(K, N, **kw)
    return fmsa_hip.lib().fmsa_gptq_lora_fwd_workspace(arr, len(Ns), M, fmsa_hip.FWD_SWIGLU if swiglu else fmsa_hip.FWD_LINEAR) > 0


def _cut_bwd(M, K, Ns, **kw):
    arr = (fmsa_hip.BwdProj * len(Ns))()
    for i, N in enumerate(Ns):
        arr[i].w, arr[i].nsz, arr[i].qweight_t, arr[i].scale_f32 = _struct(K, N, **kw), 0x4000, 0x5000, 0x6000
    return fmsa_hip.lib().fmsa_gptq_lora_bwd_dx_workspace(arr, len(Ns), M, 1) > 0


def test_tiles_are_cut_where_that_pays():
    """Few tiles are cut; so is the rest behind whole rounds while those cost less on the flavour that cuts than it gives."""
    assert _cut_fwd(1, 4096, [4096, 1024, 1024]) and _cut_fwd(200, 4096, [14336, 14336], swiglu=True)
    assert not _cut_fwd(1536, 2048, [4096, 4096], swiglu=True)     # 192 tiles: no CUs to cut for
    assert _cut_fwd(4400, 4096, [4096]) and _cut_fwd(6144, 14336, [4096])      # 288 and 384 tiles
    assert not _cut_fwd(7131, 4096, [14336, 14336], swiglu=True)   # 12 whole rounds and 64 tiles: 1359 us whole, 1394 cut
    assert _cut_bwd(1, 4096, [4096]) and _cut_bwd(300, 14336, [4096])
    assert _cut_bwd(4352, 4096, [14336]) and _cut_bwd(4352, 4096, [14336], codebook=True)  # 272 tiles, long contraction
    for M in (6107, 7131, 7387):  # five or six whole rounds in front: 617 / 656, 727 / 767, 729 / 796 us whole / cut
        assert not _cut_bwd(M, 14336, [4096])
    assert not _cut_bwd(7131, 8192, [8192, 1024, 1024])            # three rounds and 128 tiles: 941 / 986


@pytest.mark.parametrize("M,K,N", [(1, 4096, 1024), (256, 4096, 1024), (1024, 1024, 1024), (700, 4096, 2048), (2048, 2048, 2048)])
def test_short_contractions_from_a_code_book_are_cut(M, K, N):
    """16 and 32 stages on 16 to 64 tiles: whole they take 34 and 52 us, cut 18 to 42."""
    assert _cut_bwd(M, K, [N], codebook=True)


@pytest.mark.parametrize("cut,rotating", [((), (True, True)), (("k",), (True, False)), (("q",), (False, True)), (("q", "k"), (False, False))])
def test_rotation_is_decided_per_launch(monkeypatch, cut, rotating):
    """Projections that walk K in orders of their own are launched one by one: each is asked whether its launch is cut."""
    launches, passes, M = [], [], 40
    monkeypatch.setattr(fmsa_hip, "gptq_lora_fwd_splits", lambda weights, m: weights[0] in cut if len(weights) == 1 else "joint" in cut)
    monkeypatch.setattr(fmsa_hip, "permute_cols", lambda x, *a, **k: x)
    monkeypatch.setattr(fmsa_hip, "gptq_lora_fwd", lambda x, projs, *a, rope=None, **k: launches.append((projs[0]["w"], rope is not None))
                        or [_meta(M, 256) for _ in projs])
    monkeypatch.setattr(fmsa_hip, "rope_embedding_", lambda y, *a, **k: passes.append(1))
    projs = []
    for i, name in enumerate("qkv"):
        w = _Weight(256, 256)
        w.struct, w.perm, w.perm_key, w.group_size = name, torch.empty(256, device="meta"), i, 128
        projs.append(core._Proj(w, None, None, None, None, torch.bfloat16))
    table = _meta(M, 64)
    outs, _ = core._linear_forward(projs, _meta(M, 256), [_meta(M, 256)] * 3, None, (table, table, 64, 0b011))
    assert len(outs) == 3 and launches == [("q", rotating[0]), ("k", rotating[1]), ("v", False)]
    assert len(passes) == 2 - sum(rotating)


def _few(M, K, Ns, swiglu=False, **kw):
    arr = (fmsa_hip.FwdProj * len(Ns))()
    for q, N in zip(arr, Ns):
        q.w = _struct(K, N, **kw)
    return fmsa_hip.lib().fmsa_gptq_lora_fwd_is_few(arr, len(Ns), M, fmsa_hip.FWD_SWIGLU if swiglu else fmsa_hip.FWD_LINEAR) == 1


def test_the_kernel_for_few_tokens_is_taken_where_it_is_faster():
    for M in (1, 64):
        assert _few(M, 14336, [4096]) and _few(M, 4096, [14336, 14336], swiglu=True) and _few(M, 8192, [28672], codebook=True)
    assert _few(300, 4096, [4096]) and not _few(513, 4096, [4096])
    assert _few(700, 2048, [2048]) and not _few(769, 2048, [2048])
    assert _few(300, 2048, [4096, 4096], swiglu=True) and not _few(513, 2048, [4096, 4096], swiglu=True)
    assert not _few(129, 4096, [14336, 14336], swiglu=True) and not _few(64, 4096, [4096], group=32)
    assert not _few(700, 4096, [4096, 1024, 1024])
    assert not _few(1, 256, [256, 64, 64]) and _few(1, 256, [256, 256], swiglu=True)
