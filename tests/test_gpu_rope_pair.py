"""Q and K rotated by one launch where no graph is built, against a launch for each."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,cs_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("batch,seq,heads,kv_heads,head_dim,cs_batch", [
    (1, 1, 32, 8, 128, 1), (12, 1, 32, 8, 128, 12), (2, 77, 4, 4, 64, 1), (3, 5, 1, 1, 16, 3), (1, 300, 2, 7, 32, 1),
])
def test_pair_is_the_two_launches(batch, seq, heads, kv_heads, head_dim, cs_batch, dtype, cs_dtype):
    from fms_acceleration_foak.kernels.unsloth.rope_embedding import Fast_RoPE_Embedding, fast_rope_embedding

    torch.manual_seed(seq)
    Q = torch.randn(batch, seq, heads, head_dim, device="cuda").to(dtype)
    K = torch.randn(batch, seq, kv_heads, head_dim, device="cuda").to(dtype)
    cos, sin = (torch.randn(cs_batch, seq, head_dim, device="cuda").to(cs_dtype) for _ in range(2))
    want = [Fast_RoPE_Embedding.apply(t.clone(), cos, sin).transpose(1, 2) for t in (Q, K)]
    with torch.no_grad():
        got = fast_rope_embedding(Q.clone().transpose(1, 2), K.clone().transpose(1, 2), cos, sin)
    for g, w in zip(got, want):
        assert torch.equal(g, w)


@pytest.mark.parametrize("first_k", [0, 64, 128])
def test_shared_storage_is_rotated_in_order(monkeypatch, first_k):
    """K over the first token of Q, over its second, and next to it: a launch each, Q's first."""
    import fmsa_hip
    from fms_acceleration_foak.kernels.unsloth.rope_embedding import Fast_RoPE_Embedding, fast_rope_embedding

    pairs = []
    monkeypatch.setattr(fmsa_hip, "rope_embedding_pair_", lambda *a: pairs.append(a))
    base = torch.randn(192, device="cuda").to(torch.bfloat16)
    cos, sin = (torch.randn(2, 16, device="cuda").to(torch.bfloat16) for _ in range(2))

    def views(t):
        return t[:128].view(1, 2, 4, 16), t[first_k:first_k + 64].view(1, 2, 2, 16)

    want, got = base.clone(), base.clone()
    for t in views(want):
        Fast_RoPE_Embedding.apply(t, cos, sin)
    with torch.no_grad():
        fast_rope_embedding(*(t.transpose(1, 2) for t in views(got)), cos, sin)
    assert torch.equal(got, want) and not torch.equal(got[:128], base[:128]) and not pairs
