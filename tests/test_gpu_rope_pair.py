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
        both = torch.cat([Q, K], dim=2)  # one storage: a launch each, in order
        shared = fast_rope_embedding(both[:, :, :heads].transpose(1, 2), both[:, :, heads:].transpose(1, 2), cos, sin) if batch * seq == 1 else got
    for g, s, w in zip(got, shared, want):
        assert torch.equal(g, w) and torch.equal(s, w)
