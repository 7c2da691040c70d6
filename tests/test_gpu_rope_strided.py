"""The rotation read through strides against the in-place rotation of a contiguous copy: the same arithmetic, bit for bit."""
import pytest
import torch

from tests.helpers import randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qdt,cdt", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("b,t,h,d", [(1, 1, 1, 16), (2, 7, 3, 64), (3, 129, 8, 128), (1, 300, 4, 80)])
@pytest.mark.parametrize("layout", ["bhtd", "thbd", "wide", "expanded"])
def test_rope_strided(b, t, h, d, qdt, cdt, layout):
    import fmsa_hip

    if layout == "bhtd":
        q = randn((b, h, t, d), 1, qdt).cuda().transpose(1, 2)
    elif layout == "thbd":
        q = randn((t, h, b, d), 1, qdt).cuda().permute(2, 0, 1, 3)
    elif layout == "wide":
        q = randn((b, h, t, d + 16), 1, qdt).cuda()[..., 8 : 8 + d].transpose(1, 2)
    else:
        q = randn((b, 1, t, d), 1, qdt).cuda().expand(b, h, t, d).transpose(1, 2)
    ang = randn((t, d), 2).cuda()
    cos, sin = ang.cos().to(cdt), ang.sin().to(cdt)
    assert fmsa_hip.rope_strided_ok(q, cos, sin)
    keep = q.clone()
    for backward in (False, True):
        out = fmsa_hip.rope_embedding_strided(q, cos, sin, backward)
        ref = fmsa_hip.rope_embedding_(q.reshape(b * t, h * d).clone(), cos, sin, h, d, backward)
        assert torch.equal(out, ref)
    assert torch.equal(q, keep)


def test_rope_strided_refuses():
    import fmsa_hip

    cos = torch.ones(5, 64, device="cuda", dtype=torch.bfloat16)
    base = torch.zeros(2 * 5 * 4 * 64 + 8, device="cuda", dtype=torch.bfloat16)
    odd = base[1 : 1 + 2 * 5 * 4 * 64].view(2, 4, 5, 64).transpose(1, 2)  # not 16-byte aligned
    assert not fmsa_hip.rope_strided_ok(odd, cos, cos)
    apart = torch.zeros(2, 4, 5, 68, device="cuda", dtype=torch.bfloat16)[..., :64].transpose(1, 2)  # token stride 136 bytes
    assert not fmsa_hip.rope_strided_ok(apart, cos, cos)
    with pytest.raises(RuntimeError):
        fmsa_hip.rope_embedding_strided(odd, cos, cos)
