"""Where Q and K are expected to leave a projection launch rotated, and where a pass after it is the faster way: what was measured,
us rotated in the launch / after it, in the comments."""
import pytest

from tests.test_few_token_rules import _struct


def _pays(M, K, Ns, **kw):
    import fmsa_hip

    arr = (fmsa_hip.FwdProj * len(Ns))()
    for q, N in zip(arr, Ns):
        q.w = _struct(K, N, **kw)
    return fmsa_hip.lib().fmsa_gptq_lora_fwd_rope_pays(arr, len(Ns), M)


@pytest.mark.parametrize("K,Ns,M,pays", [
    (4096, (4096, 1024, 1024), 1, 0), (4096, (4096, 1024, 1024), 512, 0),  # 85 / 12, 87 / 49: cut
    (4096, (4096, 1024, 1024), 1100, 0), (4096, (4096, 1024, 1024), 1536, 0),  # 89 / 68, 88 / 82: lower tiles
    (4096, (4096, 1024, 1024), 2048, 1), (4096, (4096, 1024, 1024), 2560, 1),  # 95 / 106, 109 / 120: the same tiles
    (4096, (4096, 1024, 1024), 3217, 0), (4096, (4096, 1024, 1024), 6000, 0),  # 195 / 163, 302 / 282
    (4096, (4096, 1024, 1024), 4096, 1), (4096, (4096, 1024, 1024), 8192, 1),  # 198 / 213 (a cut one), 344 / 357
    (2048, (2048, 512, 512), 2048, 0), (2048, (2048, 512, 512), 4096, 1), (2048, (2048, 512, 512), 6000, 0),  # 52 / 42, 54 / 62, 108 / 91
    (8192, (8192, 1024, 1024), 1100, 0), (8192, (8192, 1024, 1024), 2048, 0),  # 185 / 172, 366 / 314
    (8192, (8192, 1024, 1024), 1536, 1), (8192, (8192, 1024, 1024), 2560, 1), (8192, (8192, 1024, 1024), 8192, 1),  # 209 / 220, 372 / 388, 1046 / 1080
    (256, (256, 128, 128), 1, 1), (256, (256, 128, 128), 128, 1), (512, (512, 256, 256), 700, 1),  # a few stages: the launches count
    (512, (512, 128, 192), 140, 0), (2048, (2048, 512, 512), 64, 0),  # the kernel for few tokens
])
@pytest.mark.parametrize("codebook", [False, True])
def test_the_faster_way_is_taken(K, Ns, M, pays, codebook):
    assert _pays(M, K, Ns, codebook=codebook, group=64 if codebook else 128) == pays


def test_what_the_rotating_flavours_do_not_take():
    assert _pays(0, 4096, (4096,)) == 0 and _pays(2048, 0, (4096,)) == 0
    assert _pays(8192, 4096, (4096,), group=32) == 0
