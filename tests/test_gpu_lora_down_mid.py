"""lora_down on workgroups of 64 tokens: edges of its token tiles, chunks of 64 columns and blocks of 64 ranks, against fp64 with
the bound of fp32 sums and one rounding; single calls next to the batched launch."""
import pytest
import torch

from tests.helpers import randn

pytestmark = pytest.mark.gpu


def _within(out, x, wd, dtype):
    ref = x.double() @ wd.double().t()
    size = x.double().abs() @ wd.double().abs().t()  # C products summed in fp32, one rounding of the result
    bound = x.shape[1] * 2.0 ** -24 * size + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) * ref.abs() + 1e-7
    return bool(((out.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,C,r", [(65, 64, 72), (128, 1032, 128), (129, 200, 80),      # fewer chunks than waves, ragged ends
                                   (300, 520, 128), (128, 1056, 128), (513, 3104, 64),  # a last range of one chunk, of fewer than the others
                                   (700, 4160, 64), (1100, 14336, 16), (1999, 4104, 24),
                                   (2048, 2048, 32), (2050, 8200, 8), (3001, 2056, 120)])
def test_single(M, C, r, dtype):
    import fmsa_hip

    x = randn((M, C + 8), 1, dtype).cuda()[:, 8:]
    wd = randn((r, C), 2, dtype, 0.05).cuda()
    wide = torch.full((M, r + 16), 3.0, dtype=dtype, device="cuda")
    out = fmsa_hip.lora_down(x, wd, out=wide[:, 8 : 8 + r])
    assert _within(out, x, wd, dtype)
    assert torch.all(wide[:, :8] == 3.0) and torch.all(wide[:, 8 + r :] == 3.0)
    assert torch.equal(out, fmsa_hip.lora_down(x, wd))


@pytest.mark.parametrize("M,C,r", [(700, 5120, 64), (1100, 14336, 16), (3217, 8256, 16), (2050, 2112, 32), (600, 1088, 128)])
def test_rows_of_whole_lines_and_others(M, C, r):
    """Rows on 128-byte lines are read past the caches, others through them: the same sums."""
    import fmsa_hip

    x, wd = randn((M, C), 1, torch.bfloat16).cuda(), randn((r, C), 2, torch.bfloat16, 0.05).cuda()
    out = fmsa_hip.lora_down(x, wd)
    assert _within(out, x, wd, torch.bfloat16)
    for start, ld in ((0, C + 64), (32, C + 64), (0, C + 40)):  # whole lines; half a line on; rows between lines
        view = torch.empty(M * ld + start, dtype=torch.bfloat16, device="cuda").as_strided((M, C), (ld, 1), start)
        view.copy_(x)
        assert torch.equal(fmsa_hip.lora_down(view, wd), out)


@pytest.mark.parametrize("M,shapes", [(300, [(4096, 64), (1024, 64), (1024, 64)]), (512, [(96, 128), (520, 8)]),
                                      (1100, [(14336, 64), (64, 16), (4096, 72)])])
def test_batch(M, shapes):
    import fmsa_hip

    jobs = [(randn((M, C), 3 + i, torch.bfloat16).cuda(), randn((r, C), 9 + i, torch.bfloat16, 0.05).cuda(), None) for i, (C, r) in enumerate(shapes)]
    outs = fmsa_hip.lora_down_batch(jobs)
    for (x, wd, _), out in zip(jobs, outs):
        assert _within(out, x, wd, torch.bfloat16)
    assert all(torch.equal(a, b) for a, b in zip(outs, fmsa_hip.lora_down_batch(jobs)))
