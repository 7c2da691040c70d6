"""lora_down with few tokens, where the columns are split over workgroups: against the fp32 product, next to the unsplit
kernel (fmsa_lora_down)."""
import pytest
import torch

from tests.helpers import randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,C,r", [(1, 1024, 8), (1, 14336, 16), (15, 4096, 64), (17, 1056, 128), (300, 8200, 24), (2047, 4096, 64),
                                   (4000, 1536, 16)])
def test_lora_down_few_tokens(M, C, r, dtype):
    import fmsa_hip

    lib = fmsa_hip.lib()
    x = randn((M, C + 8), 1, dtype).cuda()[:, :C]  # a column slice
    wd = randn((r, C), 2, dtype, 0.05).cuda()
    ref = x.float() @ wd.float().t()
    whole = torch.empty((M, r), dtype=dtype, device="cuda")
    assert lib.fmsa_lora_down(x.data_ptr(), x.stride(0), wd.data_ptr(), M, C, r, fmsa_hip.act_enum(dtype), whole.data_ptr(), r,
                              torch.cuda.current_stream().cuda_stream) == 0
    wide = torch.full((M, r + 16), 3.0, dtype=dtype, device="cuda")
    out = fmsa_hip.lora_down(x, wd, out=wide[:, 8 : 8 + r])
    # another order of the fp32 sums meets a few other roundings of the result, no larger ones
    assert (out.float() - ref).norm() <= 1.02 * (whole.float() - ref).norm() + 1e-6 * ref.norm()
    assert torch.all(wide[:, :8] == 3.0) and torch.all(wide[:, 8 + r :] == 3.0)
    assert torch.equal(fmsa_hip.lora_down(x, wd), out)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,shapes", [(1, [(1024, 8), (14336, 16)]), (33, [(4096, 64), (1024, 64), (520, 64)]),
                                      (2047, [(96, 8), (4096, 128), (1056, 24)]), (300, [(2048, 16)] * 4),
                                      (1023, [(4096, 64), (1056, 24)]), (1024, [(4096, 64), (1056, 8)]), (1100, [(14336, 64), (520, 32)]),
                                      (1041, [(1032, 24), (2048, 32)])])
def test_lora_down_batch(M, shapes, dtype):
    """Products of different widths and ranks in one launch, the last one into a column slice."""
    import fmsa_hip

    jobs, refs = [], []
    for i, (C, r) in enumerate(shapes):
        x = randn((M, C + 8), 10 + i, dtype).cuda()[:, :C]
        wd = randn((r, C), 20 + i, dtype, 0.05).cuda()
        wide = torch.full((M, r + 16), 3.0, dtype=dtype, device="cuda")
        jobs.append((x, wd, wide[:, 8 : 8 + r] if i + 1 == len(shapes) else None))
        refs.append(x.float() @ wd.float().t())
    outs = fmsa_hip.lora_down_batch(jobs)
    for (x, wd, _), out, ref in zip(jobs, outs, refs):
        single = fmsa_hip.lora_down(x, wd)
        assert (out.float() - ref).norm() <= 1.02 * (single.float() - ref).norm() + 1e-6 * ref.norm()
    assert torch.all(wide[:, :8] == 3.0) and torch.all(wide[:, 8 + wd.shape[0] :] == 3.0)
    assert all(torch.equal(a, b) for a, b in zip(outs, fmsa_hip.lora_down_batch(jobs)))


def test_calls_do_not_share_partial_sums():
    """Two calls on one stream may interleave their launches (threads), and a captured one is replayed after the next has
    asked for more: the buffers of partial sums are the calls' own."""
    import fmsa_hip

    a, b = fmsa_hip._workspace(1 << 20, torch.device("cuda:0")), fmsa_hip._workspace(1 << 20, torch.device("cuda:0"))
    assert a.data_ptr() != b.data_ptr()
    x, wd = randn((3, 4096), 1, torch.bfloat16).cuda(), randn((16, 4096), 2, torch.bfloat16, 0.05).cuda()
    big = randn((1500, 8192), 3, torch.bfloat16).cuda()
    wb = randn((64, 8192), 4, torch.bfloat16, 0.05).cuda()
    ref, ref_b = fmsa_hip.lora_down(x, wd), fmsa_hip.lora_down(big, wb)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = fmsa_hip.lora_down(x, wd)
    for _ in range(3):
        assert torch.equal(fmsa_hip.lora_down(big, wb), ref_b)  # eager work of its own between the replays
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
