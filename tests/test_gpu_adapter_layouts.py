"""The adapters' packed copies and the gradients' reduction at the edges of their tiles, and where parameters or outputs begin
anywhere (views into a flat buffer): against torch's own transposes and roundings, bit for bit where nothing is summed."""
import pytest
import torch

from tests.helpers import randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("param", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("act", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("r,K,N,offset", [(8, 96, 32, 0), (16, 64, 4128, 0), (72, 2080, 200, 1), (128, 128, 64, 2), (24, 32, 65 * 8, 3), (7, 33, 5, 0)])
def test_pack(r, K, N, offset, param, act):
    import fmsa_hip

    flat = randn((offset + r * K + offset + N * r,), 3, param).cuda()
    A, B = flat[offset : offset + r * K].view(r, K), flat[2 * offset + r * K :].view(N, r)
    A16, At, B16, Bt = fmsa_hip.lora_pack(A, B, act)
    for got, want in ((A16, A), (At, A.t()), (B16, B), (Bt, B.t())):
        assert torch.equal(got, want.to(act).contiguous())


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,C,r", [(1, 8, 8), (33, 264, 24), (700, 520, 72), (1100, 1032, 128)])
def test_gradients_of_both_orders(M, C, r, out_dtype):
    """scale L^T R and its transpose are the same sums, rounded once."""
    import fmsa_hip

    L, R = randn((M, r), 1, torch.bfloat16).cuda(), randn((M, C), 2, torch.bfloat16).cuda()
    straight, turned = fmsa_hip.lora_grad_batch([(L, R, 0.5, False, out_dtype), (L, R, 0.5, True, out_dtype)])
    assert torch.equal(straight, turned.t().contiguous())
    ref = 0.5 * L.double().t() @ R.double()
    # M products of two bf16 numbers summed in fp32, one rounding of the result
    bound = M * 2.0 ** -23 * (0.5 * L.double().abs().t() @ R.double().abs()) + (2.0 ** -8 if out_dtype == torch.bfloat16 else 0.0) * ref.abs()
    assert bool(((straight.double() - ref).abs() <= bound).all())
    store = torch.empty(1 + C * r, device="cuda", dtype=out_dtype)
    out = store[1:].view(C, r)
    fmsa_hip.lora_grad_static(L, R, 0.5, True, out)
    assert torch.equal(out, turned)


@pytest.mark.parametrize("param", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("r,K,N,offset", [(32, 4096, 4104, 0), (24, 1024, 5464, 4), (64, 2056, 2048, 2), (40, 36, 12, 0)])
def test_pack_on_both_sides_of_the_tile_rule(r, K, N, offset, param):
    """Matrices of up to 128 Ki elements and more in one call, rows that are no whole tiles, parameters read 8 and 2 bytes at a time."""
    test_pack(r, K, N, offset, param, torch.bfloat16)
