"""Adapter gradients of few tokens, one launch: token counts around the tiles of 32 and the eight waves that share them, columns
around the 64 of a workgroup, ranks around the tiles of 16, both orders of the output, and outputs the wide stores do not fit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _job(M, C, r, dtype, seed, transposed, out_dtype, strided):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    L = torch.randn(M, r + (8 if strided else 0), device="cuda", generator=gen).to(dtype)[:, :r]
    R = torch.randn(M, C + (16 if strided else 0), device="cuda", generator=gen).to(dtype)[:, :C]
    return L, R, 0.5, transposed, out_dtype


def _check(job, got):
    L, R, s, transposed, out_dtype = job
    ref = s * (L.double().t() @ R.double())
    ref = ref.t() if transposed else ref
    # fp32 sums of M products, each within M eps of the sum of their magnitudes, and the output's own rounding
    mag = s * (L.double().abs().t() @ R.double().abs())
    bound = (mag.t() if transposed else mag) * L.shape[0] * 2.0**-24
    bound = bound + {torch.float32: 2.0**-24, torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}[out_dtype] * (ref.abs() + bound) + 1e-7
    assert got.dtype == out_dtype and got.shape == ref.shape and bool(((got.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 31, 33, 255, 257, 289, 513, 2047])
@pytest.mark.parametrize("r", [8, 16, 24, 64, 72, 128])
def test_gradients(M, r, dtype):
    import fmsa_hip

    jobs = [_job(M, C, r, dtype, 7 * i, i % 2 == 1, out, i == 3)
            for i, (C, out) in enumerate([(8, torch.float32), (72, torch.float32), (520, dtype), (128, dtype), (64, torch.float32)])]
    got = fmsa_hip.lora_grad_batch(jobs)
    for job, g, again in zip(jobs, got, fmsa_hip.lora_grad_batch(jobs)):
        _check(job, g)
        assert torch.equal(g, again)


@pytest.mark.parametrize("M,C,r", [(2048, 4096, 16), (2049, 4096, 16), (4096, 4096, 64), (4097, 4096, 64), (4096, 2048, 96), (3072, 2048, 96), (3073, 2048, 96), (300, 33024, 128), (513, 33024, 128)])
def test_either_side_of_the_rule(M, C, r):
    import fmsa_hip

    job = _job(M, C, r, torch.bfloat16, 3, False, torch.float32, False)
    _check(job, fmsa_hip.lora_grad_batch([job])[0])


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("transposed", [False, True])
def test_an_output_between_16_byte_boundaries(out_dtype, transposed):
    import ctypes

    import fmsa_hip

    M, C, r = 100, 136, 24
    job = _job(M, C, r, torch.bfloat16, 5, transposed, out_dtype, False)
    flat = torch.full((C * r + 8,), 7.0, device="cuda", dtype=out_dtype)
    out = flat[1 : 1 + C * r]
    arr = (fmsa_hip.LoraGradJob * 1)()
    j = arr[0]
    j.L, j.R, j.out, j.ldl, j.ldr, j.C, j.r = job[0].data_ptr(), job[1].data_ptr(), out.data_ptr(), r, C, C, r
    j.scale, j.transpose_out, j.out_dtype = job[2], transposed, fmsa_hip._DTYPE_ENUM[out_dtype]
    lib = fmsa_hip.lib()
    ws = torch.empty(lib.fmsa_lora_grad_batch_workspace(arr, 1, M), dtype=torch.uint8, device="cuda")
    rc = lib.fmsa_lora_grad_batch(arr, 1, M, fmsa_hip.BF16, ws.data_ptr(), ws.numel(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    _check(job, out.view((C, r) if transposed else (r, C)))
    assert bool((flat[:1] == 7).all()) and bool((flat[1 + C * r :] == 7).all())
