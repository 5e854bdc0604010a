"""RMSNorm of rows of one to eight 1024-wide chunks (csrc/kernels/norm.hip) against the same in 64 bits."""
import pytest
import torch

from localai_tfp_amd.ops import core as K


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("chunks", range(1, 9))
@pytest.mark.parametrize("rows,res", [(1, False), (1, True), (37, False), (37, True)])
def test_each_width_in_whole_chunks(chunks, rows, res, dtype):
    H = 1024 * chunks
    g = torch.Generator().manual_seed(chunks)
    x, w = torch.randn(rows, H, generator=g) * 3, torch.randn(H, generator=g)
    r = torch.randn(rows, H, generator=g).to(torch.bfloat16) if res else None
    s = x.double() + (r.double() if res else 0)
    want = s * torch.rsqrt(s.pow(2).mean(-1, keepdim=True) + 1e-5) * w
    xd = x.cuda()
    out = torch.full((rows, H + 8), float("nan"), dtype=dtype, device="cuda")[:, :H]
    q8 = (torch.empty(rows, H, dtype=torch.int8, device="cuda"), torch.empty(rows, H // 32, 2, device="cuda"))
    K.rmsnorm(xd, w.cuda(), 1e-5, out_bf16=out, out_q8=q8, residual_bf16=r.cuda() if res else None)
    # one rounding to 16 bits, 2^-11 or 2^-8 relative, beside fp32 sums of H terms and the smallest fp16 steps
    assert ((out.cpu().double() - want).abs() <= want.abs() * (2 ** -10 if dtype == torch.float16 else 2 ** -8) + 1e-6).all()
    if res:
        assert torch.equal(xd.cpu(), x + r.float())
    b = want.view(rows, -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127
    assert ((q8[0].cpu().view(rows, -1, 32) * q8[1].cpu()[..., :1].double() - b).abs() <= d * 0.501 + 1e-6).all()  # half a step


@pytest.mark.gpu
@pytest.mark.parametrize("narrow", [1024, 2048])
def test_a_width_does_not_choose_the_rounding(narrow):
    """Rows of 1024 n numbers and the same rows with zeros up to four times the width, eps a quarter: a quarter of the mean square, the
    square root of it halved, both without rounding, so all outputs are doubled bit for bit."""
    g = torch.Generator().manual_seed(narrow)
    x, w = torch.randn(700, 4 * narrow, generator=g).cuda(), (torch.rand(4 * narrow, generator=g) + 0.5).cuda()
    x[:, narrow:] = 0
    out = [torch.empty(700, H, dtype=torch.float16, device="cuda") for H in (narrow, 4 * narrow)]
    K.rmsnorm(x[:, :narrow].contiguous(), w[:narrow].contiguous(), 2.0 ** -16, out_bf16=out[0])
    K.rmsnorm(x, w, 2.0 ** -18, out_bf16=out[1])
    a, b = out[0].float(), out[1][:, :narrow].float()
    normal = a.abs() >= 2.0 ** -14  # (smaller ones have fewer bits)
    assert torch.equal(2 * a[normal], b[normal]) and normal.float().mean() > 0.99
