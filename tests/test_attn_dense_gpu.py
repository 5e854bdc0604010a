"""Dense attention of head dims 64 / 128 (csrc/kernels/attention_dense.hip) at the edges of its query blocks and key tiles."""
import pytest
import torch

from localai_tfp_amd.ops import core as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D,Hq,Hkv", [(64, 3, 3), (128, 4, 2)])
@pytest.mark.parametrize("Sq,Sk,causal,scale,pad", [(1, 1, False, None, 0), (31, 63, False, None, 0), (33, 64, True, None, 8),
                                                    (129, 65, True, None, 0), (128, 129, True, None, 1), (300, 200, False, -0.1, 2),
                                                    (127, 193, False, 0.0, 0)])
def test_blocks_tiles_and_masks(dt, D, Hq, Hkv, Sq, Sk, causal, scale, pad):
    """Ragged query and key lengths, more queries than keys under a causal mask (rows that see nothing are zero), scales that
    are not positive, out rows of any alignment. Probabilities and outputs are rounded to 16 bits once each (2^-9 in bf16): the
    relative error of a row of sums stays below 4 x 2^-9."""
    B = 3
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(B * s, h * D, generator=g).to(dt) for s, h in ((Sq, Hq), (Sk, Hkv), (Sk, Hkv)))
    scale = D ** -0.5 if scale is None else scale
    qlen = torch.tensor([Sq, max(1, Sq - 1), max(1, Sq // 2)], dtype=torch.int32)
    klen = None if causal else torch.tensor([Sk, max(1, Sk - 1), 0], dtype=torch.int32)
    want = torch.empty(B * Sq, Hq * D)
    K.attn_dense(q, k, v, want, B, Sq, Sk, Hq, Hkv, D, scale, causal, qlen=qlen, klen=klen)
    out = torch.zeros(B * Sq, Hq * D + pad, dtype=dt, device="cuda")[:, :Hq * D]
    K.attn_dense(q.cuda(), k.cuda(), v.cuda(), out, B, Sq, Sk, Hq, Hkv, D, scale, causal, qlen=qlen.cuda(),
                 klen=None if klen is None else klen.cuda())
    got = out.float().cpu()
    assert float((got - want).norm()) <= 4 * 2 ** -9 * float(want.norm())


def test_infinite_scores_hide_and_nan_stays():
    """A key of -inf times a positive query is hidden; a row whose only finite score is none stays what the softmax makes it."""
    D, S = 64, 70
    q, k, v = torch.ones(S, D), torch.zeros(S, D), torch.randn(S, D, generator=torch.Generator().manual_seed(0))
    k[5, 0] = float("-inf")
    out = torch.empty(S, D, dtype=torch.float16, device="cuda")
    K.attn_dense(q.half().cuda(), k.half().cuda(), v.half().cuda(), out, 1, S, S, 1, 1, D, 0.125)
    keep = [i for i in range(S) if i != 5]
    # (a mean of 69 values rounded to half, probabilities all alike)
    assert (out.float().cpu() - v[keep].half().float().mean(0)).abs().max() < 2e-3
    k[7, 0] = float("nan")
    K.attn_dense(q.half().cuda(), k.half().cuda(), v.half().cuda(), out, 1, S, S, 1, 1, D, 0.125)
    assert torch.isnan(out).all()
