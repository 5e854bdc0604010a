"""Partitions of the hybrid models' decode attention (ops/hybrid.py)."""
import random
import types

import pytest
import torch

from localai_tfp_amd.ops import hybrid as HY


def test_partitions_fit_their_workspace():
    rng = random.Random(3)
    for _ in range(3000):
        seqs, G, group = rng.randint(1, 200), rng.choice((1, 2, 5, 8, 32)), rng.choice((1, 2, 4, 12, 16))
        nd, vis = rng.randint(1, seqs), rng.choice((1, 64, 700, 2048, 8192, 131072))
        plen = HY.decode_part_len(nd, G, vis, HY.decode_waves_mfma())
        parts = min(64, -(-vis // plen))
        assert plen % 64 == 0 and (parts == 1 or nd * G * group * parts <= HY.partition_rows(seqs, G * group, group))


def test_two_partitions_are_one():
    waves = HY.decode_waves_mfma()
    for nd, G, want in ((waves // 24, 8, 3), (waves // 24 + 1, 8, 1), (waves // 16, 16, 1), (1, 1, 128)):
        assert -(-8192 // HY.decode_part_len(nd, G, 8192, waves)) == want


@pytest.mark.gpu
@pytest.mark.parametrize("rows,H,G", [(9, 16, 4), (600, 16, 16)])
def test_partitions_behind_short_contexts(rows, H, G):
    """Contexts of one to 70 keys in a step whose bound asks for many partitions (one for so many rows): a workspace of NaN shows that what no
    key fills is not read. Against the same rows without partitions, within the bound of test_partitions_match_one_walk."""
    gen = torch.Generator().manual_seed(rows)
    lens = [1 + (i * 23) % 70 for i in range(rows)]
    d = dict(device="cuda", dtype=torch.int32)
    tab = torch.zeros(rows, 512, **d)
    tab[:, :5] = torch.randint(0, 40, (rows, 5), generator=gen).to(**d)
    ctx = torch.tensor(lens, **d)
    rag = types.SimpleNamespace(n_dec=rows, n_pf=0, dec_bt=tab, dec_lens=ctx, dec_max_len=8192, positions=ctx - 1)
    q, kc, vc = (torch.randn(s, generator=gen).bfloat16().cuda() for s in ((rows, H * 64), (40, 16, G * 64), (40, 16, G * 64)))
    n = HY.partition_rows(rows, H, H // G)
    ws = torch.full((n, 2), float("nan"), device="cuda"), torch.full((n, 64), float("nan"), device="cuda")
    got, want, mag = (torch.empty(rows, H * 64, device="cuda", dtype=torch.bfloat16) for _ in range(3))
    for out, v, w in ((got, vc, ws), (want, vc, None), (mag, vc.abs(), None)):
        HY.masked_attention(q, kc, v, rag, H, G, 64, 64, 0.125, out, sink=True, workspace=w)
    assert ((got.float() - want.float()).abs() <= 2 ** -8 * want.float().abs() + 2 ** -8 * 1.02 * mag.float() + 1e-5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,dk,dv,chunk", [(32, 8, 128, 128, 2048), (16, 16, 64, 64, 0), (24, 2, 128, 64, 500)])
def test_partitions_match_one_walk(H, G, dk, dv, chunk):
    """Rows of one key, at a partition's and a mask chunk's edge and of many partitions, empty ones behind short contexts. Both sides round
    each weight to bf16 against their own running maximum, by at most 2^-9 of it: together 2^-8 of the weighted sum of |v|; fp32 sums in
    another order (1e-5); results to bf16 (one unit, 2^-8)."""
    lens = [1, 64, 65, 500, 501, 1999, 2049]
    gen = torch.Generator().manual_seed(H)
    W = 160
    n = sum(-(-x // 16) for x in lens)
    pages, tab, at = torch.randperm(n, generator=gen).tolist(), [], 0
    for x in lens:
        k = -(-x // 16)
        tab.append(pages[at:at + k] + [0] * (W - k))
        at += k
    d = dict(device="cuda", dtype=torch.int32)
    ctx = torch.tensor(lens, **d)
    rag = types.SimpleNamespace(n_dec=len(lens), n_pf=0, dec_bt=torch.tensor(tab, **d), dec_lens=ctx, dec_max_len=16 * W, positions=ctx - 1)
    q, kc, vc = (torch.randn(s, generator=gen).bfloat16().cuda() for s in ((len(lens), H * dk), (n, 16, G * dk), (n, 16, G * dv)))
    rows = HY.partition_rows(len(lens), H, H // G)
    ws = torch.full((rows, 2), float("nan"), device="cuda"), torch.full((rows, dv), float("nan"), device="cuda")
    got, want = (torch.empty(len(lens), H * dv, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    mag = torch.empty_like(want)
    for out, v, w in ((got, vc, ws), (want, vc, None), (mag, vc.abs(), None)):
        HY.masked_attention(q, kc, v, rag, H, G, dk, dv, dk ** -0.5, out, chunk=chunk, sink=True, workspace=w)
    assert not torch.isnan(ws[1][0]).all()  # (partitions were used)
    assert ((got.float() - want.float()).abs() <= 2 ** -8 * want.float().abs() + 2 ** -8 * 1.02 * mag.float() + 1e-5).all()
