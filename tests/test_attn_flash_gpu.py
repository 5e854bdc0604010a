"""Prompt attention of csrc/kernels/attention_flash.hip against the fp32 reference, at the edges of its query blocks, key
tiles and key parts, and the plan that chooses it (ops/core.py flash_plan)."""
import math

import numpy as np
import pytest
import torch

from localai_tfp_amd import _native as N
from localai_tfp_amd.ops import core as K
from localai_tfp_amd.ops import kvq as KQ


def _case(Hq, Hkv, D, q_lens, pre, bs=16, fmt="bf16", seed=0):
    g = torch.Generator().manual_seed(seed)
    ctx = [a + b for a, b in zip(q_lens, pre)]
    nb = sum(-(-c // bs) for c in ctx) + 2
    ids = (torch.randperm(nb - 1, generator=g) + 1).tolist()
    bt = torch.zeros(len(ctx), max(1, max(-(-c // bs) for c in ctx)), dtype=torch.int32)
    for s, c in enumerate(ctx):
        n = -(-c // bs)
        bt[s, :n] = torch.tensor(ids[:n], dtype=torch.int32)
        ids = ids[n:]
    kc, vc = (torch.randn(nb, Hkv, bs, D, generator=g) for _ in range(2))
    if fmt in KQ.FORMATS:
        f = KQ.FORMATS[fmt]
        kc, vc = (KQ.tag(torch.from_numpy(KQ.quantize_rows(t.reshape(-1, D), f)).view(nb, Hkv, bs, -1), f) for t in (kc, vc))
    else:
        kc, vc = (t.to(torch.float8_e4m3fn if fmt == "fp8" else torch.bfloat16) for t in (kc, vc))
    q = torch.randn(sum(q_lens), Hq, D, generator=g).to(torch.bfloat16)
    return q, kc, vc, bt, torch.tensor(np.concatenate([[0], np.cumsum(q_lens)]), dtype=torch.int32), torch.tensor(ctx, dtype=torch.int32)


def _check(Hq, Hkv, D, q_lens, pre, window=0, softcap=0.0, scale=None, plan=None, monkeypatch=None, tiles=False, **kw):
    q, kc, vc, bt, cu, ctx = _case(Hq, Hkv, D, q_lens, pre, **kw)
    scale = D ** -0.5 if scale is None else scale
    want = torch.zeros(q.shape)
    for s, n in enumerate(q_lens):
        if n:
            c, r = int(ctx[s]), slice(int(cu[s]), int(cu[s]) + n)
            want[r] = K._attn_ref_one(q[r], kc, vc, bt[s], c, c - n, scale, kc.shape[2], window, softcap).nan_to_num(0.0)
    if plan is not None:
        monkeypatch.setattr(K, "flash_plan", lambda *a, **k: plan)
    kd, vd = kc.cuda(), vc.cuda()
    if hasattr(kc, "kvf"):
        kd.kvf, vd.kvf = kc.kvf, vc.kvf
    out = torch.full(q.shape, float("nan"), dtype=torch.float16, device="cuda")
    if tiles:
        rows = N.kernels().mxk_attn_prefill_rows(Hq, Hkv)
        tiles = [torch.tensor(v + [-1], dtype=torch.int32).cuda() for v in K.prefill_tiles(q_lens, rows)]
        assert K.flash_plan(q.shape[0], len(q_lens), Hq, Hkv, D, kc.shape[2], bt.shape[1], window, ctx.tolist(), softcap, True) is None
    K.attn_prefill(q.cuda(), kd, vd, bt.cuda(), cu.cuda(), ctx.cuda(), scale, out, q_lens, ctx.tolist(), window=window, softcap=softcap,
                   tiles=tiles or None)
    got = out.cpu().float()
    # probabilities and outputs are rounded to 16 bits once each (2^-9, 2^-11): over a row of summed values the relative
    # error stays below 4 x 2^-9
    assert float((got - want).norm() / want.norm()) < 4 * 2 ** -9
    assert torch.isfinite(got).all()


def test_plan_takes_what_the_kernel_takes():
    p = K.flash_plan
    assert p(100, 1, 32, 8, 256, 16, 64, 0) is None and p(100, 1, 12, 4, 64, 16, 64, 0) is None  # the other kernel's / refused
    assert p(100, 1, 30, 8, 128, 16, 64, 0) is None
    assert p(333, 1, 32, 8, 128, 16, 512, 0, [333]) == (4, 1)  # known to be short: no parts
    assert p(333, 1, 32, 8, 128, 16, 512, 0) == (4, 5) and p(333, 1, 32, 8, 128, 16, 512, 0, []) == (4, 5)
    assert p(333, 1, 32, 8, 128, 16, 512, 256) == (4, 1)  # a window hides what lies further back
    assert p(8191, 1, 32, 8, 128, 16, 512, 0) == (8, 1) and p(8191, 1, 32, 8, 64, 16, 512, 0) == (4, 1)
    assert all(1 <= p(t, s, 8 * g, 8, 128, 16, 4096, 0)[1] <= 16 for t in (1, 17, 500, 4000) for s in (1, 9, 200) for g in (1, 2, 3, 5, 7, 8, 16))


def test_plan_of_short_contexts_and_of_many_sequences():
    """Known contexts of one key tile run the 16-row kernel where it is the faster one, and only where its tile lists are at hand; 8
    waves are for sequences that fill their blocks."""
    p = K.flash_plan
    one = lambda T, n, D, ctx, cap=0.0, tiles=True, H=32: p(T, n, H, 8, D, 16, 512, 0, [ctx] * n, cap, tiles)  # noqa: E731
    assert one(33, 1, 128, 33) is None and one(64, 64, 128, 1) is None and one(200, 200, 128, 1) is None and one(1000, 100, 128, 50) is None
    assert one(33, 1, 128, 33, tiles=False) == (4, 1) and one(33, 1, 128, 65) == (4, 1) and one(4000, 100, 128, 40) == (4, 1)
    assert one(17 * 64, 64, 128, 17) == (4, 1) and p(400, 400, 16, 1, 128, 16, 512, 0, [1] * 400, 0.0, True) == (4, 1)
    assert one(33, 1, 64, 33) == (4, 1) and one(200, 200, 64, 1) is None and one(17 * 64, 64, 64, 17) == (4, 1)
    assert one(33, 1, 64, 33, 50.0) is None and one(100, 1, 128, 100, 50.0) == (4, 1) and one(4000, 100, 128, 40, 50.0) == (4, 1)
    assert one(17 * 64, 64, 128, 500) == (4, 1) and one(8000, 16, 128, 500) == (4, 1)  # (8 waves: 1.6 times as long)
    assert p(100, 1, 32, 8, 128, 16, 4, 0, None, 0.0, True) is None  # (tables of 64 keys are a bound too)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["bf16", "fp8", "q8_0", "q4_0", "q4_1", "q5_0", "q5_1", "iq4_nl"])
@pytest.mark.parametrize("Hq,Hkv,D", [(32, 8, 128), (8, 8, 128), (6, 2, 128), (28, 4, 128), (16, 1, 128), (32, 8, 64), (4, 2, 64), (8, 1, 64)])
def test_short_contexts_on_the_row_kernel(fmt, Hq, Hkv, D):
    _check(Hq, Hkv, D, [1, 15, 16, 0, 17, 33, 64], [0, 5, 48, 0, 20, 31, 0], softcap=50.0, tiles=True, fmt=fmt)
    if Hkv >= 8:  # a crowd of short sequences
        _check(Hq, Hkv, D, [i % 9 for i in range(120)], [(i * 7) % 50 for i in range(120)], tiles=True, fmt=fmt)


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,D", [(32, 8, 128), (8, 8, 128), (6, 2, 128), (28, 4, 128), (16, 1, 128), (32, 8, 64), (4, 2, 64), (40, 1, 128)])
def test_query_blocks_and_key_tiles(Hq, Hkv, D):
    """Blocks of queries and tiles of keys that end just before, at and after an edge; sequences without rows between others."""
    _check(Hq, Hkv, D, [1, 31, 0, 33, 64, 65, 0], [0, 33, 5, 31, 0, 63, 9])
    _check(Hq, Hkv, D, [130], [127], bs=24)  # pages that are no power of two


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 130])
def test_which_sequence_a_block_belongs_to(n, monkeypatch):
    """Up to 64 sequences are found by one scan over the lanes, more in rounds of 64; some have no rows."""
    _check(8, 2, 128, [(i * 7) % 45 for i in range(n)][::-1] if n > 1 else [40], [(i * 13) % 70 for i in range(n)], plan=(4, 1), monkeypatch=monkeypatch)


@pytest.mark.gpu
@pytest.mark.parametrize("waves,parts", [(4, 1), (8, 1), (4, 2), (8, 3), (4, 16)])
@pytest.mark.parametrize("D", [64, 128])
def test_key_parts(waves, parts, D, monkeypatch):
    """Sequences that one part finishes beside others that several share (parts hold 16 tiles of 64 keys, the last one what is left);
    contexts of 16 and 17 tiles."""
    _check(8, 2, D, [70, 5, 40], [1100, 0, 3000], plan=(waves, parts), monkeypatch=monkeypatch)
    _check(8, 2, D, [24, 24, 24], [1000, 1001, 1064], plan=(waves, parts), monkeypatch=monkeypatch)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["fp8", "q8_0", "q4_0", "q4_1", "q5_0", "q5_1", "iq4_nl"])
def test_cache_formats(fmt, monkeypatch):
    _check(8, 2, 128, [70, 33], [61, 1500], fmt=fmt)
    _check(8, 2, 64, [70, 33], [61, 1500], fmt=fmt, plan=(8, 2), monkeypatch=monkeypatch)


@pytest.mark.gpu
@pytest.mark.parametrize("window,softcap,scale", [(50, 0.0, None), (64, 0.0, None), (1, 0.0, None), (0, 20.0, None), (130, 30.0, None), (0, 0.0, -0.05)])
def test_windows_caps_and_scales(window, softcap, scale, monkeypatch):
    _check(8, 2, 128, [90, 40], [300, 0], window=window, softcap=softcap, scale=scale)
    _check(8, 2, 128, [90, 40], [3000, 0], window=window, softcap=softcap, scale=scale, plan=(4, 3), monkeypatch=monkeypatch)


@pytest.mark.gpu
@pytest.mark.parametrize("D,waves", [(128, 4), (128, 8), (64, 4), (64, 8)])
@pytest.mark.parametrize("bs", [4, 6, 8, 10, 24, 256, 5000])
@pytest.mark.parametrize("rise", [0.0, 40.0])
def test_pages_and_rising_scores(bs, D, waves, rise, monkeypatch):
    """Pages that hold the groups of rows a wave requests (4 of head dim 128, 8 of 64) and pages that cut them, over more tiles than one
    look-up covers (16, 32 or 64); slots behind the contexts are not numbers. rise: log2 by which the scores grow over a context, so
    that every tile finds a new maximum."""
    q, kc, vc, bt, cu, ctx = _case(8, 2, D, [70, 33], [4130, 61], bs=bs, seed=bs)
    free = torch.ones(kc.shape[0], bs, dtype=torch.bool)
    q[..., 0] = 1.0
    for i, c in enumerate(ctx.tolist()):
        at = torch.arange(c)
        b, r = bt[i].long()[at // bs], at % bs
        free[b, r] = False
        kc[b, :, r, 0] = (at[:, None] / c * rise * math.log(2) * D ** 0.5).to(torch.bfloat16)
    for t in (kc, vc):
        t.transpose(1, 2)[free] = float("nan")
    want = torch.cat([K._attn_ref_one(q[int(cu[i]):int(cu[i + 1])], kc, vc, bt[i], int(c), int(c) - int(cu[i + 1] - cu[i]), D ** -0.5, bs)
                      for i, c in enumerate(ctx)])
    monkeypatch.setattr(K, "flash_plan", lambda *a, **k: (waves, 2))
    out = torch.full(q.shape, float("nan"), dtype=torch.float16, device="cuda")
    K.attn_prefill(q.cuda(), kc.cuda(), vc.cuda(), bt.cuda(), cu.cuda(), ctx.cuda(), D ** -0.5, out, [70, 33], ctx.tolist())
    # probabilities and outputs are rounded to 16 bits once each
    assert float((out.cpu().float() - want).norm() / want.norm()) < 4 * 2 ** -9


def test_plan_of_chunks_behind_long_contexts():
    """8 waves for one sequence's chunk of two blocks or more where 64 key tiles and four times its rows are known to lie before it, and 4 waves
    would share most compute units or leave parts longer; not where each would have a compute unit to itself."""
    p = lambda T, ctx, n=1, H=32, window=0: K.flash_plan(T, n, H, 8, 128, 16, 2048, window, ctx)  # noqa: E731
    assert p(416, [12416]) == (8, 4) and p(128, [12288]) == (8, 16) and p(1024, [4096]) == (8, 2) and p(2048, [14048]) == (8, 1)
    assert p(127, [4096])[0] == 4 and p(416, [4095])[0] == 4 and p(1025, [4096])[0] == 4 and p(2049, [14048])[0] == 4
    assert p(416, None)[0] == 4 and p(416, [12416] * 2, 2)[0] == 4 and p(416, [12416], window=512)[0] == 4
    assert p(64, [9000], H=64) == (8, 16) and p(63, [9000], H=64)[0] == 4
    assert p(128, [4096])[0] == p(256, [4352])[0] == p(200, [4300])[0] == 4 and p(512, [30512], H=64) == (8, 2)


@pytest.mark.gpu
@pytest.mark.parametrize("waves,parts", [(4, 1), (4, 2), (8, 1), (8, 2)])
@pytest.mark.parametrize("blocks", [[1], [2], [4], [1, 1], [1.0, 1.0, 0.0], [2.0, 0.0, 1.0, 0.0]])
def test_grids_hold_the_most_blocks_that_sequences_have(blocks, waves, parts, monkeypatch):
    """Whole blocks (given as whole numbers) and one row more of each (given as floats, 0.0 one row), which is the most blocks for their
    rows: every row is written."""
    rows = [int(b) * 8 * waves + isinstance(b, float) for b in blocks]
    _check(8, 2, 128, rows, [1100] * len(rows), plan=(waves, parts), monkeypatch=monkeypatch)


@pytest.mark.gpu
def test_infinite_scores_behave_like_the_reference():
    """A key of infinite score makes its row NaN, and no other row."""
    q, kc, vc, bt, cu, ctx = _case(4, 1, 128, [80], [0])
    kc[bt[0, 40 // 16], 0, 40 % 16] = float("inf")
    q[:, :, :] = q.abs() + 0.1
    out = torch.zeros(q.shape, dtype=torch.float16, device="cuda")
    K.attn_prefill(q.cuda(), kc.cuda(), vc.cuda(), bt.cuda(), cu.cuda(), ctx.cuda(), 1 / math.sqrt(128), out)
    got = out.cpu().float()
    assert torch.isfinite(got[:40]).all() and torch.isnan(got[40:]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["bf16", "fp8", "q8_0", "q4_0", "q4_1", "q5_0", "q5_1", "iq4_nl"])
@pytest.mark.parametrize("Hq,Hkv,D", [(32, 8, 128), (8, 1, 64), (6, 2, 128), (16, 1, 128)])
def test_decode_rows(fmt, Hq, Hkv, D):
    """One row per sequence: contexts around the 32-key tiles of a wave, the tiles of a workgroup and the partitions."""
    pre = [0, 31, 32, 33, 126, 127, 128, 512, 700, 1500]
    q, kc, vc, bt, _, ctx = _case(Hq, Hkv, D, [1] * len(pre), pre, fmt=fmt)
    want = torch.stack([K._attn_ref_one(q[i:i + 1], kc, vc, bt[i], int(c), int(c) - 1, D ** -0.5, 16)[0] for i, c in enumerate(ctx)])
    kd, vd = kc.cuda(), vc.cuda()
    if hasattr(kc, "kvf"):
        kd.kvf, vd.kvf = kc.kvf, vc.kvf
    for rows, part in ((slice(None), 256), (slice(None), 128), (slice(None), 1024), (slice(6, 10), 512), (slice(6, 10), 256)):
        out = torch.full((len(ctx[rows]), Hq, D), float("nan"), dtype=torch.float16, device="cuda")
        K.attn_decode(q[rows].cuda(), kd, vd, bt[rows].contiguous().cuda(), ctx[rows].cuda(), D ** -0.5, out, part_size=part)
        got = out.cpu().float()
        # as for prompts: probabilities and outputs are rounded to 16 bits once each
        assert float((got - want[rows]).norm() / want[rows].norm()) < 4 * 2 ** -9, part


@pytest.mark.gpu
@pytest.mark.parametrize("bs,part", [(24, 256), (48, 512), (20, 512), (640, 512), (3, 767)])
@pytest.mark.parametrize("fmt,impl", [("bf16", "mfma"), ("q8_0", "mfma"), ("fp8", "mfma"), ("bf16", "valu"), ("fp8", "valu")])
def test_decode_partitions_that_start_inside_a_page(bs, part, fmt, impl):
    """Pages that do not divide a partition: its keys reach into one page more than its length in pages says (24-key pages, 256
    keys from key 256 on: pages 10 .. 21). The last of (3, 767) is the 257th, the most that is listed."""
    pre = [0, part - 1, part, part + 1, 2 * part - 2, 2 * part - 1, 2 * part, 3 * part - 1, 3 * part + 7]
    q, kc, vc, bt, _, ctx = _case(8, 2, 128, [1] * len(pre), pre, bs=bs, fmt=fmt)
    want = torch.stack([K._attn_ref_one(q[i:i + 1], kc, vc, bt[i], int(c), int(c) - 1, 128 ** -0.5, bs)[0] for i, c in enumerate(ctx)])
    kd, vd = kc.cuda(), vc.cuda()
    if hasattr(kc, "kvf"):
        kd.kvf, vd.kvf = kc.kvf, vc.kvf
    for rows in (slice(None), slice(4, 9)):  # (few bf16 rows take more waves a workgroup)
        out = torch.full((len(ctx[rows]), 8, 128), float("nan"), dtype=torch.float16, device="cuda")
        K.attn_decode(q[rows].cuda(), kd, vd, bt[rows].contiguous().cuda(), ctx[rows].cuda(), 128 ** -0.5, out, part_size=part, impl=impl)
        got = out.cpu().float()
        # as for prompts: probabilities and outputs are rounded to 16 bits once each
        assert float((got - want[rows]).norm() / want[rows].norm()) < 4 * 2 ** -9


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["bf16", "fp8", "q8_0"])
@pytest.mark.parametrize("Hq,Hkv,D", [(8, 2, 128), (8, 1, 64)])
@pytest.mark.parametrize("window,softcap", [(0, 0.0), (0, 4.0), (50, 0.0)])
def test_decode_reads_nothing_behind_a_context(fmt, Hq, Hkv, D, window, softcap):
    """Slots of the pool that no context holds are not numbers, those of the last page behind it among them: the last tile's mask, with
    and without a cap, in every form (few rows take more waves a workgroup)."""
    pre = [0, 1, 30, 31, 32, 95, 127, 128, 200, 511, 700]
    q, kc, vc, bt, _, ctx = _case(Hq, Hkv, D, [1] * len(pre), pre, fmt=fmt)
    want = torch.stack([K._attn_ref_one(q[i:i + 1], kc, vc, bt[i], int(c), int(c) - 1, D ** -0.5, 16, window, softcap)[0] for i, c in enumerate(ctx)])
    free = torch.ones(kc.shape[0], 16, dtype=torch.bool)
    for i, c in enumerate(ctx.tolist()):
        at = torch.arange(c)
        free[bt[i].long()[at // 16], at % 16] = False
    assert free.any()
    for c in (kc, vc):
        rows = c.view(torch.uint8 if c.element_size() == 1 else torch.int16).permute(0, 2, 1, 3)
        rows[free] = -1 if c.element_size() == 2 else 255  # bf16, fp8 and f16 scales of all ones are not numbers
    kd, vd = kc.cuda(), vc.cuda()
    if hasattr(kc, "kvf"):
        kd.kvf, vd.kvf = kc.kvf, vc.kvf
    for rows, part in ((slice(None), 128), (slice(None), 256), (slice(None), 1024), (slice(5, 11), 512), (slice(5, 11), 256)):
        out = torch.full((len(ctx[rows]), Hq, D), float("nan"), dtype=torch.float16, device="cuda")
        K.attn_decode(q[rows].cuda(), kd, vd, bt[rows].contiguous().cuda(), ctx[rows].cuda(), D ** -0.5, out, part_size=part, window=window, softcap=softcap)
        # as for prompts: probabilities and outputs are rounded to 16 bits once each
        assert float((out.cpu().float() - want[rows]).norm() / want[rows].norm()) < 4 * 2 ** -9, part


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128, 256])
def test_decode_merges_any_number_of_partitions(D):
    """One more, as many and fewer than a group of the merge's threads asks for ahead (four each of 16, 8 or 4 groups), and more than have
    their weights in LDS."""
    parts = [1, 2, 3, 15, 16, 17, 31, 32, 33, 63, 64, 65, 511, 512, 520]
    q, kc, vc, bt, _, ctx = _case(4, 2, D, [1] * len(parts), [32 * n - 1 - n % 3 for n in parts])
    want = torch.stack([K._attn_ref_one(q[i:i + 1], kc, vc, bt[i], int(c), int(c) - 1, D ** -0.5, 16)[0] for i, c in enumerate(ctx)])
    out = torch.full(q.shape, float("nan"), dtype=torch.float16, device="cuda")
    K.attn_decode(q.cuda(), kc.cuda(), vc.cuda(), bt.cuda(), ctx.cuda(), D ** -0.5, out, part_size=32)
    # as for prompts: probabilities and outputs are rounded to 16 bits once each
    assert float((out.cpu().float() - want).norm() / want.norm()) < 4 * 2 ** -9
