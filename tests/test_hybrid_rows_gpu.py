"""Kernels of the hybrid decoders (csrc/kernels/hybrid: the recurrence, gated units, convolutions) on the GPU against the same
steps on the CPU."""
import types

import pytest
import torch

from localai_tfp_amd.ops import hybrid as HY

pytestmark = pytest.mark.gpu


def _rag(n_dec, chunks, at, slots, dev):
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)  # noqa: E731
    cu = [0]
    for c in chunks:
        cu.append(cu[-1] + c)
    pos = [p for p, c in zip(at, [1] * n_dec + chunks) for p in range(p, p + c)]
    return HY.Ragged(types.SimpleNamespace(
        T=len(pos), n_decode=n_dec, positions=i32(pos), seq_state=i32(slots), slots=i32([-1] * len(pos)), pf_cu_q=i32(cu),
        pf_q_lens_host=chunks, pf_ctx_lens_host=[p + c for p, c in zip(at[n_dec:], chunks)], pf_block_tables=None, pf_ctx_lens=None,
        dec_block_tables=None, dec_seq_lens=None, dec_max_len=0))


@pytest.mark.parametrize("N,P", [(16, 64), (32, 5), (33, 16), (64, 17), (128, 16), (100, 33), (256, 20)])
@pytest.mark.parametrize("delta,channel,nout", [(True, False, False), (False, False, True), (False, True, False), (True, True, False)])
def test_rounds_of_tokens(N, P, delta, channel, nout):
    """Chunks that end just before, at and after a round of 8 or 16 tokens, beside decode rows, with and without padding of N.
    Both sides sum in fp32, in another order: a share of 2^-24 per step and term of sums whose terms shrink with the decay, some
    40 steps of up to 256 terms, stays below 2e-5 of the largest output."""
    g = torch.Generator().manual_seed(N)
    H, G, chunks = 2, 1, [1, 7, 8, 9, 15, 16, 17, 33, 48]
    n_dec, T = 2, 2 + sum(chunks)
    k = torch.randn(T, G * N, generator=g) * N ** -0.5
    q, v = torch.randn(T, G * N, generator=g), torch.randn(T, H * P, generator=g)
    decay = torch.rand(T, H * N if channel else H, generator=g)
    coef = torch.rand(T, H, generator=g)
    skip = None if delta or nout else torch.randn(H, generator=g)  # (no caller has a skip term beside a normaliser)
    slots = list(range(n_dec + len(chunks)))
    at = [3, 0] + [0, 5] * 5
    start = torch.randn(len(slots), H, P + nout, N, generator=g)
    got = {}
    for dev in ("cpu", "cuda"):
        state, out = start.clone().to(dev), torch.zeros(T, H * P, device=dev)
        no = torch.zeros(T, H, device=dev) if nout else None
        HY.state_scan(k.to(dev), q.to(dev), v.to(dev), decay.to(dev), coef.to(dev), None if skip is None else skip.to(dev), state,
                      _rag(n_dec, chunks, at[:len(slots)], slots, dev), out, H, G, N, P, delta, channel, 0.5, False, no)
        got[dev] = [t.cpu() for t in (out, state, no) if t is not None]
    for a, b in zip(got["cuda"], got["cpu"]):
        assert (a - b).abs().max() <= 2e-5 * b.abs().max()


@pytest.mark.parametrize("H,N,P,n_dec,chunks", [(2, 128, 20, 0, [1]), (2, 128, 20, 3, [2, 9, 1]), (2, 64, 33, 1, [3]), (2, 64, 33, 0, [4]),
                                                (3, 32, 70, 2, [1] * 6 + [11]), (2, 200, 17, 0, [12, 12]), (16, 128, 64, 64, [37]),
                                                (16, 128, 64, 64, [3]), (8, 256, 128, 70, [20, 0, 30])])
@pytest.mark.parametrize("delta,channel", [(True, False), (False, True), (True, True)])
def test_short_chunks_and_rows_apart(H, N, P, n_dec, chunks, delta, channel):
    """Chunks that step token by token, whole or among longer ones, and decode rows that run as a launch of their own; the bound of
    test_rounds_of_tokens."""
    g = torch.Generator().manual_seed(N + n_dec)
    T, slots = n_dec + sum(chunks), list(range(n_dec + len(chunks)))[::-1]
    k, q, v = torch.randn(T, N, generator=g) * N ** -0.5, torch.randn(T, N, generator=g), torch.randn(T, H * P, generator=g)
    decay, coef = torch.rand(T, H * N if channel else H, generator=g), torch.rand(T, H, generator=g)
    at = [(i * 3) % 5 for i in range(len(slots))]
    start = torch.randn(len(slots), H, P, N, generator=g)
    got = {}
    for dev in ("cpu", "cuda"):
        state, out = start.clone().to(dev), torch.zeros(T, H * P, device=dev)
        HY.state_scan(k.to(dev), q.to(dev), v.to(dev), decay.to(dev), coef.to(dev), None, state, _rag(n_dec, chunks, at, slots, dev), out,
                      H, 1, N, P, delta, channel, 0.5, False, None)
        got[dev] = [out.cpu(), state.cpu()]
    for a, b in zip(got["cuda"], got["cpu"]):
        assert (a - b).abs().max() <= 2e-5 * b.abs().max()


@pytest.mark.parametrize("n_dec,chunks", [(1, [33, 16, 5, 40]), (2, [15, 9, 15, 8])])
@pytest.mark.parametrize("N,P", [(128, 64), (65, 64), (64, 130)])
@pytest.mark.parametrize("delta,channel", [(True, False), (False, True), (True, True)])
def test_rounds_of_full_grids(N, P, n_dec, chunks, delta, channel):
    """Grids of more workgroups than compute units, whose whole rounds run with the others in one body where decays are per channel, and chunks of
    less than a round each; the bound of test_rounds_of_tokens."""
    g = torch.Generator().manual_seed(N + n_dec)
    H, T, slots = 16, n_dec + sum(chunks), list(range(n_dec + len(chunks)))
    k, q, v = torch.randn(T, 2 * N, generator=g) * N ** -0.5, torch.randn(T, 2 * N, generator=g), torch.randn(T, H * P, generator=g)
    decay, coef = torch.rand(T, H * N if channel else H, generator=g), torch.rand(T, H, generator=g)
    at = [(i * 3) % 5 for i in range(len(slots))]
    start = torch.randn(len(slots), H, P, N, generator=g)
    got = {}
    for dev in ("cpu", "cuda"):
        state, out = start.clone().to(dev), torch.zeros(T, H * P, device=dev)
        HY.state_scan(k.to(dev), q.to(dev), v.to(dev), decay.to(dev), coef.to(dev), None, state, _rag(n_dec, chunks, at, slots, dev), out,
                      H, 2, N, P, delta, channel, 0.5, False, None)
        got[dev] = [out.cpu(), state.cpu()]
    for a, b in zip(got["cuda"], got["cpu"]):
        assert (a - b).abs().max() <= 2e-5 * b.abs().max()


@pytest.mark.parametrize("C,off", [(1, 0), (255, 0), (256, 1), (257, 0), (1023, 0), (1024, 1), (1025, 0), (2050, 3), (4098, 0), (4096, 0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_embedding_rows_of_any_width(C, off, dtype):
    """Widths around a workgroup's numbers, rows that lie on 16 bytes and not, tokens out of the table (row 0). A scale of 2 rounds nothing, and the
    sum with the old number is rounded once on either side: the same bits."""
    g = torch.Generator().manual_seed(C)
    table, ids = torch.randn(9, C, generator=g).to(dtype), torch.tensor([3, 8, 0, -1, 9, 3], dtype=torch.int32)
    old = torch.randn(6, C + off + 5, generator=g)
    want = table.float()[ids.where((ids >= 0) & (ids < 9), torch.zeros_like(ids)).long()] * 2
    for acc in (False, True):
        buf, o16 = old.clone().cuda(), torch.zeros(6, C + off + 3, dtype=torch.bfloat16, device="cuda")
        HY.embed_rows(table.cuda(), ids.cuda(), buf[:, off:off + C], accumulate=acc, out16=o16[:, off:off + C], scale=2.0)
        w = want + old[:, off:off + C] if acc else want
        assert torch.equal(buf[:, off:off + C].cpu(), w) and torch.equal(o16[:, off:off + C].cpu(), w.bfloat16())
        buf[:, off:off + C] = old[:, off:off + C].cuda()
        assert torch.equal(buf.cpu(), old) and not o16[:, :off].any() and not o16[:, off + C:].any()


@pytest.mark.parametrize("F,group,off", [(4, 4, 0), (260, 4, 0), (2048, 256, 0), (1023, 1023, 0), (1024, 2, 0), (1024, 1024, 1)])
@pytest.mark.parametrize("act", ["silu", "gelu_tanh", "relu2", "clamped", "gelu"])
def test_glu_widths(F, group, off, act):
    """Four elements a thread and one (odd widths, factor groups and offsets), fp32 and 16-bit out, with biases and factors of
    zero. A handful of fp32 operations and one function of a few units in the last place, whose arguments are sums of numbers up
    to ~10: 2e-5 of a result (or of 1); two such numbers may round to neighbouring bf16 numbers, 2^-7 of them apart."""
    g = torch.Generator().manual_seed(F)
    T = 5
    y = torch.randn(T, 2 * F + 16, generator=g) * 2
    ba, bb = torch.randn(F, generator=g), torch.randn(F, generator=g)
    scale = torch.rand(T, F // group, generator=g)
    scale[1] = 0.0
    two = act not in ("relu2", "gelu")
    res = {}
    for dev in ("cpu", "cuda"):
        z = y.to(dev)
        b = z[:, F + 8 + off:2 * F + 8 + off] if two else None
        for dt in (torch.float32, torch.bfloat16):
            out = torch.full((T, F + 8), 7.0, dtype=dt, device=dev)
            HY.glu(z[:, off:off + F], b, ba.to(dev), bb.to(dev) if two else None, out[:, off:off + F], scale=scale.to(dev),
                   group=group, act=act, **({"limit": 1.5, "alpha": 1.7} if act == "clamped" else {}))
            res[dev, dt] = out.float().cpu()
    a, b = res["cuda", torch.float32], res["cpu", torch.float32]
    assert ((a - b).abs() <= 2e-5 * (1 + b.abs())).all()
    a, b = res["cuda", torch.bfloat16], res["cpu", torch.bfloat16]
    assert ((a - b).abs() <= 2 ** -7 * b.abs() + 2e-5 * (1 + b.abs())).all()


@pytest.mark.parametrize("taps", [1, 2, 3, 4, 5])
def test_conv_blocks_of_rows(taps):
    """Chunks that end around a block of 16 rows, fresh and carried, beside decode rows: sums of up to five products in fp32."""
    g = torch.Generator().manual_seed(taps)
    C, chunks, n_dec = 70, [1, 2, 15, 16, 17, 33], 2
    T, slots = n_dec + sum(chunks), list(range(n_dec + len(chunks)))
    x, w, bias = torch.randn(T, C + 3, generator=g), torch.randn(C, taps, generator=g), torch.randn(C, generator=g)
    at = [4, 0, 0, 7, 0, 9, 0, 3]
    start = torch.randn(len(slots), max(1, taps - 1), C, generator=g)
    res = []
    for dev in ("cpu", "cuda"):
        tails, out = start.clone().to(dev), torch.zeros(T, C, device=dev)
        HY.causal_conv(x.to(dev)[:, 3:], w.to(dev), bias.to(dev), tails, _rag(n_dec, chunks, at, slots, dev), out, silu=True)
        res.append((out.cpu(), tails.cpu()))
    assert (res[0][0] - res[1][0]).abs().max() < 1e-5 and torch.equal(res[0][1], res[1][1])


@pytest.mark.parametrize("act", ["silu", "relu2", "clamped", "gelu"])
def test_glu_of_many_elements(act):
    """A million numbers and more run four elements a thread where widths and addresses allow it; the bound of test_glu_widths."""
    g = torch.Generator().manual_seed(2)
    T, F = 300, 4096
    a, b, sc = (torch.randn(T, n, generator=g) for n in (F + 1, F, F // 256))
    for off in (0, 1):
        for dt in (torch.float32, torch.bfloat16):
            got = {}
            for dev in ("cpu", "cuda"):
                out = torch.empty(T, F, dtype=dt, device=dev)
                HY.glu(a.to(dev)[:, off:off + F], None if act in HY.GLU_SINGLE else b.to(dev), None, None, out, sc.to(dev), 256, True, act, 2.0, 1.7)
                got[dev] = out.cpu().float()
            tol = 2e-5 if dt == torch.float32 else 2 ** -7
            assert ((got["cuda"] - got["cpu"]).abs() <= tol * got["cpu"].abs().clamp_min(1)).all()


@pytest.mark.parametrize("off", [0, 1])
def test_glu_biases_of_any_alignment(off):
    """Four elements a thread with biases that start on 16 bytes or not; the bound of test_glu_widths."""
    g = torch.Generator().manual_seed(off)
    T, F = 300, 4096
    a, b, bias = torch.randn(T, F, generator=g), torch.randn(T, F, generator=g), torch.randn(2 * F + 8, generator=g)
    for dt in (torch.float32, torch.bfloat16):
        got = {}
        for dev in ("cpu", "cuda"):
            out, d = torch.empty(T, F, dtype=dt, device=dev), bias.to(dev)
            HY.glu(a.to(dev), b.to(dev), d[off:off + F], d[F + 4 + off:2 * F + 4 + off], out)
            got[dev] = out.cpu().float()
        tol = 2e-5 if dt == torch.float32 else 2 ** -7
        assert ((got["cuda"] - got["cpu"]).abs() <= tol * got["cpu"].abs().clamp_min(1)).all()


@pytest.mark.parametrize("F", [257, 1028])
def test_glu_of_more_workgroups_than_a_grid_dimension(F):
    """Rows x chunks of a row beyond the 2^24 - 1 workgroups of 256 threads that a grid dimension holds, with one element a thread (odd
    widths) and with four: rows at both ends and where a second launch begins."""
    T = (1 << 23) + 5
    a, out = torch.full((T, F), 1.5, device="cuda"), torch.zeros(T, F, device="cuda", dtype=torch.bfloat16)
    at = torch.tensor([0, 1, (1 << 23) - 2, (1 << 23) - 1, 1 << 23, (1 << 23) + 1, T - 2, T - 1], device="cuda")
    x = torch.randn(len(at), F, generator=torch.Generator().manual_seed(F))
    a[at] = x.cuda()
    HY.glu(a, None, None, None, out, act="relu2")
    want = torch.relu(x).pow(2).bfloat16()
    assert torch.equal(out[at].cpu(), want) and bool((out[5:(1 << 23) - 5:4099] == 2.25).all())
    del a, out
    torch.cuda.empty_cache()


@pytest.mark.parametrize("H,G,Gv,dk,dv,rot,half", [(18, 3, 3, 64, 40, 64, False), (9, 8, 7, 100, 64, 36, True), (24, 0, 0, 32, 32, 0, False)])
def test_rotary_rows_of_many_heads(H, G, Gv, dk, dv, rot, half):
    """Steps of 32768 heads and more take eight heads a wave: head counts that leave a group part empty or mix queries with keys, partial
    rotation, rows without a slot. fp32 angles of positions below 3000 differ from fp32 of another order by 3000 * 2^-23 = 4e-4."""
    T, g = 1367, torch.Generator().manual_seed(H)
    q, k, v = torch.randn(T, H * dk, generator=g), torch.randn(T, max(G, 1) * dk, generator=g), torch.randn(T, max(Gv, 1) * dv, generator=g)
    pos = torch.randint(0, 3000, (T,), generator=g, dtype=torch.int32)
    slots = torch.randperm(T + 8, generator=g)[:T].to(torch.int32)
    slots[::7] = -1
    got = {}
    for dev in ("cpu", "cuda"):
        qo = torch.zeros(T, H * dk, device=dev)
        kc, vc = torch.zeros(T + 8, 1, max(G, 1) * dk, device=dev), torch.zeros(T + 8, 1, max(Gv, 1) * dv, device=dev)
        HY.rope_norm_append(q.to(dev), k.to(dev) if G else None, v.to(dev) if G else None, pos.to(dev), H, G, dk, dv, rot, 1e4, True, 1e-6, qo,
                            kc if G else None, vc if G else None, slots.to(dev), half=half, v_heads=Gv, q_temp=(0.1, 100))
        got[dev] = [t.cpu() for t in (qo, kc, vc)]
    for a, b in zip(got["cuda"], got["cpu"]):
        assert (a - b).abs().max() <= 1e-3 * max(1.0, float(b.abs().max()))


@pytest.mark.parametrize("dk", [130, 191, 192, 194, 256, 258, 383, 384, 386, 512])
def test_rotary_rows_of_wide_heads(dk):
    """Heads at the edges of three, four, six and eight numbers a lane: pairs of neighbours and of halves, whole and partial rotation,
    biases, rows without a slot; the bound of test_rotary_rows_of_many_heads."""
    T, H, G, g = 9, 3, 2, torch.Generator().manual_seed(dk)
    q, k, v = torch.randn(T, H * dk + 4, generator=g), torch.randn(T, G * dk, generator=g), torch.randn(T, G * dk, generator=g)
    bias, w = torch.randn((H + 2 * G) * dk, generator=g), torch.rand(2, dk, generator=g) + 0.5
    pos, slots = torch.randint(0, 3000, (T,), generator=g, dtype=torch.int32), torch.randperm(T + 3, generator=g)[:T].to(torch.int32)
    slots[3] = -1
    for rot, half, dt in ((dk // 2 * 2, False, torch.float32), (dk // 2 * 2, True, torch.bfloat16), (64, True, torch.float32), (0, False, torch.float32)):
        got = {}
        for dev in ("cpu", "cuda"):
            b, hw = bias.to(dev), w.to(dev)
            qo, kc, vc = torch.zeros(T, H * dk, device=dev, dtype=dt), torch.zeros(T + 3, 1, G * dk, device=dev, dtype=dt), torch.zeros(T + 3, 1, G * dk, device=dev, dtype=dt)
            HY.rope_norm_append(q.to(dev)[:, 4:], k.to(dev), v.to(dev), pos.to(dev), H, G, dk, dk, rot, 1e4, True, 1e-6, qo, kc, vc, slots.to(dev), q_weight=hw[0],
                                k_weight=hw[1], half=half, q_bias=b[:H * dk], k_bias=b[H * dk:(H + G) * dk], v_bias=b[(H + G) * dk:])
            got[dev] = [t.cpu().float() for t in (qo, kc, vc)]
        for a, b in zip(got["cuda"], got["cpu"]):
            assert (a - b).abs().max() <= (1e-3 if dt == torch.float32 else 2 ** -7) * max(1.0, float(b.abs().max()))


@pytest.mark.parametrize("T,H,dk", [(33, 8, 64), (33, 8, 128), (1300, 32, 128), (33, 4, 192), (33, 4, 512)])
def test_rotations_round_the_same_in_every_instance(T, H, dk):
    """x' = x c -+ round(y s) with one rounding of the sum, however many heads share a wave: c and s are read off unit vectors, the rest is
    float64 (the products of fp32 numbers are exact there; its own rounding can tip one fp32 rounding in 2^28)."""
    g = torch.Generator().manual_seed(dk + T)
    pos, slots = torch.randint(0, 3000, (T,), generator=g, dtype=torch.int32).cuda(), torch.zeros(T, dtype=torch.int32, device="cuda")

    def turn(x):
        out = torch.zeros(T, H * dk, device="cuda")
        HY.rope_norm_append(x.cuda(), None, None, pos, H, 0, dk, dk, dk, 1e4, False, 1e-6, out, None, None, slots)
        return out.cpu().view(T, H, dk // 2, 2)
    unit, x = torch.zeros(T, H * dk), torch.randn(T, H * dk, generator=g)
    unit[:, ::2] = 1.0
    cs = turn(unit).double()
    c, s = cs[..., 0], cs[..., 1]
    a, b = x.view(T, H, dk // 2, 2).double().unbind(-1)
    want = torch.stack([a * c - (b * s).float().double(), b * c + (a * s).float().double()], -1).float()
    assert (turn(x) != want).float().mean() < 1e-6


@pytest.mark.parametrize("chunk,window", [(0, 0), (128, 0), (0, 40)])
def test_chunks_of_many_sequences(chunk, window):
    """The chunks of a step are launched sixteen at a time, the longest first: eighteen sequences (with short ones between, which run on
    the row kernel) behind cached tokens, each as it is alone on the CPU. bf16 weights and outputs: 2^-8 of numbers of order 1."""
    H, G, D, bs = 4, 2, 64, 8
    lens = [16, 70, 3, 129, 64, 33, 17, 200, 16, 48, 1, 90, 20, 31, 66, 16, 130, 25, 80, 40]
    pre = [5 * i % 37 for i in range(len(lens))]
    g, T = torch.Generator().manual_seed(3), sum(lens)
    need = [-(-(p + n) // bs) for p, n in zip(pre, lens)]
    order = torch.randperm(sum(need), generator=g).tolist()
    tables, at = torch.zeros(len(lens), max(need), dtype=torch.int32), 0
    for i, n in enumerate(need):
        tables[i, :n] = torch.tensor(order[at:at + n], dtype=torch.int32)
        at += n
    q = torch.randn(T, H * D, generator=g).bfloat16()
    kc, vc = (torch.randn(sum(need), bs, G * D, generator=g).bfloat16() for _ in range(2))
    cu = [sum(lens[:i]) for i in range(len(lens) + 1)]
    i32 = lambda x, dev: torch.tensor(x, dtype=torch.int32, device=dev)  # noqa: E731
    got = {}
    for dev in ("cpu", "cuda"):
        ctx = [p + n for p, n in zip(pre, lens)]
        rag = HY.Ragged(types.SimpleNamespace(T=T, n_decode=0, positions=i32([0] * T, dev), seq_state=None, slots=None, pf_cu_q=i32(cu, dev),
                                              pf_q_lens_host=lens, pf_ctx_lens_host=ctx, pf_block_tables=tables.to(dev), pf_ctx_lens=i32(ctx, dev),
                                              dec_block_tables=None, dec_seq_lens=None, dec_max_len=0))
        out = torch.zeros(T, H * D, device=dev, dtype=torch.bfloat16)
        HY.masked_attention(q.to(dev), kc.to(dev), vc.to(dev), rag, H, G, D, D, D ** -0.5, out, chunk=chunk, window=window)
        got[dev] = out.float().cpu()
    assert (got["cuda"] - got["cpu"]).abs().max() <= 2 ** -6 and (got["cuda"] - got["cpu"]).norm() <= 2 ** -8 * got["cpu"].norm()


@pytest.mark.parametrize("H,P,chunks", [(48, 64, [33, 16]), (49, 64, [20, 17]), (64, 64, [33, 16, 5, 40]), (7, 300, [15, 1, 31]), (8, 256, [40, 17, 8])])
@pytest.mark.parametrize("N", [65, 128])
@pytest.mark.parametrize("delta,channel", [(True, False), (False, True), (False, False), (True, True)])
def test_lanes_of_a_column(H, P, chunks, N, delta, channel):
    """Grids around the size where a column's numbers move from 32 lanes to 16 (384 blocks; 768 without delta rule and channel decays) and well beyond
    it; the bound of test_rounds_of_tokens."""
    g = torch.Generator().manual_seed(N + H)
    T, slots = 1 + sum(chunks), list(range(1 + len(chunks)))
    k, q, v = torch.randn(T, N, generator=g) * N ** -0.5, torch.randn(T, N, generator=g), torch.randn(T, H * P, generator=g)
    decay, coef = torch.rand(T, H * N if channel else H, generator=g), torch.rand(T, H, generator=g)
    at = [(i * 3) % 5 for i in range(len(slots))]
    start = torch.randn(len(slots), H, P, N, generator=g)
    got = {}
    for dev in ("cpu", "cuda"):
        state, out = start.clone().to(dev), torch.zeros(T, H * P, device=dev)
        HY.state_scan(k.to(dev), q.to(dev), v.to(dev), decay.to(dev), coef.to(dev), None, state, _rag(1, chunks, at, slots, dev), out,
                      H, 1, N, P, delta, channel, 0.5, False, None)
        got[dev] = [out.cpu(), state.cpu()]
    for a, b in zip(got["cuda"], got["cpu"]):
        assert (a - b).abs().max() <= 2e-5 * b.abs().max()


@pytest.mark.parametrize("lens,pre,H,G,D,bs,kw", [
    ([33], [0], 8, 2, 128, 16, {}), ([100, 17], [30, 283], 6, 2, 64, 10, dict(sink=True)), ([70], [430], 4, 4, 128, 16, dict(chunk=128, sink=True)),
    ([150], [250], 12, 1, 64, 16, dict(window=70)), ([64, 65, 16], [0, 135, 1], 32, 1, 128, 8, dict(window=33, softcap=5.0, sink="each")),
    ([200], [60], 3, 1, 128, 16, dict(chunk=50)), ([40, 0, 63], [0, 0, 65], 8, 8, 64, 16, dict(gate=1)),
    ([90], [0], 8, 4, 128, 16, dict(gate=128, softcap=20.0, dtype=torch.float32)), ([128, 129], [1, 62], 5, 1, 64, 4, dict(dtype=torch.float32))])
@pytest.mark.parametrize("off", [0, 1])
def test_chunks_on_key_tiles(lens, pre, H, G, D, bs, kw, off):
    """Query heads that fill a workgroup's columns and that do not, key counts around whole tiles, chunk borders and window edges inside a tile, pages
    that are no power of two, sinks, caps, gates, outputs that allow wide stores and that do not. bf16 weights (and outputs): 2^-8 of numbers of order 1."""
    g, T, kw = torch.Generator().manual_seed(D + H), sum(lens), dict(kw)
    dt = kw.pop("dtype", torch.bfloat16)
    need = [-(-(p + n) // bs) for p, n in zip(pre, lens)]
    order = torch.randperm(sum(need), generator=g).tolist()
    tables, at = torch.zeros(len(lens), max(need), dtype=torch.int32), 0
    for i, n in enumerate(need):
        tables[i, :n] = torch.tensor(order[at:at + n], dtype=torch.int32)
        at += n
    q = torch.randn(T, H * D, generator=g).bfloat16()
    kc, vc = (torch.randn(sum(need), bs, G * D, generator=g).bfloat16() for _ in range(2))
    if kw.get("sink") == "each":
        kw["sink"] = torch.randn(H, generator=g)
    if "gate" in kw:
        kw["gate"] = torch.randn(T, H * kw["gate"], generator=g)
    cu, ctx = [sum(lens[:i]) for i in range(len(lens) + 1)], [p + n for p, n in zip(pre, lens)]
    i32 = lambda x, dev: torch.tensor(x, dtype=torch.int32, device=dev)  # noqa: E731
    got = {}
    for dev in ("cpu", "cuda"):
        rag = HY.Ragged(types.SimpleNamespace(T=T, n_decode=0, positions=i32([0] * T, dev), seq_state=None, slots=None, pf_cu_q=i32(cu, dev),
                                              pf_q_lens_host=lens, pf_ctx_lens_host=ctx, pf_block_tables=tables.to(dev), pf_ctx_lens=i32(ctx, dev),
                                              dec_block_tables=None, dec_seq_lens=None, dec_max_len=0))
        # (the reference in fp32 throughout)
        x = [t.float() if dev == "cpu" else t.to(dev) for t in (q, kc, vc)]
        buf = torch.full((T + 1, H * D + 4 + 3 * off), 7.0, device=dev, dtype=torch.float32 if dev == "cpu" else dt)
        HY.masked_attention(*x, rag, H, G, D, D, D ** -0.5, buf[:T, off:off + H * D], out_scale=0.7,
                            **{k: v.to(dev) if torch.is_tensor(v) else v for k, v in kw.items()})
        got[dev] = buf[:T, off:off + H * D].float().cpu()
        assert (buf[T] == 7).all() and (buf[:, off + H * D:] == 7).all() and (not off or (buf[:, 0] == 7).all())
    assert (got["cuda"] - got["cpu"]).norm() <= 2 ** -8 * got["cpu"].norm() and (got["cuda"] - got["cpu"]).abs().max() <= 2 ** -6


@pytest.mark.parametrize("groups,group", [(3, 16), (5, 60), (2, 64), (3, 68), (16, 128), (1, 256), (2, 260), (1, 512), (3, 516), (1, 2048), (1, 2052), (2, 4096), (1, 4100), (1, 8192)])
@pytest.mark.parametrize("T,gate_first,act,den,dtype", [(33, True, "silu", False, torch.bfloat16), (5, False, "silu", True, torch.float32),
                                                       (7, False, "sigmoid", False, torch.bfloat16), (1, True, "sigmoid", True, torch.float32)])
def test_group_norms_of_quadruples(groups, group, T, gate_first, act, den, dtype):
    """Groups around each number of threads, rows whose groups end inside a block, weights of a group and of a row; aligned rows and rows a number off
    (the scalar form). fp32 sums of up to 8192 squares in another order: below 2^-17 of the result; bf16 outputs, of eight
    significant bits, round by up to half of 2^-7 of it more."""
    g, C = torch.Generator().manual_seed(group), groups * group
    y, gate = torch.randn(T, C, generator=g), 3 * torch.randn(T, C, generator=g)
    gate[0, :4] = torch.tensor([-200.0, 200.0, 0.0, -90.0])
    dn = dict(den=torch.randn(T, groups, generator=g), den_min=torch.rand(T, groups, generator=g) + 0.1, den_eps=1e-3) if den else {}
    for off in (0, 1):
        for wlen in (group, C):
            w = torch.rand(wlen, generator=g) + 0.5
            got = {}
            for dev in ("cpu", "cuda"):
                yb, gb = (torch.zeros(T, C + 8, device=dev) for _ in range(2))
                yb[:, off:off + C], gb[:, off:off + C] = y.to(dev), gate.to(dev)
                out = torch.full((T + 1, C + 8), 7.0, device=dev, dtype=torch.float32 if dev == "cpu" else dtype)
                HY.gated_group_norm(yb[:, off:off + C], gb[:, off:off + C], w.to(dev), 1e-6, group, out[:T, off:off + C], gate_first=gate_first, out_scale=0.7,
                                    act=act, **{k: v.to(dev) if torch.is_tensor(v) else v for k, v in dn.items()})
                got[dev] = out[:T, off:off + C].float().cpu()
                assert (out[T] == 7).all() and (out[:, off + C:] == 7).all() and (not off or (out[:, 0] == 7).all())
            bound = 2 ** -17 + (2 ** -8 if dtype == torch.bfloat16 else 0)
            assert ((got["cuda"] - got["cpu"]).abs() <= bound * got["cpu"].abs() + 1e-7).all()
