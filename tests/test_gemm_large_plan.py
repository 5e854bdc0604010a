"""GEMM plans beyond the autotuner's buckets (ops/linear.py _large_plan) and the banded tile order they run in."""
import pytest
import torch

from localai_tfp_amd.formats.gguf import QType
from localai_tfp_amd.ops import linear as L
from localai_tfp_amd.ops import quant as Q

QTYPES = [QType.Q4_K, QType.Q5_K, QType.Q6_K, QType.Q3_K, QType.Q2_K, QType.Q8_0]


def test_plans_are_compiled_tiles():
    for qt in L._STAGE_BYTES:
        for m in (513, 640, 1000, 2049, 8191, 40000):
            for n, k in ((32, 256), (1024, 4096), (4096, 14336), (28672, 4096), (2080, 512)):
                for split in (False, True):
                    kind, wm, ks, wn, s = L._gemm_pick(m, n, k, qt, split)
                    assert kind == "q2" and (wm, ks, wn) in L.QMM2_CONFIGS and s in (1, 2, 4)
                    assert s == 1 or (split and (k // 256) // s >= 2)
                    assert not (ks == 17 and wm == 7 and qt not in (int(QType.Q4_K), int(QType.Q2_K), int(QType.MX4F)))
                    assert not (ks == 17 and wm >= 6 and qt == int(QType.Q8_0))


@pytest.mark.gpu
@pytest.mark.parametrize("qt", QTYPES)
@pytest.mark.parametrize("M,n", [(513, 32), (769, 416), (1025, 1056), (2100, 288)])
def test_large_plan_product(qt, M, n):
    """Whole and partial bands of row tiles, tails of rows and columns, plans that split K and plans that do not."""
    import numpy as np
    k = 1536
    raw = Q.random_quantized(np.random.default_rng(M + n), int(qt), n, k).reshape(n, -1)
    W = L.QWeight.from_ggml(raw, int(qt), n, k, "cuda", t32=True)
    dense = torch.from_numpy(Q.dequantize(raw.reshape(-1), int(qt), (k, n)).reshape(n, k).copy())
    assert W.to_t32()
    x = (torch.randn(M, k, generator=torch.Generator().manual_seed(1)) * 0.5).half()
    want = x.double() @ dense.double().t()
    for zeroed in (False, True):
        out = torch.zeros(M, n, device="cuda")
        L.qmatmul(W, x.cuda(), L.EPI_F32, out, out_zeroed=zeroed)
        # weights are rounded to f16 once (2^-11), products summed in fp32
        assert float((out.cpu().double() - want).norm() / want.norm()) < 2 ** -10
    act = torch.zeros(M, n // 2, device="cuda", dtype=torch.float16)
    L.qmatmul(W, x.cuda(), L.EPI_SWIGLU, act)
    y = want.view(M, -1, 2, 16)
    g = (torch.nn.functional.silu(y[:, :, 0]) * y[:, :, 1]).reshape(M, -1)
    assert float((act.cpu().double() - g).norm() / g.norm()) < 4 * 2 ** -10


def test_real_shapes_pick_every_tile():
    """What the products below force is what shapes of models ask for."""
    shapes = ((1024, 4096), (4096, 4096), (6144, 4096), (28672, 4096), (4096, 14336), (1536, 8960), (14336, 8192), (57344, 8192))
    picks = {L._gemm_pick(m, n, k, int(QType.Q4_K), split) for m in range(513, 8192, 113) for n, k in shapes for split in (False, True)}
    assert {p[1:4] for p in picks} == {t[:3] for t in L._LARGE_TILES} and {p[4] for p in picks} >= {1, 2, 4}


def test_square_tile_stays_where_the_estimate_is_too_close():
    pick = lambda m, n, k: L._gemm_pick(m, n, k, int(QType.Q4_K), True)  # noqa: E731
    assert pick(1024, 1536, 8960) == ("q2", 4, 2, 1, 2) and pick(520, 1536, 8960) == ("q2", 4, 2, 1, 4)
    assert pick(8191, 28672, 4096)[1:4] == (6, 17, 1) and pick(1024, 1024, 4096)[1:4] == (2, 2, 1)


_WEIGHTS = {}


def _weight(qt, n, k):
    """(weight on the GPU, its numbers) of a format; Q4_0 / Q5_0 / Q5_1 files load as MX4F / MX5F."""
    import numpy as np
    if qt not in _WEIGHTS:
        raw = Q.random_quantized(np.random.default_rng(n), int(qt), n, k).reshape(n, -1)
        W = L.QWeight.from_ggml(raw, int(qt), n, k, "cuda", t32=True)
        assert W.to_t32() and int(W.qtype) in L._STAGE_BYTES
        _WEIGHTS[qt] = W, torch.from_numpy(Q.dequantize(raw.reshape(-1), int(qt), (k, n)).reshape(n, k).copy())
    return _WEIGHTS[qt]


@pytest.mark.gpu
@pytest.mark.parametrize("qt", [*QTYPES, QType.Q4_0, QType.Q5_0, QType.Q5_1])
@pytest.mark.parametrize("tile", [t[:3] for t in L._LARGE_TILES])
def test_every_tile_in_bands(qt, tile):
    """Each tile the plans choose from, on five and six row tiles (a band of four and a partial one, its last tile part empty), two
    column panels of which the second is part empty, whole K and two and three parts of it."""
    n, k = 288, 1536
    W, dense = _weight(qt, n, k)
    wm, ks, wn = tile
    bm, ng = 32 * wm * wn, 8 if ks == 17 else 4
    qb, hb = L._STAGE_BYTES[int(W.qtype)]
    if 4 * (bm * 128 + ng * qb) + 2 * ng * hb > 160 * 1024:
        pytest.skip("this tile's ring does not fit the LDS for the format (never chosen)")
    for M in (4 * bm + 33, 6 * bm - 1):
        x = (torch.randn(M, k, generator=torch.Generator().manual_seed(M)) * 0.5).half()
        want = x.double() @ dense.double().t()
        base = torch.randn(M, n, generator=torch.Generator().manual_seed(1))
        for splits in (1, 2, 4):  # (six super-blocks: 4 asks for three parts of two)
            out = torch.zeros(M, n, device="cuda")
            L.run_plan(("q2", *tile, splits), W, x.cuda(), L.EPI_F32, out, True)
            assert float((out.cpu().double() - want).norm() / want.norm()) < 2 ** -10  # weights rounded to f16 once (2^-11)
            out = base.cuda()
            L.run_plan(("q2", *tile, splits), W, x.cuda(), L.EPI_ADD_F32, out, False)
            assert float((out.cpu().double() - base - want).norm() / want.norm()) < 2 ** -10
        act = torch.zeros(M, n // 2, device="cuda", dtype=torch.float16)
        L.run_plan(("q2", *tile, 1), W, x.cuda(), L.EPI_SWIGLU, act, False)
        y = want.view(M, -1, 2, 16)
        g = (torch.nn.functional.silu(y[:, :, 0]) * y[:, :, 1]).reshape(M, -1)
        assert float((act.cpu().double() - g).norm() / g.norm()) < 4 * 2 ** -10


def test_expanded_plans():
    """Weights are expanded where rows are many and the tiles fill the chip; the scratch is bounded and whole column tiles wide."""
    pick = lambda m, n, k, glu=False: L._expanded_plan(m, n, k, int(QType.Q4_K), not glu, glu)  # noqa: E731
    assert pick(8191, 28672, 4096, True)[0] == pick(8191, 4096, 14336)[0] == "x16" and pick(2048, 4096, 14336) is None
    assert pick(8191, 1024, 4096) is None and pick(1100, 1024, 4096) is None
    kind, cols, plan = pick(8191, 57344, 8192, True)
    assert cols % 256 == 0 and 256 <= cols and cols * 8192 * 2 <= L.X16_SCRATCH and plan == L._large_plan(8191, 57344, 8192, int(QType.Q4_K), False)


def test_expanded_plans_count_rounds_by_piece():
    """Weights of more than the scratch are multiplied piece by piece: where a piece leaves half the chip idle, the quantised plan."""
    pick = lambda m, n, k, glu, qt: L._expanded_plan(m, n, k, int(qt), not glu, glu)  # noqa: E731
    for qt in (QType.Q4_K, QType.Q3_K, QType.Q2_K, QType.Q5_K, QType.Q8_0, QType.MX4F):
        assert pick(1800, 8192, 28672, False, qt) is None and pick(2048, 8192, 28672, False, qt) is None
        assert pick(8191, 8192, 28672, False, qt)[0] == pick(4096, 57344, 8192, True, qt)[0] == pick(8191, 28672, 4096, True, qt)[0] == "x16"
    assert pick(2304, 57344, 8192, True, QType.Q4_K) is None and pick(4096, 8192, 28672, False, QType.Q4_K) is None


@pytest.mark.parametrize("switch", ["NORM_FUSE", "ROPE_FUSE"])
def test_fused_epilogues_keep_their_kernel(switch, monkeypatch):
    """The RMSNorm and rotation epilogues exist in qmm2 alone: with their switches few and many rows run it, tuned or not."""
    import types
    from localai_tfp_amd.ops import autotune as AT
    W = types.SimpleNamespace(N=4096, K=4096, qtype=int(QType.Q4_K), bf16_cache=None)
    plans = lambda: {L._t32_plan(W, m, L.EPI_ADD_F32, False)[0] for m in (5, 32, 128, 8191)}  # noqa: E731
    kinds = lambda: {p[0] for p in AT.candidates(32, 4096, 4096, int(QType.Q4_K), True)}  # noqa: E731
    assert plans() == {"qr", "q2", "x16"} and "qr" in kinds()
    monkeypatch.setattr(L, switch, True)
    assert plans() == {"q2"} and kinds() == {"q2", "q3"}


@pytest.mark.gpu
@pytest.mark.parametrize("qt", [*QTYPES, QType.Q4_0, QType.Q5_0, QType.Q5_1])
def test_expanded_products(qt):
    """gemm16.hip on expanded weights: part-empty tiles of rows and columns, three pieces of columns, every epilogue, rows that lie
    together and apart."""
    n, k = 288, 1536
    W, dense = _weight(qt, n, k)
    for M, cols in ((1, 512), (255, 256), (257, 256), (600, 32)):
        plan = ("x16", cols, ("q2", 4, 2, 1, 1))
        wide = (torch.randn(M, k + 8, generator=torch.Generator().manual_seed(M)) * 0.5).half()
        x, xd = wide[:, :k], wide[:, :k].cuda()
        want = x.double() @ dense.double().t()
        base = torch.randn(M, n, generator=torch.Generator().manual_seed(1))
        for rows in (xd.contiguous(), wide.cuda()[:, :k]):
            out = torch.full((M, n), 7.0, device="cuda")
            L.run_plan(plan, W, rows, L.EPI_F32, out, False)
            assert float((out.cpu().double() - want).norm() / want.norm()) < 2 ** -10  # weights rounded to f16 once (2^-11)
        out = base.cuda()
        L.run_plan(plan, W, xd, L.EPI_ADD_F32, out, False)
        assert float((out.cpu().double() - base - want).norm() / want.norm()) < 2 ** -10
        o16 = torch.zeros(M, n, device="cuda", dtype=torch.float16)
        L.run_plan(plan, W, xd, L.EPI_BF16, o16, False)
        assert float((o16.cpu().double() - want).norm() / want.norm()) < 2 * 2 ** -10
        y = want.view(M, -1, 2, 16)
        for epi, act in ((L.EPI_SWIGLU, torch.nn.functional.silu), (L.EPI_GEGLU, lambda z: torch.nn.functional.gelu(z, approximate="tanh"))):
            glu = torch.zeros(M, n // 2, device="cuda", dtype=torch.float16)
            L.run_plan(plan, W, xd, epi, glu, False)
            g = (act(y[:, :, 0]) * y[:, :, 1]).reshape(M, -1)
            assert float((glu.cpu().double() - g).norm() / g.norm()) < 4 * 2 ** -10


def test_few_rows_by_format():
    """Untuned products of up to 32 rows: the formats that decode slowest leave the register kernel where qmm2's K splits fill the chip
    or its workgroups make a second round; what measured faster there stays."""
    kind = lambda m, n, k, qt, split=False: L._gemm_pick(m, n, k, int(qt), split)[0]  # noqa: E731
    for m in (5, 9, 16, 32):
        for qt in (QType.Q6_K, QType.MX5F):
            assert kind(m, 4096, 14336, qt, True) == kind(m, 6144, 4096, qt, True) == kind(m, 8192, 28672, qt, True) == "q2"
            assert kind(m, 57344, 8192, qt) == kind(m, 128256, 4096, qt, True) == "q2"
            assert kind(m, 1024, 4096, qt, True) == kind(m, 2048, 2048, qt, True) == kind(m, 4096, 4096, qt) == "qr"
        assert kind(m, 28672, 4096, QType.Q6_K) == "qr" and kind(m, 28672, 4096, QType.MX5F) == "q2"
        for qt in (QType.Q4_K, QType.MX4F, QType.Q8_0):
            assert kind(m, 28672, 4096, qt) == kind(m, 57344, 8192, qt) == kind(m, 4096, 4096, qt, True) == "qr"
        assert kind(m, 8192, 28672, QType.Q8_0, True) == "qr" and kind(m, 8192, 28672, QType.Q4_K, True) == "q2"
        assert kind(m, 4096, 14336, QType.Q2_K, True) == "q2" and kind(m, 151936, 1536, QType.Q3_K, True) == "q2"
    assert kind(9, 6144, 4096, QType.Q3_K, True) == "q2" and kind(16, 6144, 4096, QType.Q3_K, True) == kind(9, 4096, 14336, QType.Q4_K, True) == "qr"
    assert kind(5, 3584, 3584, QType.Q6_K, True) == kind(16, 4096, 4096, QType.Q6_K, True) == "qr" and kind(5, 4096, 4096, QType.Q6_K, True) == "q2"
    assert kind(5, 14336, 1024, QType.MX4F, True) == "q2" and kind(12, 14336, 1024, QType.MX4F, True) == "qr"


def _launches(monkeypatch):
    """Names of the kernel entries called from here on."""
    names, call = [], L.N.kcall
    monkeypatch.setattr(L.N, "kcall", lambda name, *a: (names.append(name), call(name, *a))[1])
    return names


@pytest.mark.gpu
def test_expansion_is_not_captured(monkeypatch):
    """A captured step of more than 1024 rows (256 decode rows beside a chunk of 1024) runs the quantised plan and its graph keeps no
    scratch; replays give what the eager call of that plan gives."""
    qt, n, k, M = QType.Q4_K, 288, 1536, 1280  # (the size that the weights of this file are kept in)
    W, _ = _weight(qt, n, k)
    x = (torch.randn(M, k, generator=torch.Generator().manual_seed(3)) * 0.5).half().cuda()
    out, want, plan = torch.zeros(M, n, device="cuda"), torch.zeros(M, n, device="cuda"), ("x16", 512, ("q2", 4, 2, 1, 1))
    names = _launches(monkeypatch)
    L.run_plan(plan, W, x, L.EPI_F32, want, False)
    assert names == ["mxk_t32_expand", "mxk_gemm16"]
    L.run_plan(plan[2], W, x, L.EPI_F32, want, False)
    names.clear()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        L.run_plan(plan, W, x, L.EPI_F32, out, False)
    assert names == ["mxk_qmm2"]
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.gpu
@pytest.mark.parametrize("qt", [*QTYPES, QType.Q4_0, QType.Q5_0, QType.Q5_1])
def test_expanded_products_equal_the_wide_tiles(qt, monkeypatch):
    """gemm16.hip adds a sum's products in the order of qmm2's wide tiles (one wave through K) and rounds outputs where they do: every
    epilogue bit for bit. Five row tiles (a band of four and its rest) and three column tiles in one launch."""
    n, k, M = 768, 1536, 1100
    raw = Q.random_quantized(__import__("numpy").random.default_rng(5), int(qt), n, k).reshape(n, -1)
    W = L.QWeight.from_ggml(raw, int(qt), n, k, "cuda", t32=True)
    assert W.to_t32()
    x = (torch.randn(M, k, generator=torch.Generator().manual_seed(1)) * 0.5).half().cuda()
    base = torch.randn(M, n, generator=torch.Generator().manual_seed(2)).cuda()
    for epi in (L.EPI_F32, L.EPI_ADD_F32, L.EPI_BF16, L.EPI_SWIGLU, L.EPI_GEGLU):
        got = []
        for plan in (("q2", 4, 17, 1, 1), ("x16", n, None)):
            out = base.clone() if epi in (L.EPI_F32, L.EPI_ADD_F32) else torch.zeros(M, n // 2 if epi in L.GLU_EPIS else n, device="cuda", dtype=torch.float16)
            names = _launches(monkeypatch)
            L.run_plan(plan, W, x, epi, out, False)
            monkeypatch.undo()
            assert names == (["mxk_t32_expand", "mxk_gemm16"] if plan[0] == "x16" else ["mxk_qmm2"])
            got.append(out)
        assert torch.equal(*got), (epi, int((got[0] != got[1]).sum()))


@pytest.mark.gpu
def test_expansion_gives_way_to_the_quantised_plan(monkeypatch):
    """Outputs off 16 bytes or with rows off four numbers, rows that repeat, and no memory for the scratch run the qmm2 plan, with its
    results; activations off 16 bytes are refused, as qmm2 refuses them."""
    n, k, M = 288, 1536, 70
    W, dense = _weight(QType.Q4_K, n, k)
    x = (torch.randn(M, k, generator=torch.Generator().manual_seed(1)) * 0.5).half()
    want, plan = x.double() @ dense.double().t(), ("x16", 512, ("q2", 4, 2, 1, 1))

    def run(rows, epi, out, kernel, ref=want):
        names = _launches(monkeypatch)
        L.run_plan(plan, W, rows, epi, out, False)
        monkeypatch.undo()
        assert names[-1] == kernel and float((out.cpu().double() - ref).norm() / ref.norm()) < 2 * 2 ** -10
    for epi, dt in ((L.EPI_F32, torch.float32), (L.EPI_BF16, torch.float16)):
        for left, width, kernel in ((0, n, "mxk_gemm16"), (1, n + 3, "mxk_qmm2"), (0, n + 2, "mxk_qmm2"), (8, n + 8, "mxk_gemm16")):
            run(x.cuda(), epi, torch.zeros(M, width, device="cuda", dtype=dt)[:, left:left + n], kernel)
    run(x[:1].cuda().expand(M, k), L.EPI_F32, torch.zeros(M, n, device="cuda"), "mxk_qmm2", want[:1].expand(M, n))
    out, xd, empty = torch.zeros(M, n, device="cuda"), x.cuda(), torch.empty

    def full(*a, **kw):
        raise torch.cuda.OutOfMemoryError("none left")
    monkeypatch.setattr(torch, "empty", full)
    names = _launches(monkeypatch)
    L.run_plan(plan, W, xd, L.EPI_F32, out, False)
    monkeypatch.undo()
    assert torch.empty is empty and names == ["mxk_qmm2"] and float((out.cpu().double() - want).norm() / want.norm()) < 2 ** -10
    off = torch.zeros(M, k + 8, device="cuda", dtype=torch.float16)[:, 1:k + 1]
    for p in (plan, plan[2]):
        with pytest.raises(L.N.NativeError):
            L.run_plan(p, W, off, L.EPI_F32, out, False)
