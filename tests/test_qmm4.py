"""qmm4.hip: tiles of 128 to 224 rows x 256 columns of every format and epilogue, and the rule that takes untuned products to it."""
import numpy as np
import pytest
import torch

from localai_tfp_amd.formats.gguf import QType
from localai_tfp_amd.ops import autotune as A
from localai_tfp_amd.ops import linear as L
from localai_tfp_amd.ops import quant as Q

FORMATS = [QType.Q4_K, QType.Q5_K, QType.Q6_K, QType.Q3_K, QType.Q2_K, QType.Q8_0, QType.Q4_1, QType.Q5_1]


def test_row_tiles_the_rule_asks_for():
    for qt, (top, step, _) in L._QMM4_TILES.items():
        qb, hb = L._STAGE_BYTES[qt]
        lds = lambda b: 4 * (b * 2048 + 8 * qb) + 16 * hb  # noqa: E731
        assert lds(top) <= 160 * 1024 and (top == 14 or lds(top + 1) > 160 * 1024 or top % step == 0 and step == 2 and lds(top + 2) > 160 * 1024)
        for m in (129, 257, 416, 1000, 2049, 8191):
            kind, nb, s = L._wide_best(m, 28672, 4096, qt)[1]
            assert kind == "q4" and 8 <= nb <= top and nb % step == 0 and s == 1


def test_rule_takes_wide_products_that_do_not_accumulate():
    q4, q6 = int(QType.Q4_K), int(QType.Q6_K)
    pick = lambda m, n, k, qt=q4, glu=True: L._wide_plan(L._gemm_pick(m, n, k, qt, False), m, n, k, qt, False, glu)[0]  # noqa: E731
    assert pick(416, 28672, 4096) == pick(700, 28672, 4096) == pick(1100, 57344, 8192, q6) == "q4"
    assert pick(200, 28672, 4096) != "q4" and pick(416, 6144, 4096, q4, False) == pick(700, 6144, 4096, q4, False) == "q2"
    x16 = L._expanded_plan(8191, 28672, 4096, q4, False, True)
    assert L._wide_plan(x16, 8191, 28672, 4096, q4, False, True) is x16
    W = L.QWeight(28672, 4096, q4, torch.empty(0))
    W.layout = "t32"
    kinds = {e: L._t32_plan(W, 700, e, False)[0] for e in (L.EPI_F32, L.EPI_BF16, L.EPI_SWIGLU, L.EPI_GEGLU, L.EPI_ADD_F32)}
    assert kinds.pop(L.EPI_ADD_F32) == "q2" and set(kinds.values()) == {"q4"}


def test_rule_splits_long_products():
    q4, q6 = int(QType.Q4_K), int(QType.Q6_K)
    for m in (513, 700, 1100, 1700, 8191):
        for n, k, qt in ((4096, 14336, q4), (4096, 14336, q6), (8192, 28672, q4), (5120, 13824, int(QType.Q5_K)), (32, 8192, q4)):
            p = L._parts_plan(m, n, k, qt)
            assert p is None or p[0] == "q4" and 2 <= p[2] <= k // 512 and 8 <= p[1] <= L._QMM4_TILES[qt][0] and p[2] * m * n <= L.QMM4_PARTS
    assert L._parts_plan(700, 4096, 14336, q4) and not L._parts_plan(512, 4096, 14336, q4) and not L._parts_plan(700, 4096, 4096, q4)
    for m in (128, 333, 416, 512):
        for c in (c for c in A.candidates(m, 4096, 14336, q6, True) if c[0] == "q4"):
            assert c[1] <= 12 and (c[2] == 1 or c[2] * m * 4096 <= L.QMM4_PARTS)
        assert all(c[2] == 1 for c in A.candidates(m, 4096, 14336, q6, False) if c[0] == "q4")
    W = L.QWeight(4096, 14336, q4, torch.empty(0))
    W.layout = "t32"
    assert L._t32_plan(W, 700, L.EPI_ADD_F32, False)[0] == L._t32_plan(W, 700, L.EPI_F32, True)[0] == "q4"
    assert L._t32_plan(W, 700, L.EPI_F32, False)[-1] == L._t32_plan(W, 700, L.EPI_BF16, False)[-1] == 1


@pytest.mark.gpu
@pytest.mark.parametrize("qt", FORMATS)
@pytest.mark.parametrize("M,nb,n,k,splits", [(1, 8, 32, 512, 2), (129, 14, 288, 1280, 2), (333, 12, 544, 2816, 11), (417, 14, 256, 2560, 9)])
def test_parts_of_k(qt, M, nb, n, k, splits):
    """Parts of one super-block and of several, a last part with fewer, fewer parts than asked for (9 of ten super-blocks: five of two), more than one turn
    of the sum's loads, columns past the last whole 256; outputs off 16 bytes; nothing outside the output changes."""
    raw = Q.random_quantized(np.random.default_rng(M + n), int(qt), n, k).reshape(n, -1)
    W = L.QWeight.from_ggml(raw, int(qt), n, k, "cuda", t32=True)
    dense = torch.from_numpy(Q.dequantize(raw.reshape(-1), int(qt), (k, n)).reshape(n, k).copy()).double()
    assert W.to_t32()
    x = (torch.randn(M, k, generator=torch.Generator().manual_seed(M)) * 0.5).half()
    old = torch.randn(M, n, generator=torch.Generator().manual_seed(M + 1))
    want = x.double() @ dense.t()
    for epi, zeroed in ((L.EPI_ADD_F32, False), (L.EPI_F32, True)):
        for off in (0, 1):
            buf = torch.full((M + 1, n + 4 + 3 * off), -7.0, device="cuda")
            out = buf[:M, off:off + n]
            out.copy_(old if epi == L.EPI_ADD_F32 else torch.zeros_like(old))
            L.run_plan(("q4", nb, splits), W, x.cuda(), epi, out, zeroed)
            got = out.cpu().double() - (old.double() if epi == L.EPI_ADD_F32 else 0)
            # weights are rounded to f16 once (2^-11), products and parts summed in fp32
            assert float((got - want).norm() / want.norm()) < 2 ** -10
            assert (buf[M:] == -7).all() and (buf[:, off + n:] == -7).all() and (not off or (buf[:, 0] == -7).all())


@pytest.mark.gpu
@pytest.mark.parametrize("qt", FORMATS)
@pytest.mark.parametrize("M,nb,n,k", [(1, 8, 32, 256), (129, 14, 288, 512), (208, 14, 256, 1024), (333, 12, 544, 512), (417, 14, 1056, 256)])
def test_qmm4(qt, M, nb, n, k):
    """One row, whole and partial 16-row blocks, every row tile's size, columns past the last whole 256, one super-block and several;
    outputs that allow the four-column stores and outputs that do not."""
    raw = Q.random_quantized(np.random.default_rng(M + n), int(qt), n, k).reshape(n, -1)
    W = L.QWeight.from_ggml(raw, int(qt), n, k, "cuda", t32=True)
    dense = torch.from_numpy(Q.dequantize(raw.reshape(-1), int(qt), (k, n)).reshape(n, k).copy()).double()
    assert W.to_t32()
    x = (torch.randn(M, k, generator=torch.Generator().manual_seed(M)) * 0.5).half()
    want = x.double() @ dense.t()
    y = want.view(M, -1, 2, 16)
    gated = {L.EPI_SWIGLU: torch.nn.functional.silu(y[:, :, 0]) * y[:, :, 1],
             L.EPI_GEGLU: torch.nn.functional.gelu(y[:, :, 0], approximate="tanh") * y[:, :, 1]}
    for epi, ref, dt in [(L.EPI_F32, want, torch.float32), (L.EPI_BF16, want, torch.float16),
                         *((e, g.reshape(M, -1), torch.float16) for e, g in gated.items())]:
        for off in (0, 1):  # off 1: rows start at 2- or 4-byte steps
            buf = torch.full((M, ref.shape[1] + 3 * off), -7.0, device="cuda", dtype=dt)
            out = buf[:, off:off + ref.shape[1]]
            L.run_plan(("q4", nb, 1), W, x.cuda(), epi, out, False)
            # weights are rounded to f16 once (2^-11), products summed in fp32, f16 outputs and gates rounded again
            assert float((out.cpu().double() - ref).norm() / ref.norm()) < (1 if dt == torch.float32 else 4) * 2 ** -10
            if off:
                assert (buf[:, 0] == -7).all() and (buf[:, ref.shape[1] + 1:] == -7).all()


@pytest.mark.gpu
def test_qmm4_refuses_what_it_does_not_do():
    raw = Q.random_quantized(np.random.default_rng(0), int(QType.Q4_K), 64, 256).reshape(64, -1)
    W = L.QWeight.from_ggml(raw, int(QType.Q4_K), 64, 256, "cuda", t32=True)
    assert W.to_t32()
    x = torch.zeros(8, 256, device="cuda", dtype=torch.float16)
    with pytest.raises(RuntimeError):
        L.run_plan(("q4", 8, 1), W, x, L.EPI_ADD_F32, torch.zeros(8, 64, device="cuda"), False)
    with pytest.raises(ValueError):
        L.run_plan(("q4", 8, 2), W, x, L.EPI_BF16, torch.zeros(8, 64, device="cuda", dtype=torch.float16), False)
