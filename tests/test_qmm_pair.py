"""qmmp.hip: two weights of different block formats by the same rows in one launch (ops/linear.py qmatmul_pair)."""
import numpy as np
import pytest
import torch

from localai_tfp_amd.formats.gguf import QType
from localai_tfp_amd.ops import autotune as A
from localai_tfp_amd.ops import linear as L
from localai_tfp_amd.ops import quant as Q

PAIRS = [(QType.Q4_K, QType.Q6_K), (QType.Q5_K, QType.Q6_K), (QType.Q3_K, QType.Q5_K)]


def fake(n, k, qt):
    w = L.QWeight(n, k, int(qt), torch.empty(0))
    w.layout = "t32"
    return w


def test_rule_and_tuned_plans():
    a, b = fake(5120, 4096, QType.Q4_K), fake(1024, 4096, QType.Q6_K)
    for m in (5, 32, 64, 128, 333, 416, 512, 700, 4096):
        p = L._pair_plan(a, b, m)
        assert p is None or p[:-1] in L.PAIR_PLANS and (p[-1] == 1 or 4096 // 256 // p[-1] >= 2)
    assert L._pair_plan(a, b, 32) is not None and L._pair_plan(a, b, 416) is not None
    key = (5120, 1024, 4096, int(QType.Q4_K), int(QType.Q6_K))
    A.TUNED_PAIRS[key] = [(64, ("qr", 2, 2, 4, 1)), (128, ())]
    try:
        assert L._pair_plan(a, b, 40) == ("qr", 2, 2, 4, 1) and L._pair_plan(a, b, 100) is None and L._pair_plan(a, b, 300) is not None
    finally:
        del A.TUNED_PAIRS[key]
    assert not L.pair_ok((a, b)) and not L.pair_ok((a,))  # (not on a GPU)
    assert not L.qmatmul_pair((a, b), torch.zeros(8, 4096), torch.zeros(8, 6144))


def test_pairs_that_are_expanded():
    q4, q6 = int(QType.Q4_K), int(QType.Q6_K)
    take = lambda m, na=5120, nb=1024, k=4096: L._pair_expands(na, nb, k, q4, q6, m)  # noqa: E731
    assert take(8191) and take(5000) and not take(2600) and not take(L.X16_MIN_M - 1) and not take(512) and not take(1040)
    assert not take(8191, 32768, 8192) and take(8191, 9216, 1024, 8192)  # (scratch)


@pytest.mark.gpu
def test_expanded_pair(monkeypatch):
    """Both weights in one launch, rows and columns off its tiles, nothing outside; rows off 16 bytes run as they did."""
    M, na, nb, k = 300, 160, 96, 512
    ws, dense = [], []
    for i, (qt, n) in enumerate(zip(PAIRS[1], (na, nb))):
        raw = Q.random_quantized(np.random.default_rng(i), int(qt), n, k).reshape(n, -1)
        w = L.QWeight.from_ggml(raw, int(qt), n, k, "cuda", t32=True)
        assert w.to_t32()
        ws.append(w)
        dense.append(torch.from_numpy(Q.dequantize(raw.reshape(-1), int(qt), (k, n)).reshape(n, k).copy()).double())
    x = (torch.randn(M, k, generator=torch.Generator().manual_seed(M)) * 0.5).half()
    want = x.double() @ torch.cat(dense).t()
    monkeypatch.setattr(L, "_pair_expands", lambda *a: True)
    buf = torch.full((M + 1, na + nb + 8), -7.0, device="cuda")
    assert L.qmatmul_pair(ws, x.cuda(), buf[:M, :na + nb])
    # weights are rounded to f16 once (2^-11), products summed in fp32
    assert float((buf[:M, :na + nb].cpu().double() - want).norm() / want.norm()) < 2 ** -10
    assert (buf[M:] == -7).all() and (buf[:, na + nb:] == -7).all()
    off = torch.zeros(M, na + nb + 1, device="cuda")[:, 1:]
    assert not L._run_pair_x16(*ws, x.cuda(), off) and L.qmatmul_pair(ws, x.cuda(), off)
    assert float((off.cpu().double() - want).norm() / want.norm()) < 2 ** -10


@pytest.mark.gpu
@pytest.mark.parametrize("pair", PAIRS)
@pytest.mark.parametrize("M", [5, 33, 64, 129, 300])
@pytest.mark.parametrize("na,nb,k", [(160, 32, 256), (416, 96, 1536)])
def test_pair_product(pair, M, na, nb, k):
    """Every plan: rows, columns and super-blocks off the tiles' edges, workgroups of the second weight that are no whole eight, splits of K."""
    ws, dense = [], []
    for i, (qt, n) in enumerate(zip(pair, (na, nb))):
        raw = Q.random_quantized(np.random.default_rng(7 * M + i), int(qt), n, k).reshape(n, -1)
        w = L.QWeight.from_ggml(raw, int(qt), n, k, "cuda", t32=True)
        assert w.to_t32()
        ws.append(w)
        dense.append(torch.from_numpy(Q.dequantize(raw.reshape(-1), int(qt), (k, n)).reshape(n, k).copy()).double())
    assert L.pair_ok(ws)
    x = (torch.randn(M, k, generator=torch.Generator().manual_seed(M)) * 0.5).half()
    want = x.double() @ torch.cat(dense).t()
    for plan in L.PAIR_PLANS:
        for splits in (1, 2, 3):
            buf = torch.zeros(M + 1, na + nb + 8, device="cuda")
            buf[M:] = buf[:, na + nb:] = -7.0
            L.run_pair((*plan, splits), *ws, x.cuda(), buf[:M, :na + nb])
            # weights are rounded to f16 once (2^-11), products summed in fp32
            assert float((buf[:M, :na + nb].cpu().double() - want).norm() / want.norm()) < 2 ** -10, (plan, splits)
            assert (buf[M:] == -7).all() and (buf[:, na + nb:] == -7).all()
    out = torch.zeros(M, na + nb, device="cuda")
    took = L.qmatmul_pair(ws, x.cuda(), out)
    assert took == (L._pair_plan(*ws, M) is not None)
    if took:
        assert float((out.cpu().double() - want).norm() / want.norm()) < 2 ** -10
