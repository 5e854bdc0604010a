"""bf16 products by tiles (csrc/kernels/dense16.hip) and the rules that choose them and their tiles (ops/dense.py)."""
import pytest
import torch

from localai_tfp_amd.ops import dense as D

TILES = [(8, 8), (7, 8), (6, 8), (5, 8), (8, 6), (6, 6), (8, 4), (5, 4), (4, 4), (2, 8), (2, 4)]


def test_plans_are_within_what_the_kernel_takes():
    """Every plan: a tile that exists, whole tiles or parts for all, parts of plain tiles alone, of a k-tile at least, one round of them."""
    for M in (1, 33, 64, 65, 130, 257, 700, 1990, 4001, 70000):
        for N, K, F in ((4, 64, 0), (132, 320, 0), (4096, 20480, 0), (2048, 10240, 0), (128256, 4096, 0), (12320, 4096, 14336), (100, 512, 8200), (8, 4096, 30000)):
            mi, nj, whole, parts = D.dense16_plan(M, N, K, F)
            assert (mi, nj) in TILES and 1 <= parts <= max(1, K // 64)
            m, n, g = -(-M // (32 * mi)), -(-N // (32 * nj)), -(-2 * F // (32 * nj))
            rest = m * (n + g) - whole
            assert 0 <= rest <= m * n and rest * parts <= 256 if parts > 1 else rest == 0 or (parts == 1 and whole == 0 and not F)


def test_rules():
    t, g = D.takes_dense16, D.takes_gated16
    assert t(1, 4096, 20480) and t(3000, 4096, 18432) and t(64, 2048, 10240) and t(96, 1536, 9216) and t(33, 32000, 4096) and t(16, 25000, 5120)
    assert not (t(16, 2048, 10240) or t(80, 1536, 9216) or t(100, 4096, 4096) or t(65, 32000, 4096) or t(33, 25000, 5120) or t(8, 32000, 8192))
    assert not (t(8, 4096, 20512) or t(8, 4098, 20480) or t(0, 4096, 20480))
    assert g(1, 12320, 4096, 14336) and g(2000, 6176, 2048, 8192) and g(100, 1600, 1024, 2816)
    assert not (g(100, 352, 256, 512) or g(8, 1600, 1024, 2816) or g(8, 12320, 4096, 14338) or g(8, 12322, 4096, 14336) or g(0, 12320, 4096, 14336))


def test_rules_leave_to_others_what_they_are_faster_at():
    """Few rows by few columns, many columns by short K, large products of short K or one round of 192-column tiles, gated units that are the smaller part."""
    t, g = D.takes_dense16, D.takes_gated16
    assert t(40, 2048, 20480) and t(1, 3072, 20480) and t(9, 3072, 49152) and t(64, 1024, 16448) and t(96, 256, 65536) and t(900, 2048, 8192)
    assert not (t(39, 2048, 20480) or t(8, 3072, 49152) or t(64, 1024, 16384) or t(128, 128, 131072) or t(901, 2048, 8192) or t(1024, 1536, 8960))
    assert D.dense16_plan(1800, 5120, 13824)[:2] == (8, 6) and not t(1800, 5120, 13824) and t(1400, 5120, 13824) and t(4000, 5120, 13824)
    assert t(16, 100352, 1280) and t(64, 100352, 1536) and t(33, 32000, 576) and not (t(16, 100352, 1024) or t(17, 100352, 1280) or t(33, 32000, 512) or t(8, 32004, 1024))
    assert g(1, 4608, 3072, 6144) and g(65, 3840, 2560, 5120) and g(1001, 9216, 3072, 3072) and g(80, 4608, 1536, 1536)
    assert not (g(64, 3840, 2560, 5120) or g(1000, 9216, 3072, 3072) or g(65, 6144, 2048, 2048))


def _run(epi, tile, x, w, out, whole, parts, bias=None, gated=None):
    from localai_tfp_amd import _native as Nv
    M, K = x.shape
    tm, tn = 32 * tile[0], 32 * tile[1]
    F = gated[0] if gated else 0
    m, n = -(-M // tm), -(-out.shape[1] // tn)
    t = m * (n + -(-2 * F // tn))
    whole = t if parts == 1 else whole * m
    part = torch.full(((t - whole) * parts * tm * tn,), float("nan"), device="cuda") if parts > 1 else None
    g = (F, gated[1], gated[2], gated[3].data_ptr(), Nv.ptr(gated[4]), gated[5].data_ptr(), gated[5].stride(0)) if gated else (0, 0, 0, None, None, None, 0)
    Nv.kcall("mxk_dense16", epi, 16 * tile[0] + tile[1], x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), M, out.shape[1], K, Nv.ptr(bias), out.data_ptr(),
             out.stride(0), whole, parts, Nv.ptr(part), *g, Nv.stream_ptr())


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("acc", [False, True])
def test_tiles_match_64_bits(tile, acc):
    """One row short of, at and past a tile's rows, columns of a part-empty tile, one k-tile and rings that wrap, parts without and with
    whole tiles ahead, rows with room between them. Products are exact in fp32, a sum of K terms, the bias and the start are off by at
    most (K + 2) x 2^-24 of the sum of magnitudes."""
    tm, tn = 32 * tile[0], 32 * tile[1]
    gen = torch.Generator().manual_seed(tm + tn)
    for M, N, K, whole, parts in ((tm - 1, tn + 4, 64, 0, 1), (tm + 1, tn, 640, 0, 1), (1, 4, 1344, 0, 1), (tm, 2 * tn - 4, 320, 0, 3), (tm + 5, tn + 36, 832, 1, 5),
                                  (33, tn - 8, 64 * 21, 0, 8)):
        x = torch.randn(M, K + 8, generator=gen).bfloat16().cuda()[:, :K]
        w = torch.randn(N, K, generator=gen).bfloat16().cuda()
        b = torch.randn(N, generator=gen).cuda()
        y = torch.randn(M, N + 8, generator=gen).cuda()
        xd, wd = x.double(), w.double()
        start = y[:, :N].double() if acc else 0
        want, mag, rest = xd @ wd.t() + b.double() + start, xd.abs() @ wd.abs().t() + b.abs() + y[:, :N].abs(), y[:, N:].clone()
        _run(int(acc), tile, x, w, y[:, :N], whole, parts, b)
        assert ((y[:, :N].double() - want).abs() <= (K + 2) * 2 ** -24 * mag).all(), (tile, M, N, K)
        assert torch.equal(y[:, N:], rest)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
def test_gated_columns_match_64_bits(tile):
    """Features of part-empty tiles, gate and up rows apart from the plain ones, parts of the plain tiles, no bias on one side. g and u are
    off by d = (K + 1) x 2^-24 of their magnitudes; silu's slope is at most 1.1 and it is at most |g|: 1.1 dg |u| + du |g| + dg du, the unit's own fp32
    rounding (2^-20) and bf16's (2^-8 of the result)."""
    tm, tn = 32 * tile[0], 32 * tile[1]
    gen = torch.Generator().manual_seed(tm * tn)
    for M, n, F, K, whole, parts in ((tm + 1, 36, tn // 2 + 8, 576, 0, 1), (tm - 1, tn + 4, 24, 320, 1, 2), (3, 4, tn, 64, 0, 1)):
        x, w = torch.randn(M, K, generator=gen).bfloat16().cuda(), (torch.randn(n + 8 + 2 * F + 4, K, generator=gen) * K ** -0.5).bfloat16().cuda()
        gb, y, G = torch.randn(F, generator=gen).cuda(), torch.zeros(M, n, device="cuda"), torch.zeros(M, F + 16, device="cuda").bfloat16()
        gate, up = n + 8, n + 8 + F + 4
        _run(4, tile, x, w, y, whole and -(-2 * F // tn) + whole, parts, None, (F, gate, up, gb, None, G[:, 8:F + 8]))
        xd, wd, d = x.double(), w.double(), (K + 1) * 2 ** -24
        assert ((y.double() - xd @ wd[:n].t()).abs() <= d * (xd.abs() @ wd[:n].abs().t())).all()
        g, u = xd @ wd[gate:gate + F].t() + gb.double(), xd @ wd[up:up + F].t()
        dg, du = d * (xd.abs() @ wd[gate:gate + F].abs().t() + gb.abs()), d * (xd.abs() @ wd[up:up + F].abs().t())
        want = torch.nn.functional.silu(g) * u
        tol = 1.1 * dg * u.abs() + du * g.abs() + dg * du + (2 ** -8 + 2 ** -20) * want.abs() + 1e-30
        assert ((G[:, 8:F + 8].double() - want).abs() <= tol).all(), (tile, M, n, F, K)
        assert not G[:, :8].any() and not G[:, F + 8:].any()


@pytest.mark.gpu
def test_routes(monkeypatch):
    """The layer's entries take the kernel where the rules say, leave it operands that it cannot read as they lie, replay from a graph, and
    run whole tiles where the parts' room cannot be had."""
    from localai_tfp_amd import _native as Nv
    calls, real = [], Nv.kcall
    monkeypatch.setattr(Nv, "kcall", lambda name, *a: (calls.append((name, a)), real(name, *a))[1])
    gen = torch.Generator().manual_seed(1)
    layer = D.Dense(torch.randn(1024, 16448, generator=gen) * 0.01, torch.randn(1024, generator=gen), "cuda", torch.bfloat16)
    x, start = torch.randn(70, 16448, generator=gen).bfloat16().cuda(), torch.randn(70, 1024, generator=gen).cuda()
    want = start.double() + x.double() @ layer.w.double().t() + layer.b32.double()
    mag = (16448 + 2) * 2 ** -24 * (x.double().abs() @ layer.w.double().abs().t() + start.abs() + layer.b32.abs())

    def used():
        n = [c[0] for c in calls]
        calls.clear()
        return n
    got = layer.acc(x, start.clone())
    assert used() == ["mxk_dense16"] and ((got.double() - want).abs() <= mag).all()
    y = layer.into(x, torch.empty(70, 1024, device="cuda"))
    assert used() == ["mxk_dense16"] and ((y.double() + start.double() - want).abs() <= mag).all()
    wide = torch.zeros(70, 16456, device="cuda").bfloat16()
    odd = wide[:, 4:16452]
    odd.copy_(x)
    layer.into(odd, y)  # (rows off 16 bytes)
    assert used() == [] and ((y.double() + start.double() - want).abs() <= mag).all()
    with torch.enable_grad():
        layer.into(x, torch.empty(70, 1024, device="cuda").requires_grad_(False))
        assert used() == ["mxk_dense16"]
        assert not D._dense16(x.detach().requires_grad_(True), layer.w, torch.empty(70, 1024, device="cuda"), False, None) and used() == []
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    z, gr = start.clone(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(st):
        layer.acc(x, z)
    torch.cuda.current_stream().wait_stream(st)
    with torch.cuda.graph(gr):
        layer.acc(x, z)
    for _ in range(3):
        z.copy_(start)
        gr.replay()
        assert torch.equal(z, got)
    used()

    def refuse(*a, **k):
        raise torch.cuda.OutOfMemoryError("no room")
    with monkeypatch.context() as mp:
        z.copy_(start)
        mp.setattr(torch, "empty", refuse)
        layer.acc(x, z)
    assert calls[-1][1][13] == 1 and ((z.double() - want).abs() <= mag).all()
