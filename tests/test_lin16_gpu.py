"""Products of a few 16-bit rows (csrc/kernels/lin16.hip) and the rule that chooses them (ops/dense.py)."""
import types

import pytest
import torch

from localai_tfp_amd.ops import dense as D


def test_rule():
    p = D.few_rows_parts
    assert p(1, 4096, 17408) == p(64, 4096, 20480) == 4 and p(33, 2048, 20480) == 8 and p(8, 1024, 32768) == 8
    assert p(65, 4096, 20480) == p(33, 4096, 16384) == p(16, 5120, 20480) == p(0, 4096, 20480) == 0
    assert p(8, 28672, 4096) == 1 and p(9, 28672, 4096) == p(8, 16384, 4096) == 0
    assert p(4, 4000, 20480) == p(4, 4096, 20488) == 0
    assert all(0 <= p(m, n, k) <= 8 for m in (1, 64) for n in range(64, 4097, 64) for k in (16416, 40960))


def test_rule_leaves_the_library_what_it_does_better():
    p = D.few_rows_parts
    assert p(1, 24576, 2048) == p(8, 28672, 2304) == p(4, 32768, 4096) == 1
    assert p(1, 24576, 4096) == p(8, 32768, 5120) == p(1, 28672, 8192) == p(8, 51200, 1280) == p(1, 256000, 2304) == p(8, 41024, 4096) == 0
    assert p(32, 64, 65536) == p(64, 64, 32768) == 8 and p(33, 64, 65536) == 0 and p(64, 128, 65536) == 8


def test_route_takes_only_what_the_kernel_reads(monkeypatch):
    """What lin16.hip would read past, or from another device, stays with the library's product. On descriptions of tensors: no
    call may reach a kernel."""
    from localai_tfp_amd import _native as Nv
    calls = []
    monkeypatch.setattr(Nv, "kcall", lambda name, *a: calls.append((name, a)))
    monkeypatch.setattr(Nv, "stream_ptr", lambda: 0)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)

    def t(shape, strides=None, dev="cuda:0", dtype=torch.bfloat16, ptr=4096, grad=False):
        strides = strides or (shape[1], 1)
        return types.SimpleNamespace(shape=torch.Size(shape), dtype=dtype, device=torch.device(dev), is_cuda=dev != "cpu",
                                     requires_grad=grad, dim=lambda: len(shape), stride=lambda i: strides[i],
                                     data_ptr=lambda: ptr, is_contiguous=lambda: strides == (shape[1], 1))

    def route(x=None, w=None, out=None):
        calls.clear()
        took = D._few_rows(x or t((8, K)), w or t((N, K)), out or t((8, N), dtype=torch.float32), False)
        assert took == (len(calls) == 1)
        return took
    N, K = 28672, 4096
    assert route() and calls[0][1][1] == K
    assert route(x=t((8, K), (K + 16, 1))) and calls[0][1][1] == K + 16
    assert route(x=t((1, K), (0, 1)), out=t((1, N), dtype=torch.float32)) and calls[0][1][1] == K  # one row: no stride to follow
    for s in (0, 8, K - 8, K + 4):  # expanded rows, windows, rows of which every other is not 16-byte aligned
        assert not route(x=t((8, K), (s, 1)))
    assert not route(w=t((N, K), dev="cpu")) and not route(out=t((8, N), dtype=torch.float32, dev="cpu"))
    assert not route(w=t((N, K), dev="cuda:1")) and not route(w=t((N, K - 32))) and not route(w=t((N, K + 32)))
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    assert not route()
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    assert not route(x=t((8, K), grad=True)) and not route(out=t((8, N), dtype=torch.float32, grad=True))
    with torch.no_grad():
        assert route(x=t((8, K), grad=True))


@pytest.mark.gpu
def test_rows_that_overlap_match_the_library():
    g = torch.Generator().manual_seed(3)
    layer = D.Dense(torch.randn(64, 16416, generator=g) * 0.01, None, "cuda", torch.bfloat16)
    row = torch.randn(16416 + 7 * 8, generator=g).bfloat16().cuda()
    for x in (row[:16416].expand(8, 16416), row.unfold(0, 16416, 8)):
        want = x.double() @ layer.w.double().t()
        got = layer.into(x, torch.empty(8, 64, device="cuda"))
        mag = 16417 * 2 ** -24 * (x.double().abs() @ layer.w.double().abs().t())  # products exact, a sum of K terms in fp32
        assert ((got.double() - want).abs() <= mag).all()
        assert ((layer.acc(x, torch.zeros(8, 64, device="cuda")).double() - want).abs() <= mag).all()
    with pytest.raises(RuntimeError):
        D.Dense(layer.w.cpu(), None, "cpu", torch.bfloat16).into(row[:16416].expand(8, 16416), torch.empty(8, 64, device="cuda"))


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,parts", [(1, 64, 32, 1), (15, 68, 96, 2), (16, 128, 256, 8), (17, 64, 2080, 3), (33, 192, 20480, 4),
                                         (48, 4, 288, 1), (64, 100, 800, 5), (64, 64, 17408, 8)])
@pytest.mark.parametrize("acc", [False, True])
def test_few_rows_match_64_bits(dt, M, N, K, parts, acc):
    """Ends of row tiles, column panels and k-steps, parts without a step of their own, rows of x and y with room between them.
    Every product is exact in fp32 and a sum of K terms (and y) is off by at most (K + 1) x 2^-24 of the sum of magnitudes."""
    from localai_tfp_amd import _native as Nv
    g = torch.Generator().manual_seed(M + K)
    x = torch.randn(M, K + 8, generator=g).to(dt).cuda()[:, :K]
    w = torch.randn(N, K, generator=g).to(dt).cuda()
    y = torch.randn(M, N + 3, generator=g).cuda()
    xd, wd, yd = (t.double().cpu() for t in (x, w, y[:, :N]))
    want = xd @ wd.t() + (yd if acc else 0)
    mag = xd.abs() @ wd.abs().t() + yd.abs()
    rest = y[:, N:].clone()
    part = torch.full((parts, M, N), float("nan"), device="cuda")
    Nv.kcall("mxk_lin16", x.data_ptr(), x.stride(0), w.data_ptr(), y.data_ptr(), y.stride(0), part.data_ptr(), parts, M, N, K,
             int(dt == torch.float16), int(acc), Nv.stream_ptr())
    assert ((y[:, :N].double().cpu() - want).abs() <= (K + 1) * 2 ** -24 * mag).all() and torch.equal(y[:, N:], rest)


@pytest.mark.gpu
def test_dense_routes_few_rows(monkeypatch):
    """The layer's two entries on the routed shapes against the library's product: the same sums in another order."""
    g = torch.Generator().manual_seed(0)
    layer = D.Dense(torch.randn(256, 16416, generator=g) * 0.01, torch.randn(256, generator=g), "cuda", torch.bfloat16)
    plain = D.Dense(layer.w, None, "cuda", torch.bfloat16)
    x = torch.randn(33, 16416, generator=g).bfloat16().cuda()
    start = torch.randn(33, 256, generator=g).cuda()
    got = [layer.acc(x, start.clone()), plain.into(x, torch.empty(33, 256, device="cuda")), plain.acc(x, start.clone())]
    monkeypatch.setattr(D, "few_rows_parts", lambda *a: 0)
    want = [layer.acc(x, start.clone()), plain.into(x, torch.empty(33, 256, device="cuda")), plain.acc(x, start.clone())]
    mag = 2 * 16417 * 2 ** -24 * (x.double().abs().cpu() @ layer.w.double().abs().t().cpu() + 8)
    for a, b in zip(got, want):
        assert ((a.double() - b.double()).abs().cpu() <= mag).all()
    # a replayed graph allocates its parts once and sums them in the same order every time
    monkeypatch.undo()
    y = start.clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        plain.acc(x, y)
    torch.cuda.current_stream().wait_stream(s)
    gr = torch.cuda.CUDAGraph()
    with torch.cuda.graph(gr):
        plain.acc(x, y)
    for _ in range(3):
        y.copy_(start)
        gr.replay()
        assert torch.equal(y, got[2])
