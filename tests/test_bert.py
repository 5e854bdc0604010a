"""BERT embeddings / reranker backend: model numerics vs a plain fp32 PyTorch encoder, worker
micro-batching, and the HTTP surface (/v1/embeddings, /v1/rerank) — reference coverage:
core/http/app_test.go embeddings + rerank cases, backend/python/rerankers/test.py."""
import math

import numpy as np
import pytest
import torch
import yaml
from fastapi.testclient import TestClient

from localai_tfp_amd.config.app_config import ApplicationConfig
from localai_tfp_amd.gateway.app import create_app
from localai_tfp_amd.models import bert as BM


def _reference_encode(cfg, get, ids):
    """Straightforward fp32 BERT (post-LN) of one sequence."""
    t = lambda n: torch.from_numpy(get(n))  # noqa: E731
    S = len(ids)
    x = t("token_embd.weight")[ids] + t("position_embd.weight")[:S] + t("token_types.weight")[0]
    x = torch.nn.functional.layer_norm(x, (cfg.hidden,), t("token_embd_norm.weight"), t("token_embd_norm.bias"), cfg.eps)
    hd = cfg.hidden // cfg.n_heads
    for i in range(cfg.n_layers):
        p = f"blk.{i}."
        q, k, v = (x @ t(p + f"attn_{n}.weight").T + t(p + f"attn_{n}.bias") for n in "qkv")
        q, k, v = (z.view(S, cfg.n_heads, hd).transpose(0, 1) for z in (q, k, v))
        a = torch.softmax(q @ k.transpose(1, 2) / math.sqrt(hd), -1) @ v
        a = a.transpose(0, 1).reshape(S, cfg.hidden)
        o = a @ t(p + "attn_output.weight").T + t(p + "attn_output.bias")
        x = torch.nn.functional.layer_norm(x + o, (cfg.hidden,), t(p + "attn_output_norm.weight"),
                                           t(p + "attn_output_norm.bias"), cfg.eps)
        u = torch.nn.functional.gelu(x @ t(p + "ffn_up.weight").T + t(p + "ffn_up.bias"))
        d = u @ t(p + "ffn_down.weight").T + t(p + "ffn_down.bias")
        x = torch.nn.functional.layer_norm(x + d, (cfg.hidden,), t(p + "layer_output_norm.weight"),
                                           t(p + "layer_output_norm.bias"), cfg.eps)
    return x


def test_bert_matches_reference_and_padding_invariant():
    cfg = BM.BERT_TINY
    get = BM.synthetic_bert(cfg, 3)
    m = BM.BertModel.load(cfg, get, "cpu")
    seqs = [[2, 17, 40, 9, 3], [2, 50, 3]]
    hid, lens = m.encode(seqs)
    for b, s in enumerate(seqs):
        ref = _reference_encode(cfg, get, s)
        assert torch.allclose(hid[b, :len(s)], ref, atol=2e-4), (hid[b, :len(s)] - ref).abs().max()
    e = m.embed(seqs)
    e1 = m.embed([seqs[1]])
    assert torch.allclose(e[1], e1[0], atol=1e-5)
    assert torch.allclose(e.norm(dim=-1), torch.ones(2), atol=1e-5)


def test_worker_batches_and_reranks():
    from localai_tfp_amd.grpc import pb
    from localai_tfp_amd.workers.bert import BertServicer
    s = BertServicer(device="cpu")
    assert s.LoadModel(pb.ModelOptions(Model="synthetic:bert-tiny-rerank"), None).success
    import concurrent.futures as cf
    texts = [f"doc number {i}" for i in range(12)]
    with cf.ThreadPoolExecutor(8) as ex:
        embs = list(ex.map(lambda t: s.Embedding(pb.PredictOptions(Embeddings=t), None).embeddings, texts))
    solo = s.Embedding(pb.PredictOptions(Embeddings=texts[5]), None).embeddings
    assert max(abs(a - b) for a, b in zip(embs[5], solo)) < 1e-5
    r = s.Rerank(pb.RerankRequest(query="q", documents=["aa", "bbb", "c"], top_n=2), None)
    assert len(r.results) == 2 and r.results[0].relevance_score >= r.results[1].relevance_score
    assert r.usage.total_tokens > 0


@pytest.fixture(scope="module")
def client(tmp_path_factory):
    d = tmp_path_factory.mktemp("bert")
    models = d / "models"
    models.mkdir()
    (models / "emb.yaml").write_text(yaml.safe_dump({
        "name": "emb", "embeddings": True, "parameters": {"model": "synthetic:bert-tiny"}}))
    (models / "rr.yaml").write_text(yaml.safe_dump({
        "name": "rr", "backend": "rerankers", "parameters": {"model": "synthetic:bert-tiny-rerank"}}))
    cfg = ApplicationConfig(models_path=str(models), generated_content_dir=str(d / "gen"),
                            upload_dir=str(d / "up"), config_dir=str(d / "cfg"), api_keys=[])
    app = create_app(cfg, inproc=True)
    with TestClient(app) as c:
        yield c
    app.state.localai.shutdown()


def test_http_embeddings_and_rerank(client):
    r = client.post("/v1/embeddings", json={"model": "emb", "input": ["hello world", "goodbye"]})
    assert r.status_code == 200, r.text
    d = r.json()["data"]
    assert len(d) == 2 and len(d[0]["embedding"]) == BM.BERT_TINY.hidden
    assert abs(sum(x * x for x in d[0]["embedding"]) - 1) < 1e-4
    r = client.post("/v1/rerank", json={"model": "rr", "query": "what", "documents": ["x y", "z", "w w w"],
                                        "top_n": 3})
    assert r.status_code == 200, r.text
    j = r.json()
    assert sorted(x["index"] for x in j["results"]) == [0, 1, 2]
    sc = [x["relevance_score"] for x in j["results"]]
    assert sc == sorted(sc, reverse=True) and j["usage"]["total_tokens"] > 0


def test_one_call_layers_are_chosen_by_rows_and_width():
    """A one-call layer reads its weights once per 64 rows: wide encoders leave it at fewer rows (measured: small_rows)."""
    rows = BM.small_rows
    assert rows(384, 1536) == rows(768, 3072) == BM.ENC_SMALL_ROWS
    assert 192 <= rows(1024, 4096) < 320 and rows(1024, 4096) < rows(1024, 2816) < 384
    assert 64 <= rows(1280, 5120) < 192 and 64 <= rows(1536, 6144) < 128 and 48 <= rows(2048, 8192) < 96
    assert rows(3072, 12288) == rows(4096, 16384) == 0


def test_narrow_layers_stay_in_one_call():
    """Layers of few weights leave the 16-column products later than others, at most where any does; wide ones where they leave them for the library."""
    assert BM.few_rows(64, 256) == BM.few_rows(128, 512) == BM.few_rows(256, 1024) == BM.ENC_SMALL_ROWS and 128 <= BM.few_rows(512, 2048) < 192
    assert 128 <= BM.few_rows(384, 1536) < 256 and BM.few_rows(768, 3072) == BM.few_rows(1024, 4096) == BM.ENC_FEW_ROWS and BM.few_rows(2048, 8192) == BM.small_rows(2048, 8192) < 64
    assert BM.few_rows(4096, 16384) == 0


@pytest.mark.gpu
def test_bert_gpu_matches_fp32():
    """GPU path (hipBLASLt GEMMs + attention_dense.hip + norm.hip LayerNorm) vs the fp32 encoder."""
    cfg = BM.BertConfig(vocab=400, hidden=256, n_layers=2, n_heads=4, ffn=1024, max_pos=128, name="t")
    get = BM.synthetic_bert(cfg, 5)
    g = BM.BertModel.load(cfg, get, "cuda:0")
    seqs = [[2] + list(range(10, 10 + n)) + [3] for n in (70, 5, 33)]
    hid, _ = g.encode(seqs)
    for b, s in enumerate(seqs):
        ref = _reference_encode(cfg, get, s)
        err = (hid[b, :len(s)].cpu() - ref).abs().max().item()
        assert err < 5e-2, err
    e = g.embed(seqs).cpu()
    c = BM.BertModel.load(cfg, get, "cpu").embed(seqs)
    assert (e - c).abs().max() < 1e-2


@pytest.mark.gpu
@pytest.mark.parametrize("hidden,heads,ffn,pooling", [(256, 4, 1024, "mean"), (128, 1, 160, "last"), (1056, 11, 96, "mean"),
                                                      (768, 12, 3072, "cls")])
def test_packed_rows_match_fp32(hidden, heads, ffn, pooling, monkeypatch):
    """Packed texts (encoder.hip) at the edges of its 16-row tiles, one-call and library GEMMs, against the fp32 encoder: hidden
    rows within the bound of 16-bit activations (a LayerNorm output of up to ~5 is rounded to 2^-11 of itself some 8 times a
    layer, 3e-3 each), pooled unit vectors ten times closer. Head dims it does not take (1056 / 11 = 96) run padded."""
    cfg = BM.BertConfig(vocab=400, hidden=hidden, n_layers=2, n_heads=heads, ffn=ffn, max_pos=256, pooling=pooling, name="t")
    get = BM.synthetic_bert(cfg, 5)
    g, c = BM.BertModel.load(cfg, get, "cuda:0"), BM.BertModel.load(cfg, get, "cpu")
    assert (g._packed_weights([[1]]) is None) == (hidden == 1056)
    gen = torch.Generator().manual_seed(1)
    for lens in ([1], [16], [17], [1, 63, 64, 65, 3], [200, 2, 31]):
        ids = [torch.randint(0, 400, (n,), generator=gen).tolist() for n in lens]
        want, _ = c.encode(ids)
        for rows in (0, 4096):  # library GEMMs, the one-call layers
            monkeypatch.setattr(BM, "ENC_SMALL_ROWS", rows)
            hid, n = g.encode(ids)
            assert n.tolist() == lens and hid.shape == want.shape and hid.dtype == torch.float32
            for b, k in enumerate(lens):
                assert (hid[b, :k].cpu() - want[b, :k]).abs().max() < 5e-2
            assert (g.embed(ids).cpu() - c.embed(ids)).abs().max() < 5e-3
            assert (g.embed(ids, normalize=False).cpu() - c.embed(ids, normalize=False)).abs().max() < 5e-2
    if hidden != 1056:
        with pytest.raises(IndexError):
            g.embed([[400]])
        with pytest.raises(IndexError):
            g.embed([[1] * 257])
    assert g.embed([[5, 6], []]).shape == (2, hidden)
    # weights that are not where the kernels can read them: padded
    w = g.w["blk.0.ffn_up.bias"]
    g.w["blk.0.ffn_up.bias"] = torch.cat([w[:1], w])[1:]
    assert g._packed_weights([[1]]) is None and (g.embed([[5, 6]]).cpu() - c.embed([[5, 6]])).abs().max() < 5e-3


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("H", [8, 256, 504, 512, 520, 1024, 1032, 1536, 1544, 2048, 2056, 3072, 3080, 4096])
def test_row_kernels_at_the_edges_of_their_widths(H, dtype):
    """Sum of embeddings and x = LN(a + x), rows that fill a lane's chunks, leave lanes without one and start the next chunk, against
    float64: the output is rounded to 16 bits (half a unit, relative 2^-11 / 2^-8), sums of 4096 fp32 numbers of order 1 are within
    1e-5 of their length. Rows behind the last are left alone."""
    from localai_tfp_amd import _native as N
    g = torch.Generator().manual_seed(H)
    gain, off = torch.randn(H, generator=g), torch.randn(H, generator=g)
    tok, pos, typ = (torch.randn(n, H, generator=g) for n in (50, 20, 2))
    unit = 2 ** -11 if dtype == torch.float16 else 2 ** -8
    N.ensure_act(dtype)
    for rows in (1, 6):
        ids = torch.stack([torch.randint(0, n, (rows,), generator=g) for n in (50, 20, 2)])
        a, x = torch.randn(rows, H, generator=g).to(dtype), torch.randn(rows, H, generator=g).to(dtype)
        for b, t in ((off, typ), (None, None)):
            e = tok[ids[0]].double() + pos[ids[1]].double() + (t[ids[2]].double() if t is not None else 0)
            d = [v.cuda() if v is not None else None for v in (tok, pos, t, gain, b)]
            i32, y, z = ids.int().cuda(), torch.full((rows + 1, H), 7.0, dtype=dtype, device="cuda"), torch.full((rows + 1, H), 7.0, dtype=dtype, device="cuda")
            N.kcall("mxk_enc_embed", i32.data_ptr(), rows, *(N.ptr(v) for v in d), H, 1e-6, y.data_ptr(), N.stream_ptr())
            z[:rows] = x.cuda()
            ad = a.cuda()
            N.kcall("mxk_enc_add_ln", ad.data_ptr(), z.data_ptr(), rows, d[3].data_ptr(), N.ptr(d[4]), H, 1e-6, N.stream_ptr())
            for got, v in ((y, e), (z, a.double() + x.double())):
                want = (v - v.mean(1, keepdim=True)) * torch.rsqrt(v.var(1, unbiased=False, keepdim=True) + 1e-6) * gain.double()
                want = want + (b.double() if b is not None else 0)
                assert ((got[:rows].cpu().double() - want).abs() <= unit * want.abs() + 1e-4).all() and (got[rows:] == 7.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("hidden", [1536, 2560])
def test_wide_one_call_layers(hidden, monkeypatch):
    """Rows of three and of five chunks a lane through the one-call layers (sums of one and of four parts of K): bounds as above."""
    cfg = BM.BertConfig(vocab=400, hidden=hidden, n_layers=1, n_heads=hidden // 64, ffn=2048, max_pos=64, name="t")
    get = BM.synthetic_bert(cfg, 5)
    g, c = BM.BertModel.load(cfg, get, "cuda:0"), BM.BertModel.load(cfg, get, "cpu")
    monkeypatch.setattr(BM, "small_rows", lambda H, F: 4096)
    ids = [list(range(10, 10 + n)) for n in (17, 3)]
    hid, n = g.encode(ids)
    want, _ = c.encode(ids)
    for i, k in enumerate(n.tolist()):
        assert (hid[i, :k].cpu() - want[i, :k]).abs().max() < 5e-2


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hidden,heads,ffn", [(64, 1, 96), (512, 8, 2048), (576, 9, 2080), (1024, 16, 2048), (1024, 8, 160), (1088, 17, 96)])
def test_few_rows_with_norms_and_attention_inside_the_products(hidden, heads, ffn, dtype, monkeypatch):
    """Norms inside the products up to 16 rows, attention of one text up to 64: at the edges of the 16-row tiles and of the widths a lane
    holds in one chunk or two, products in one part and in four, heads of 64 and of 128; 1088 columns beside them. The bound of test_packed_rows_match_fp32 (bf16:
    eight times, its rounding)."""
    cfg = BM.BertConfig(vocab=400, hidden=hidden, n_layers=3, n_heads=heads, ffn=ffn, max_pos=64, name="t")
    get = BM.synthetic_bert(cfg, 5)
    monkeypatch.setattr(BM, "ACT_DTYPE", dtype)
    g, c = BM.BertModel.load(cfg, get, "cuda:0"), BM.BertModel.load(cfg, get, "cpu")
    used = []
    real = BM.N.kcall
    monkeypatch.setattr(BM.N, "kcall", lambda name, *a: (used.append(name), real(name, *a))[1])
    for lens in ([1], [0], [8], [9], [16], [17], [32], [33], [48], [49], [64], [3, 0, 12], [9, 8], [1] * 16):
        ids = [list(range(10, 10 + n)) for n in lens]
        got, want = g.embed(ids).cpu(), c.embed(ids)
        assert "mxk_enc_layers" in used and (got - want).abs().max() < (5e-3 if dtype == torch.float16 else 4e-2), lens


@pytest.mark.gpu
@pytest.mark.parametrize("hidden,heads,ffn", [(512, 8, 2048), (576, 9, 2080), (1024, 16, 2048), (1024, 8, 160)])
def test_norms_of_several_texts(hidden, heads, ffn):
    """Norms inside the products of several texts: up to 16 rows of 512 columns, up to 8 beyond; apart from there on. The bound of
    test_packed_rows_match_fp32."""
    cfg = BM.BertConfig(vocab=400, hidden=hidden, n_layers=3, n_heads=heads, ffn=ffn, max_pos=64, name="t")
    get = BM.synthetic_bert(cfg, 5)
    g, c = BM.BertModel.load(cfg, get, "cuda:0"), BM.BertModel.load(cfg, get, "cpu")
    for lens in ([1, 1], [3, 5], [0, 7], [4, 5], [7, 1, 8], [9, 8]):
        ids = [list(range(10, 10 + n)) for n in lens]
        assert (g.embed(ids).cpu() - c.embed(ids)).abs().max() < 5e-3, lens


@pytest.mark.gpu
@pytest.mark.parametrize("pooling", ["mean", "cls", "last"])
def test_empty_texts_match_the_padded_batch(pooling):
    """An empty text has a row too: nothing for the mean, its first row, or the batch's last position."""
    cfg = BM.BertConfig(vocab=400, hidden=128, n_layers=2, n_heads=2, ffn=256, max_pos=64, pooling=pooling, name="t")
    get = BM.synthetic_bert(cfg, 5)
    g, c = BM.BertModel.load(cfg, get, "cuda:0"), BM.BertModel.load(cfg, get, "cpu")
    ids = [[5, 6, 7, 8, 9], [], [11, 12], []]
    assert g._packed_weights(ids) is not None
    assert (g.embed(ids).cpu() - c.embed(ids)).abs().max() < 5e-3  # (the bound of test_packed_rows_match_fp32)


def test_encoder_plans_are_within_what_the_kernels_take():
    from localai_tfp_amd.ops import dense as D
    tiles = {16 * a + b for a, b in D._D16_ENC_COST[0]}
    for rows in (1, 65, 449, 1000, 6428, 100000):
        for H, F in ((64, 64), (128, 512), (768, 3072), (1024, 2816), (4096, 16384)):
            q, o, po, u, d, pd = D.encoder_plan(rows, H, F)
            assert {q, o, u, d} <= tiles and po in (1, 2, 3, 4, 8) and pd in (1, 2, 3, 4, 8) and po <= H // 64 and pd <= F // 64
            assert max(po, pd) == 1 or rows * H * max(po, pd) <= 1 << 25


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [136, 120, 104, 88, 134, 102, 132, 84, 68, 40, 36])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_tiled_layers_match_fp32(tile, dtype, monkeypatch):
    """Every tile in every product of a layer, undivided and in each number of parts, one row, part-empty tiles and some of each: the bound
    of test_packed_rows_match_fp32 (bf16: eight times, its rounding)."""
    cfg = BM.BertConfig(vocab=400, hidden=192, n_layers=2, n_heads=3, ffn=576, max_pos=300, name="t")
    get = BM.synthetic_bert(cfg, 5)
    monkeypatch.setattr(BM, "ACT_DTYPE", dtype)
    g, c = BM.BertModel.load(cfg, get, "cuda:0"), BM.BertModel.load(cfg, get, "cpu")
    monkeypatch.setattr(BM, "ENC_FEW_ROWS", 0)
    used = []
    real = BM.N.kcall
    monkeypatch.setattr(BM.N, "kcall", lambda name, *a: (used.append(name), real(name, *a))[1])
    for lens, po, pd in (([1], 1, 1), ([33, 200, 24], 3, 8), ([258, 3], 2, 4), ([63], 1, 3)):
        monkeypatch.setattr(BM, "encoder_plan", lambda R, H, F: (tile, tile, po, tile, tile, pd))
        ids = [list(range(10, 10 + n)) for n in lens]
        got, want = g.embed(ids).cpu(), c.embed(ids)
        assert "mxk_enc_layers_tiled" in used and (got - want).abs().max() < (5e-3 if dtype == torch.float16 else 4e-2), (lens, po, pd)


def test_attention_blocks_cover_each_row_once():
    for rows in ([1], [64, 65, 63, 1], [5, 300, 300, 128, 129], [1] * 70):
        for q in (64, 128):
            b = BM.attn_blocks(np.array(rows), q)
            assert sorted(map(tuple, b.tolist())) == sorted((i, f) for i, n in enumerate(rows) for f in range(0, n, q))
            assert (np.diff(np.array(rows)[b[:, 0]]) <= 0).all() and b.dtype == np.int32
    assert BM.attn_blocks(np.full(65535, 1), 64).shape == (65535, 2) and BM.attn_blocks(np.array([64] * 65535 + [1]), 64) is None


@pytest.mark.gpu
@pytest.mark.parametrize("heads", [2, 4])
def test_texts_of_blocks_edges_in_any_order(heads, monkeypatch):
    """Heads of 128 and 64: texts of no token, of one, around whole blocks of 64 and 128 rows; the bound of test_packed_rows_match_fp32. Calls follow
    each other without a wait between them: an image may not be written over while it is copied."""
    cfg = BM.BertConfig(vocab=400, hidden=256, n_layers=2, n_heads=heads, ffn=512, max_pos=300, name="t")
    get = BM.synthetic_bert(cfg, 5)
    g, c = BM.BertModel.load(cfg, get, "cuda:0"), BM.BertModel.load(cfg, get, "cpu")
    monkeypatch.setattr(BM, "ENC_FEW_ROWS", 0)
    batches = [[1, 63, 64, 65, 128, 129, 257], [129, 0, 2], [64, 64], [300, 1, 127], [65]]
    ids = [[[(7 * i + j) % 390 + 5 for j in range(n)] for i, n in enumerate(lens)] for lens in batches]
    got = [g.embed(x) for x in ids * 3]
    for e, x in zip(got, ids * 3):
        want = c.embed(x)
        assert (e.cpu() - want)[[i for i, t in enumerate(x) if t]].abs().max() < 5e-3


@pytest.mark.gpu
@pytest.mark.parametrize("hidden,rows", [(64, 65), (128, 300), (384, 448), (512, 200), (640, 300), (768, 400), (832, 350)])
def test_sums_stay_in_fp32_until_the_norm(hidden, rows, monkeypatch):
    """Biases of 1000, which the norms take away again: an f16 there has steps of 0.5, fp32 of 6e-5, beside rows of order 1. Up to small_rows
    the bound of test_wide_one_call_layers holds all the same; the smallest widths have undivided products throughout."""
    monkeypatch.setattr(BM, "ENC_FEW_ROWS", 0)
    cfg = BM.BertConfig(vocab=400, hidden=hidden, n_layers=2, n_heads=hidden // 64, ffn=4 * hidden, max_pos=300, name="t")
    src = BM.synthetic_bert(cfg, 5)

    def get(name):
        t = src(name)
        return t + 1000 if t is not None and name in [f"blk.{i}.{b}.bias" for i in (0, 1) for b in ("attn_output", "ffn_down")] else t
    g, c = BM.BertModel.load(cfg, get, "cuda:0"), BM.BertModel.load(cfg, get, "cpu")
    assert rows <= BM.small_rows(hidden, 4 * hidden) and float(c.w["blk.0.ffn_down.bias"].float().mean()) > 900
    ids = [list(range(10, 10 + n)) for n in (rows // 2, rows - rows // 2)]
    hid, n = g.encode(ids)
    want, _ = c.encode(ids)
    for i, k in enumerate(n.tolist()):
        assert (hid[i, :k].cpu() - want[i, :k]).abs().max() < 5e-2


@pytest.mark.gpu
@pytest.mark.parametrize("small", [448, 0])
def test_parts_that_do_not_fit_are_done_without(small, monkeypatch):
    """No room for a product's parts (refused here from the host): undivided products, in one fp32 part up to small_rows, else with
    16-bit sums. The bound of test_packed_rows_match_fp32."""
    cfg = BM.BertConfig(vocab=400, hidden=192, n_layers=2, n_heads=3, ffn=576, max_pos=300, name="t")
    get = BM.synthetic_bert(cfg, 5)
    g, c = BM.BertModel.load(cfg, get, "cuda:0"), BM.BertModel.load(cfg, get, "cpu")
    monkeypatch.setattr(BM, "small_rows", lambda H, F: small)
    monkeypatch.setattr(BM, "ENC_FEW_ROWS", 0)
    monkeypatch.setattr(BM, "encoder_plan", lambda R, H, F: (36, 68, 3, 36, 40, 8))
    ids = [list(range(10, 10 + n)) for n in (200, 57)]
    want, refused, real = c.embed(ids), [], torch.empty

    def empty(*a, **k):
        if k.get("dtype") == torch.float32 and len(a) == 3 and a[0] > 1:
            refused.append(a)
            raise torch.cuda.OutOfMemoryError("no room")
        return real(*a, **k)
    monkeypatch.setattr(torch, "empty", empty)
    got = g.embed(ids)
    monkeypatch.setattr(torch, "empty", real)
    assert refused == [(8, 257, 192)] and (got.cpu() - want).abs().max() < 5e-3


@pytest.mark.gpu
def test_gelu_rounds_like_64_bits():
    """Every finite f16: within a unit of the last place, and the nearest f16 for all but one in a thousand (fp32 arithmetic near the
    middle of two). Infinities and NaN as 0.5 x (1 + erf(x / sqrt 2)) has them."""
    from localai_tfp_amd import _native as N
    N.ensure_act(torch.float16)
    x = torch.arange(1 << 16, dtype=torch.int32).to(torch.int16).view(torch.float16)
    y = x.cuda()
    N.kcall("mxk_enc_gelu", y.data_ptr(), y.numel(), N.stream_ptr())
    y, d = y.cpu(), x.double()
    want = 0.5 * d * torch.special.erfc(-d * 2 ** -0.5)
    ok = torch.isfinite(x)
    near = want.to(torch.float16)
    # (neighbours in order: sign and magnitude bits as one whole number)
    step = (y.view(torch.int16).int() & 0x7FFF) - (near.view(torch.int16).int() & 0x7FFF)
    assert (step[ok].abs() <= 1).all() and (step[ok] != 0).float().mean() < 1e-3
    assert (y[ok & (want.abs() > 1e-7)].sign() == near[ok & (want.abs() > 1e-7)].sign()).all()
    inf = float("inf")
    assert y[x == inf].item() == inf and torch.isnan(y[x == -inf]).all() and torch.isnan(y[torch.isnan(x)]).all()
