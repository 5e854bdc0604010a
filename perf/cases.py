"""What this framework is timed on: the forward passes behind its text endpoints, at the sizes they are served with.

A pass is one step of a serving loop, called the way the engine and the workers call it:

* ``llama``  one `LlamaModel.forward` over a paged cache: `dec` decode rows whose contexts spread from `ctx_lo` to
  `ctx_hi` tokens, and `pf` prompt chunks of `pf_lo` .. `pf_hi` tokens behind `pre_lo` .. `pre_hi` cached ones. Layers of
  Llama-3-8B ("8b") or Llama-3.2-1B ("1b") size in Q4_K_M, four of them, under a 32000-word head.
* ``hybrid`` the same for the hybrid decoder (`VugotarModel`): layers of its 7B configuration, one of attention beside
  a gated delta rule and one state-space layer, bf16.
* ``embed``  `BertModel.embed` of the embeddings endpoint, BERT-base sized, a batch of texts of `lo` .. `hi` tokens.

Steps of up to 1024 tokens replay a captured graph like the engine's, larger ones run eagerly; the GEMM plans are tuned
when the model is loaded, as the engine does. Weights are a checkpoint: one per model, whatever the seed. Tokens, cache
contents, page tables and recurrent states come from the seed.
"""
import dataclasses
import math

import torch

from localai_tfp_amd.engine.engine import kv_format_id, kv_torch_dtype
from localai_tfp_amd.engine.kv_cache import KVCache
from localai_tfp_amd.models import bert as B
from localai_tfp_amd.models import config as C
from localai_tfp_amd.models import vugotar as V
from localai_tfp_amd.models.llama import ForwardBatch, LlamaModel, Workspace
from localai_tfp_amd.models.synthetic import synthetic_source
from localai_tfp_amd.ops.autotune import tune_gemms
from localai_tfp_amd.ops.core import prefill_tiles

DEV = "cuda"
F64 = torch.float64
BS = 16  # tokens of a cache page
GRAPH_TOKENS = 1024  # steps up to this size are captured
LLAMA = {"8b": C.LLAMA3_8B, "1b": C.LLAMA32_1B}
LAYERS, VOCAB = 4, 32000
HYBRID = dict(V.SYNTHETIC["vugotar-7b"], pattern=("parallel", "mamba2"))


# ------------------------------------------------------------------------------------------------ the cases
def _llama(name, model="8b", kv="bf16", dec=0, ctx=(1, 1), pf=0, rows=(1, 1), pre=(0, 0)):
    return {"name": name, "kind": "llama", "model": model, "kv": kv, "dec": dec, "ctx_lo": ctx[0], "ctx_hi": ctx[1], "pf": pf,
            "pf_lo": rows[0], "pf_hi": rows[1], "pre_lo": pre[0], "pre_hi": pre[1]}


def _hybrid(name, dec=0, ctx=(1, 1), pf=0, rows=(1, 1)):
    return {"name": name, "kind": "hybrid", "dec": dec, "ctx_lo": ctx[0], "ctx_hi": ctx[1], "pf": pf, "pf_lo": rows[0], "pf_hi": rows[1]}


def listed():
    return [
        # one user chatting: the latency of a token
        _llama("chat_1", dec=1, ctx=(711, 711)),
        # a small team on one GPU, conversations of very different length
        _llama("chat_32", dec=32, ctx=(97, 4003)),
        # the saturated server: the serving benchmark's decode batch
        _llama("chat_128", dec=128, ctx=(65, 1021)),
        # long documents in an 8-bit block cache (cache_type_k / v: q8_0)
        _llama("chat_9_long_q8", kv="q8_0", dec=9, ctx=(3001, 24001)),
        # continuous batching: a full decode batch with a prompt chunk, the engine's default step budget
        _llama("mixed_127_289", dec=127, ctx=(65, 1021), pf=1, rows=(289, 289)),
        # time to first token of a chat turn
        _llama("prompt_333", pf=1, rows=(333, 333)),
        # one default-sized chunk of a long prompt, most of it cached, in an fp8 cache
        _llama("chunk_416_fp8", kv="fp8", pf=1, rows=(416, 416), pre=(12000, 12000)),
        # a document of 8191 tokens in one step (batch: 8192)
        _llama("prompt_8191", pf=1, rows=(8191, 8191)),
        # the hybrid decoder: three prompts of one step, and a decode batch
        _hybrid("hybrid_prompts", pf=3, rows=(301, 1111)),
        _hybrid("hybrid_chat_33", dec=33, ctx=(101, 4001)),
        # embeddings: one search query, and a batch of passages
        {"name": "embed_query", "kind": "embed", "texts": 1, "lo": 19, "hi": 19},
        {"name": "embed_48", "kind": "embed", "texts": 48, "lo": 23, "hi": 401},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "mixed", "hybrid", "hybrid", "embed"])
    model = rng.choice(["8b", "8b", "1b"])
    kv = rng.choice(["bf16", "bf16", "fp8"])  # (q8_0 in decode steps alone: a prompt's own codes sit on rounding edges)
    if kind == "decode":
        kv = rng.choice([kv, kv, kv, "q8_0"])
        n = _log(rng, 1, 192)
        hi = _log(rng, 64, min(24000, 300000 // n))
        c = _llama("", model, kv, dec=n, ctx=(max(2, int(hi * rng.uniform(0.03, 1))), hi))
    elif kind == "prompt":
        n = rng.choice([1, 1, 2, 3])
        hi = _log(rng, 17, 6000 // n)
        pre = _log(rng, 16, 12000) if hi <= 1024 and rng.random() < 0.4 else 0
        c = _llama("", model, kv, pf=n, rows=(max(2, int(hi * rng.uniform(0.3, 1))), hi), pre=(pre // 2, pre))
    elif kind == "mixed":
        n = _log(rng, 4, 160)
        hi = _log(rng, 64, 2000)
        r = _log(rng, 16, 512)
        c = _llama("", model, kv, dec=n, ctx=(max(2, int(hi * rng.uniform(0.05, 1))), hi), pf=1, rows=(r, r), pre=(0, 0))
    elif kind == "hybrid" and rng.random() < 0.5:
        n = _log(rng, 1, 64)
        hi = _log(rng, 64, 8000)
        c = _hybrid("", dec=n, ctx=(max(2, int(hi * rng.uniform(0.03, 1))), hi))
    elif kind == "hybrid":
        n = rng.choice([1, 2, 3, 4])
        hi = _log(rng, 18, 3000 // n)
        c = _hybrid("", pf=n, rows=(max(2, int(hi * rng.uniform(0.3, 1))), hi))
    else:
        n = _log(rng, 1, 96)
        hi = _log(rng, 8, min(512, 24000 // n))
        c = {"kind": "embed", "texts": n, "lo": max(3, int(hi * rng.uniform(0.05, 1))), "hi": hi}
    c.pop("name", None)
    return c


def _spread(n, lo, hi):
    """n lengths from lo to hi, evenly spaced over their logarithm."""
    return [int(round(lo * (hi / lo) ** (i / max(1, n - 1)))) if lo > 0 else int(hi * i / max(1, n - 1)) for i in range(n)] if n > 1 else [hi] * n


def _lens(case):
    """(contexts of the decode rows with their new token, rows of the chunks, cached tokens before each chunk)."""
    return (_spread(case["dec"], case["ctx_lo"], case["ctx_hi"]), _spread(case["pf"], case["pf_lo"], case["pf_hi"]),
            _spread(case["pf"], case.get("pre_lo", 0), case.get("pre_hi", 0)))


# ------------------------------------------------------------------------------------------------ the checkpoints
_LOADED = {}


def _llama_cfg(model):
    return dataclasses.replace(LLAMA[model], n_layers=LAYERS, vocab=VOCAB, ctx_train=32768)


def _hybrid_tensors(cfg):
    """name -> bf16 tensor, random in the scales of `VugotarModel`'s synthetic checkpoints, made on the GPU."""
    shapes, made = V.tensor_shapes(cfg), {}

    def get(name):
        if name not in made:
            s, leaf = shapes[name], name.rsplit(".", 1)[-1]
            g = torch.Generator(device=DEV).manual_seed(17 + sorted(shapes).index(name))
            a = torch.randn(s, generator=g, device=DEV)
            if leaf == "norm1" or name == "final.norm":
                a = 0.1 * a
            elif leaf == "norm":
                a = 1 + 0.1 * a
            elif leaf == "A_log":
                a = torch.log(0.5 + 2 * torch.rand(s, generator=g, device=DEV))
            elif leaf == "dt_bias":
                a = a - 1
            elif leaf == "D":
                a = 1 + 0.2 * a
            elif leaf == "conv" or (leaf == "b" and len(s) == 1):
                a = 0.5 * a
            else:
                a = a * s[-1] ** -0.5
            made[name] = a.to(torch.bfloat16)
        return made[name]
    return get


def _loaded(kind, model=""):
    """The loaded model and what names its weights: a serving process loads a checkpoint once."""
    key = (kind, model)
    if key not in _LOADED:
        if kind == "llama":
            cfg = _llama_cfg(model)
            src = synthetic_source(cfg, "Q4_K_M", seed=5)
            m = LlamaModel.load(cfg, src, DEV)
            tune_gemms(m.gemm_specs())
        elif kind == "hybrid":
            cfg = V.make_config(name="hybrid", **HYBRID)
            src = _hybrid_tensors(cfg)
            m = V.VugotarModel.load(cfg, src, DEV)
        else:
            src = B.synthetic_bert(B.BERT_BASE, seed=5)
            m = B.BertModel.load(B.BERT_BASE, src, DEV)
        _LOADED[key] = (m, src)
    return _LOADED[key]


# ------------------------------------------------------------------------------------------------ a step's inputs
def _i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


def _batch(case, seed, rows_per_tile, max_len):
    """ForwardBatch of the case with pages handed out in a random order, and the number of pages."""
    ctx, rows, pre = _lens(case)
    total = [*ctx, *(r + p for r, p in zip(rows, pre))]
    n_pages = sum(-(-t // BS) for t in total) + 1
    g = torch.Generator().manual_seed(seed)
    order = (torch.randperm(n_pages - 1, generator=g) + 1).tolist()
    tables, at = [], 0
    for t in total:
        n = -(-t // BS)
        tables.append(order[at:at + n])
        at += n
    tokens = torch.randint(0, VOCAB, (case["dec"] + sum(rows),), generator=g, dtype=torch.int32)
    pos, slots, last = [], [], []
    for c, t in zip(ctx, tables):
        pos.append(c - 1)
        slots.append(t[(c - 1) // BS] * BS + (c - 1) % BS)
        last.append(len(pos) - 1)
    for r, p, t in zip(rows, pre, tables[len(ctx):]):
        pos += range(p, p + r)
        slots += [t[x // BS] * BS + x % BS for x in range(p, p + r)]
        last.append(len(pos) - 1)
    width = -(-max_len // BS)
    padded = [t + [0] * (width - len(t)) for t in tables]
    fb = ForwardBatch(tokens.to(DEV), _i32(pos), _i32(slots), _i32(last), n_decode=len(ctx))
    if ctx:
        fb.dec_block_tables, fb.dec_seq_lens = _i32(padded[:len(ctx)]), _i32(ctx)
        # the engine's graph buckets: short contexts of a few rows and full batches run one attention partition
        hi = max(ctx)
        fb.dec_max_len = 512 if len(ctx) < 8 and hi <= 512 and not rows else 1024 if len(ctx) >= 64 and hi <= 1024 else max_len
    if rows:
        fb.pf_block_tables, fb.pf_ctx_lens = _i32(padded[len(ctx):]), _i32([r + p for r, p in zip(rows, pre)])
        fb.pf_cu_q = _i32([sum(rows[:i]) for i in range(len(rows) + 1)])
        fb.pf_q_lens_host, fb.pf_ctx_lens_host = list(rows), [r + p for r, p in zip(rows, pre)]
        if rows_per_tile:
            a, b = prefill_tiles(rows, rows_per_tile)
            fb.pf_tiles = (_i32(a), _i32(b))
    return fb, n_pages


def _fill(t, g, fmt, D):
    """A cache pool as a conversation leaves it: unit-sized keys and values in the pool's format."""
    for i in range(t.shape[0]):
        if fmt == "q8_0":
            n = t[i].numel() // t.shape[-1]
            x = torch.randint(-127, 128, (n, D), generator=g, device=DEV, dtype=torch.int8)
            d = (torch.rand((n, D // 32), generator=g, device=DEV) * 0.01 + 0.015).to(torch.float16)
            t[i].copy_(torch.cat([x.view(torch.uint8), d.view(torch.uint8)], 1).view(t[i].shape))
        else:
            t[i].copy_(torch.randn(t[i].shape, generator=g, device=DEV).to(t.dtype))


def _max_len(case):
    ctx, rows, pre = _lens(case)
    need = max([*ctx, *(r + p for r, p in zip(rows, pre))]) + 1
    return next(n for n in (8192, 16384, 32768) if n >= need)


def prepare(case, seed):
    if case["kind"] == "embed":
        m, _ = _loaded("embed")
        g = torch.Generator().manual_seed(seed)
        ids = [[101, *torch.randint(1000, B.BERT_BASE.vocab, (max(1, n - 2),), generator=g).tolist(), 102] for n in _spread(case["texts"], case["lo"], case["hi"])]
        return {"call": lambda: m.embed(ids), "ids": ids}
    g = torch.Generator(device=DEV).manual_seed(seed)
    n_dec, n_seqs, max_len = case["dec"], case["dec"] + case["pf"], _max_len(case)
    T = n_dec + sum(_lens(case)[1])
    if case["kind"] == "llama":
        m, _ = _loaded("llama", case["model"])
        cfg = m.cfg
        fb, pages = _batch(case, seed, m.prefill_rows(), max_len)
        cache = KVCache(cfg.n_layers, pages, m.n_kv, BS, cfg.head_dim, DEV, kv_torch_dtype(case["kv"]), kvf=kv_format_id(case["kv"]))
        for t in (cache.k, cache.v):
            _fill(t, g, case["kv"], cfg.head_dim)
        ws = Workspace(cfg, T, n_seqs, DEV, 1, -(-max_len // 256))
        kept = {"k": cache.k, "v": cache.v}
    else:
        m, _ = _loaded("hybrid")
        fb, pages = _batch(case, seed, 0, max_len)
        fb.seq_state = _i32(list(range(n_seqs))[::-1])
        cache = m.make_cache(pages, BS, n_seqs)
        for kv, state, tails in zip(cache.kv, cache.state, cache.tails):
            for t in kv or ():
                t.copy_(torch.randn(t.shape, generator=g, device=DEV).to(t.dtype))  # (keys of unit root mean square)
            state.copy_(0.3 * torch.randn(state.shape, generator=g, device=DEV))
            tails.copy_(0.5 * torch.randn(tails.shape, generator=g, device=DEV))
        ws = m.make_workspace(T, n_seqs, 0, -(-max_len // 256))
        kept = {"state": cache.state, "tails": cache.tails, "kv": [t for kv in cache.kv for t in kv or ()]}
    state = {"fb": fb, "cache": cache, "ws": ws, "kept": kept, "model": m, "graph": None}
    if T <= GRAPH_TOKENS:
        # warm up and capture as the engine does; what the steps wrote is put back
        saved = [t.clone() for t in (*cache.state, *cache.tails)] if case["kind"] == "hybrid" else []
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            m.forward(fb, cache, ws)
        torch.cuda.current_stream().wait_stream(s)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            state["logits"] = m.forward(fb, cache, ws)
        for t, x in zip((*cache.state, *cache.tails) if saved else (), saved):
            t.copy_(x)
        state["graph"] = graph
    return state


def run(state):
    if "call" in state:
        return state["call"]()
    if state["graph"] is not None:
        state["graph"].replay()
        logits = state["logits"]
    else:
        logits = state["model"].forward(state["fb"], state["cache"], state["ws"])
    return {"logits": logits, **state["kept"]}


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _visible(lo, n, chunk=0):
    """Sum over positions lo .. lo + n - 1 of the keys each sees."""
    return sum((p % chunk if chunk else p) + 1 for p in range(lo, lo + n))


def work(case):
    if case["kind"] == "embed":
        c, lens = B.BERT_BASE, _spread(case["texts"], case["lo"], case["hi"])
        T, per = sum(lens), 4 * c.hidden * c.hidden + 2 * c.hidden * c.ffn
        return {"bytes": 2 * per * c.n_layers + 8 * T + 4 * c.hidden * (T + len(lens)), "flops": c.n_layers * (2 * per * T + sum(4 * c.hidden * n * n for n in lens))}
    ctx, rows, pre = _lens(case)
    T, S = len(ctx) + sum(rows), len(ctx) + len(rows)
    if case["kind"] == "llama":
        cfg = _llama_cfg(case["model"])
        q4, q6 = 144 / 256, 210 / 256
        H, F, qd, kvd = cfg.hidden, cfg.ffn, cfg.q_dim, cfg.kv_dim
        per = H * (qd + 2 * kvd) + qd * H + 3 * H * F
        more = [i for i in range(LAYERS) if i < LAYERS // 8 or i >= 7 * LAYERS // 8 or (i - LAYERS // 8) % 3 == 2]
        head = H * cfg.vocab
        weights = LAYERS * per * q4 + len(more) * (H * kvd + H * F) * (q6 - q4) + head * (q4 if cfg.tie_embeddings else q6)
        row = {"bf16": 4.0, "fp8": 2.0, "q8_0": 2 * 34 / 32}[case["kv"]] * kvd  # one token's keys and values in a layer
        kv = LAYERS * row * (sum(ctx) + sum(rows) + sum(pre) + T)
        seen = sum(ctx) + sum(_visible(p, r) for p, r in zip(pre, rows))
        return {"bytes": weights + kv + T * H * q4 + 4 * S * cfg.vocab, "flops": 2 * (LAYERS * per * T + head * S) + LAYERS * 4 * qd * seen}
    cfg = V.make_config(**HYBRID)
    shapes = V.tensor_shapes(cfg)
    w = sum(math.prod(s) for n, s in shapes.items() if n != "embed" and len(s) == 2)
    a, r, m2 = cfg.layers[0].mixer.left, cfg.layers[0].mixer.right, cfg.layers[1].mixer
    seen = sum((c - 1) % a.chunk + 1 for c in ctx) + sum(_visible(0, n, a.chunk) for n in rows)
    cells = r.heads * r.vdim * r.dim + m2.heads * m2.vdim * m2.state  # recurrent state numbers
    tails = sum(e["tails"][0] * e["tails"][1] for e in V.VugotarModel(cfg, "cpu").cache_spec())
    kv = 2 * a.kv_heads * (a.dim + a.vdim)
    reads = sum((c - 1) % a.chunk + 1 for c in ctx) + sum(rows)
    head = cfg.vocab * cfg.hidden
    return {"bytes": 2 * w + S * (cells + tails) * (8 if ctx else 4) + kv * (reads + T) + 2 * T * cfg.hidden + 4 * S * cfg.vocab,
            "flops": 2 * (w - head) * T + 2 * head * S + 2 * a.heads * (a.dim + a.vdim) * seen + 6 * cells * T}


def tolerance(case):
    # 16-bit activations (fp16 beside quantised weights, bf16 in the hybrid decoder) through a few layers; steps of up to four
    # rows multiply 8-bit activations (two runs differ by 0.014: sums in another order, rounded to other codes); eight-bit
    # caches round what a step appends
    if case["kind"] == "embed":
        return {"rel": 5e-3, "max": 0.05}
    if case["kind"] == "hybrid":
        return {"rel": 0.02, "max": 0.5}
    if case["kv"] != "bf16" or case["dec"] + sum(_lens(case)[1]) <= 4:
        return {"rel": 0.03, "max": 0.9, "differ": 0.01}
    return {"rel": 0.02, "max": 0.5}


# ------------------------------------------------------------------------------------------------ the same in 64 bits
def _u8(raw, block):
    return torch.from_numpy(raw.view("uint8").reshape(-1, block).copy()).to(DEV)


def _half(b):
    return b.contiguous().view(torch.float16).to(F64)


def _dequant(src, name):
    """A checkpoint tensor of ggml's Q4_K, Q6_K or F32 type as 64-bit [rows, columns]."""
    raw, qt, shape = src(name)
    rows = math.prod(shape[1:])
    if qt == 0:
        return torch.from_numpy(raw.view("float32").copy()).to(DEV, F64).view(rows, -1)
    if qt == 12:
        b = _u8(raw, 144)
        s, q = b[:, 4:16].int(), b[:, 16:].view(-1, 4, 32).int()
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6 << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | (s[:, 4:8] >> 6 << 4)], 1)
        q = torch.stack([q & 15, q >> 4], 2).view(-1, 8, 32).to(F64)
        return (_half(b[:, :2])[:, :, None] * sc[:, :, None] * q - _half(b[:, 2:4])[:, :, None] * mn[:, :, None]).view(rows, -1)
    if qt != 14:
        raise ValueError("type %d" % qt)
    b = _u8(raw, 210)
    lo, hi = b[:, :128].view(-1, 2, 2, 32).int(), b[:, 128:192].view(-1, 2, 1, 32).int()
    q = torch.cat([(lo & 15) | ((hi >> torch.tensor([0, 2], device=DEV)[:, None]) & 3) << 4, (lo >> 4) | ((hi >> torch.tensor([4, 6], device=DEV)[:, None]) & 3) << 4], 2)
    sc = b[:, 192:208].contiguous().view(torch.int8).to(F64)
    return (_half(b[:, 208:])[:, :, None] * sc[:, :, None] * (q.view(-1, 16, 16) - 32).to(F64)).view(rows, -1)


def _pool_rows(t, fmt, D):
    """Cache rows as 64-bit numbers."""
    if fmt != "q8_0":
        return t.to(F64)
    codes, d = t[..., :D].contiguous().view(torch.int8).to(F64), _half(t[..., D:])
    return (codes.unflatten(-1, (-1, 32)) * d[..., None]).flatten(-2)


def _stored(x, fmt):
    """What a cache of the format holds of new rows."""
    if fmt == "q8_0":
        b = x.unflatten(-1, (-1, 32))
        d = b.abs().amax(-1, keepdim=True) / 127
        return (torch.round(b / d.clamp_min(1e-30)) * d.to(torch.float16).to(F64)).flatten(-2)
    return x.to(torch.float8_e4m3fn if fmt == "fp8" else torch.bfloat16).to(F64)


def _attend(q, k, v, pos, scale, chunk=0, sink=False):
    """q [n, H, d] at positions pos, k / v [m, G, d] of positions 0 .. m - 1 -> [n, H, d]; `sink` adds exp(0) to the
    denominator, `chunk` hides keys before the query's own block of so many positions."""
    n, H, G = q.shape[0], q.shape[1], k.shape[1]
    out = torch.empty(n, H, v.shape[2], dtype=F64, device=DEV)
    keys = torch.arange(k.shape[0], device=DEV)
    for r in range(0, n, 1024):
        p = pos[r:r + 1024, None]
        seen = (keys <= p) & (keys >= (p // chunk * chunk if chunk else 0))
        for g in range(G):
            hs = slice(g * (H // G), (g + 1) * (H // G))
            s = torch.einsum("nhd,md->nhm", q[r:r + 1024, hs], k[:, g]) * scale
            s = s.masked_fill(~seen[:, None], -math.inf)
            top = s.amax(-1, keepdim=True)
            e = torch.exp(s - top)
            den = e.sum(-1, keepdim=True) + (torch.exp(-top) if sink else 0)
            out[r:r + 1024, hs] = torch.einsum("nhm,md->nhd", e / den, v[:, g])
    return out


def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _turn(x, pos, base):
    """Rotary positions on neighbouring pairs; x [n, heads, d]."""
    d = x.shape[-1]
    a = pos.to(F64)[:, None] * base ** (-torch.arange(0, d, 2, dtype=F64, device=DEV) / d)
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    u, v = x[..., ::2], x[..., 1::2]
    return torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)


def _segments(case):
    """(first row, rows, first position) of each sequence of the step."""
    ctx, rows, pre = _lens(case)
    out = [(i, 1, c - 1) for i, c in enumerate(ctx)]
    at = len(ctx)
    for r, p in zip(rows, pre):
        out.append((at, r, p))
        at += r
    return out


def _tables(fb):
    return [t for t in (fb.dec_block_tables, fb.pf_block_tables) if t is not None for t in t]


def exact(case, seed):
    with torch.no_grad():
        return {"llama": _exact_llama, "hybrid": _exact_hybrid, "embed": _exact_embed}[case["kind"]](case, seed)


def _exact_llama(case, seed):
    st = prepare(case, seed)
    m, src = _loaded("llama", case["model"])
    cfg, fb, fmt = m.cfg, st["fb"], case["kv"]
    D, Hq, Hk = cfg.head_dim, cfg.n_heads, cfg.n_kv_heads
    pos, slots = fb.positions.long(), fb.slots.long()
    # the graph's warm-up wrote the new rows into the cache already: they are written again here, the others are inputs
    kept = [[_pool_rows(p[i], fmt, D).transpose(1, 2).reshape(-1, Hk, D) for p in (st["kept"]["k"], st["kept"]["v"])] for i in range(cfg.n_layers)]
    h = _dequant(src, "token_embd.weight")[fb.tokens.long()]
    for i in range(cfg.n_layers):
        w = lambda n: _dequant(src, "blk.%d.%s.weight" % (i, n))  # noqa: E731
        x = _rms(h, cfg.rms_eps) * w("attn_norm").view(-1)
        q = _turn((x @ w("attn_q").T).view(-1, Hq, D), pos, cfg.rope_base)
        new = [_turn((x @ w("attn_k").T).view(-1, Hk, D), pos, cfg.rope_base), (x @ w("attn_v").T).view(-1, Hk, D)]
        a = torch.empty(q.shape, dtype=F64, device=DEV)
        for pool, y in zip(kept[i], new):
            pool[slots] = _stored(y, fmt)
        for (r0, n, p0), table in zip(_segments(case), _tables(fb)):
            at = (table.long()[:, None] * BS + torch.arange(BS, device=DEV)).view(-1)[:p0 + n]
            a[r0:r0 + n] = _attend(q[r0:r0 + n], kept[i][0][at], kept[i][1][at], pos[r0:r0 + n], D ** -0.5)
        if fmt != "q8_0":
            for pool, y in zip(kept[i], new):
                pool[slots] = y
        h = h + a.flatten(1) @ w("attn_output").T
        x = _rms(h, cfg.rms_eps) * w("ffn_norm").view(-1)
        h = h + (torch.nn.functional.silu(x @ w("ffn_gate").T) * (x @ w("ffn_up").T)) @ w("ffn_down").T
    x = _rms(h[fb.logits_idx.long()], cfg.rms_eps) * _dequant(src, "output_norm.weight").view(-1)
    out = {"logits": x @ _dequant(src, "token_embd.weight" if cfg.tie_embeddings else "output.weight").T, "k": None, "v": None}
    if fmt != "q8_0":
        for j, name in enumerate("kv"):
            out[name] = torch.stack([kept[i][j].view(-1, BS, Hk, D).transpose(1, 2) for i in range(cfg.n_layers)])
    return out


def _taps(x, w, bias, tail):
    """Causal convolution over a sequence's rows behind its carried inputs, with SiLU; and the inputs it carries on."""
    full = torch.cat([tail, x], 0)
    y = sum(w[:, j] * full[j:j + x.shape[0]] for j in range(w.shape[1]))
    return torch.nn.functional.silu(y + bias if bias is not None else y), full[x.shape[0]:]


def _exact_hybrid(case, seed):
    st = prepare(case, seed)
    m, get = _loaded("hybrid")
    cfg, fb, cache = m.cfg, st["fb"], st["cache"]
    W = lambda n: get(n).to(F64)  # noqa: E731
    sl, F = torch.nn.functional.silu, torch.nn.functional
    pos, slots, eps, seg = fb.positions.long(), fb.slots.long(), cfg.rms_eps, _segments(case)
    slot = fb.seq_state.tolist()
    states, tails = [t.to(F64) for t in cache.state], [t.to(F64) for t in cache.tails]
    pools = [[t.to(F64).view(-1, t.shape[-1]) for t in kv] if kv else None for kv in cache.kv]

    def recur(i, k, q, v, a, b, delta, skip):
        """k, q [T, H, N], v [T, H, P], a, b [T, H] -> [T, H, P]; states[i] moves on."""
        out = torch.empty_like(v)
        for j, (r0, n, p0) in enumerate(seg):
            S = states[i][slot[j]].clone() if p0 else torch.zeros_like(states[i][slot[j]])  # [H, P, N]
            for t in range(r0, r0 + n):
                S = a[t, :, None, None] * S
                u = b[t, :, None] * (v[t] - (S @ k[t, :, :, None])[..., 0] if delta else v[t])
                S = S + u[:, :, None] * k[t, :, None, :]
                out[t] = (S @ q[t, :, :, None])[..., 0]
            states[i][slot[j]] = S
        return out if skip is None else out + skip[:, None] * v

    def conv(i, x, w, bias):
        out = torch.empty_like(x)
        for j, (r0, n, p0) in enumerate(seg):
            tail = tails[i][slot[j]].clone() if p0 else torch.zeros_like(tails[i][slot[j]])
            out[r0:r0 + n], tails[i][slot[j]] = _taps(x[r0:r0 + n], w, bias, tail)
        return out

    x = W("embed")[fb.tokens.long()]
    T = x.shape[0]
    for i, L in enumerate(cfg.layers):
        p, mx = "l%d.mix." % i, L.mixer
        h = _rms(x, eps) * (1 + W("l%d.norm1" % i))
        decay = lambda raw, q=p: torch.exp(-torch.exp(W(q + "A_log")) * F.softplus(raw + W(q + "dt_bias")))  # noqa: E731
        if L.type == "parallel":
            a, r, pl, p = mx.left, mx.right, p + "left.", p + "right."
            q = _rms(_turn((h @ W(pl + "q").T).view(T, a.heads, a.dim), pos, a.rot_base), eps)
            k = _rms(_turn((h @ W(pl + "k").T).view(T, a.kv_heads, a.dim), pos, a.rot_base), eps)
            v = (h @ W(pl + "v").T).view(T, a.kv_heads, a.vdim)
            o = torch.empty(T, a.heads, a.vdim, dtype=F64, device=DEV)
            for pool, y in zip(pools[i], (k, v)):
                pool[slots] = y.flatten(1).to(torch.bfloat16).to(F64)
            for (r0, n, p0), table in zip(seg, _tables(fb)):
                at = (table.long()[:, None] * BS + torch.arange(BS, device=DEV)).view(-1)[:p0 + n]
                o[r0:r0 + n] = _attend(q[r0:r0 + n], pools[i][0][at].view(-1, a.kv_heads, a.dim), pools[i][1][at].view(-1, a.kv_heads, a.vdim), pos[r0:r0 + n], a.scale, a.chunk, True)
            for pool, y in zip(pools[i], (k, v)):
                pool[slots] = y.flatten(1)
            mix = mx.left_scale * (o.flatten(1) @ W(pl + "o").T)
            nq = r.kv_heads * r.dim
            y = conv(i, torch.cat([h @ W(p + n).T for n in "qkv"], 1), torch.cat([W(p + n + ".conv") for n in "qkv"], 0), None)
            unit = lambda z: z * torch.rsqrt((z * z).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
            q, k = (unit(z.reshape(T, r.kv_heads, r.dim)).repeat_interleave(r.heads // r.kv_heads, 1) for z in (y[:, :nq], y[:, nq:2 * nq]))
            o = recur(i, k, q * r.dim ** -0.5, y[:, 2 * nq:].reshape(T, r.heads, r.vdim), decay(h @ W(p + "a").T, p), torch.sigmoid(h @ W(p + "b").T), True, None)
            o = _rms(o, eps) * W(p + "norm") * sl(h @ W(p + "g").T).view(T, r.heads, r.vdim)
            mix = mix + mx.right_scale * (o.flatten(1) @ W(p + "o").T)
        else:
            inner, gn = mx.inner, mx.groups * mx.state
            z, xbc, dt = (h @ W(p + "in").T).split([inner, inner + 2 * gn, mx.heads], 1)
            y = conv(i, xbc, W(p + "conv"), W(p + "conv.b"))
            k, q = (t.reshape(T, mx.groups, mx.state).repeat_interleave(mx.heads // mx.groups, 1) for t in (y[:, inner:inner + gn], y[:, inner + gn:]))
            o = recur(i, k, q, y[:, :inner].reshape(T, mx.heads, mx.vdim), decay(dt, p), F.softplus(dt + W(p + "dt_bias")), False, W(p + "D"))
            o = _rms((o.flatten(1) * sl(z)).view(T, mx.norm_groups, -1), eps).view(T, inner) * W(p + "norm")
            mix = o @ W(p + "o").T
        f = "l%d.mlp." % i
        up = sl(h @ W(f + "gate").T + W(f + "gate.b")) * (h @ W(f + "up").T + W(f + "up.b"))
        x = x + mix + up @ W(f + "down").T + W(f + "down.b")
    logits = (_rms(x[fb.logits_idx.long()], eps) * (1 + W("final.norm"))) @ W("head").T
    return {"logits": logits, "state": states, "tails": tails, "kv": [t.view(s.shape) for kv, ss in zip(pools, cache.kv) if kv for t, s in zip(kv, ss)]}


def _exact_embed(case, seed):
    ids = prepare(case, seed)["ids"]
    _, src = _loaded("embed")
    c = B.BERT_BASE
    W = lambda n: torch.from_numpy(src(n)).to(DEV, F64)  # noqa: E731
    norm = lambda x, n: torch.nn.functional.layer_norm(x, (c.hidden,), W(n + ".weight"), W(n + ".bias"), c.eps)  # noqa: E731
    lin = lambda x, n: x @ W(n + ".weight").T + W(n + ".bias")  # noqa: E731
    lens = [len(x) for x in ids]
    at = torch.tensor([p for n in lens for p in range(n)], device=DEV)
    tok = torch.tensor([t for x in ids for t in x], device=DEV)
    x = norm(W("token_embd.weight")[tok] + W("position_embd.weight")[at] + W("token_types.weight")[0], "token_embd_norm")
    for i in range(c.n_layers):
        p = "blk.%d." % i
        q, k, v = (lin(x, p + "attn_" + n).view(-1, c.n_heads, c.hidden // c.n_heads) for n in "qkv")
        o, r0 = torch.empty_like(q), 0
        for n in lens:
            s = slice(r0, r0 + n)
            o[s] = _attend(q[s], k[s], v[s], torch.full((n,), n, device=DEV), (c.hidden // c.n_heads) ** -0.5)
            r0 += n
        x = norm(x + lin(o.flatten(1), p + "attn_output"), p + "attn_output_norm")
        x = norm(x + lin(torch.nn.functional.gelu(lin(x, p + "ffn_up")), p + "ffn_down"), p + "layer_output_norm")
    e = torch.stack([t.mean(0) for t in x.split(lens)])
    return e / e.norm(dim=-1, keepdim=True)
