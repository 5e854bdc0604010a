"""BERT-family encoder for embeddings and cross-encoder reranking.

Parity target: the reference serves these through llama.cpp's `bert` GGUF architecture (embeddings
with mean / CLS pooling + L2 normalisation, grpc-server.cpp send_embedding) and the Python
sentence-transformers / rerankers backends (backend/python/transformers/backend.py:286-322,
backend/python/rerankers/backend.py:72-91).

MI355X path: 16-bit activations (the library's act16 format) in packed rows, no padding (encoder.hip): embeddings, LayerNorms
with the fp32 residual sum, GELU and pooling in one pass each, attention on the fused MFMA flash kernel (attention_dense.hip);
all layers run from one native call, few rows on 16-column GEMMs (encoder.hip), more on tiles with bias and GELU in their epilogues
(dense16_enc.hip); feed-forwards that are not whole 64s wide multiply on hipBLASLt. Shapes encoder.hip does not take run padded, the LayerNorms on norm.hip. Weights load from GGUF (llama.cpp `bert` /
`nomic-bert` / `jina-bert-v2` tensor names, any ggml type -> dequantised to 16-bit) or are
random-initialised for `synthetic:bert-*`.
"""
from __future__ import annotations

import ctypes
import math
from dataclasses import dataclass

import numpy as np
import torch
import torch.nn.functional as F

from .. import _native as N
from ..ops import core as K
from ..ops.dense import ENC_SMALL_ROWS, encoder_plan, small_rows  # noqa: F401
from ..ops.linear import ACT_DTYPE

# packed rows up to which encoder.hip's 16-column GEMMs run the layers. Whole embed calls, us, these / tiles (dense16_enc.hip): 768 x 3072, 12 layers, 19 / 64 /
# 65 / 128 / 448 rows 371 / 519, 490 / 551, 587 / 563, 633 / 568, 1092 / 608; 1024 x 4096, 8 layers, 64 / 65 385 / 425, 455 / 422; 1536 x 6144 33 / 48 / 65 408 / 426,
# 457 / 449, 529 / 412. Beyond, the library's GEMMs issued from Python and a pass for GELU before / tiles: 384 x 1536 600 / 3000 rows 1360 / 508, 1393 / 732; 768 x 3072
# 600 / 1700 / 6428 / 12000 rows 1378 / 640, 1392 / 1036, 2450 / 2191, 4233 / 3602; 1024 x 4096 1000 / 6428 927 / 617, 2288 / 2232; 2048 x 8192, 4 layers, 100 /
# 1700 / 12000 492 / 352, 1043 / 924, 5407 / 4938 (6428 rows 2769 / 2837).
ENC_FEW_ROWS = 64
# layers of fewer weights than this run on them up to as many more rows. The layers alone, captured, us, these / tiles: 4 of 128 x 512 at 447 rows 106 / 121, 256 x
# 1024 at 128 / 300 / 400 rows 114 / 119, 136 / 140, 154 / 154, 512 x 2048 at 65 / 128 / 200 120 / 139, 124 / 144, 165 / 158, 640 x 2560 at 65 / 100 157 / 159, 165 /
# 162; 6 of 384 x 1536 at 65 / 128 / 200 196 / 198, 201 / 203, 233 / 224, 768 x 3072 at 64 / 65 225 / 217, 264 / 243
ENC_FEW_WEIGHTS = 6_400_000


def few_rows(hidden: int, ffn: int) -> int:
    """Packed rows up to which the layers run on encoder.hip's 16-column GEMMs where dense16.hip's tiles take the widths too."""
    weights = 4 * hidden * hidden + 2 * hidden * ffn
    return min(small_rows(hidden, ffn), ENC_FEW_ROWS * max(weights, ENC_FEW_WEIGHTS) // weights)


@dataclass
class BertConfig:
    vocab: int = 30522
    hidden: int = 768
    n_layers: int = 12
    n_heads: int = 12
    ffn: int = 3072
    max_pos: int = 512
    type_vocab: int = 2
    eps: float = 1e-12
    pooling: str = "mean"  # mean | cls | last | none | rank
    act: str = "gelu"
    name: str = "bert"

    @classmethod
    def from_gguf_metadata(cls, md: dict) -> "BertConfig":
        a = str(md.get("general.architecture", "bert"))

        def g(k, d=None):
            return md.get(f"{a}.{k}", d)
        pool = {0: "none", 1: "mean", 2: "cls", 3: "last", 4: "rank"}.get(int(g("pooling_type", 1) or 1), "mean")
        toks = md.get("tokenizer.ggml.tokens") or []
        return cls(vocab=len(toks) or int(g("vocab_size", 30522)), hidden=int(g("embedding_length")),
                   n_layers=int(g("block_count")), n_heads=int(g("attention.head_count")),
                   ffn=int(g("feed_forward_length")), max_pos=int(g("context_length", 512)),
                   eps=float(g("attention.layer_norm_epsilon", 1e-12)), pooling=pool, name=str(md.get("general.name", a)))


BERT_BASE = BertConfig()
BERT_TINY = BertConfig(vocab=400, hidden=128, n_layers=2, n_heads=2, ffn=512, max_pos=128, name="bert-tiny")


def attn_blocks(rows: np.ndarray, queries: int) -> np.ndarray | None:
    """The attention's blocks of `queries` rows of each text, [blocks, 2] = (text, first row), the longest texts' first. None: more than a grid
    takes (they run in the texts' order)."""
    order = np.argsort(-rows, kind="stable")
    n = -(-rows[order] // queries)
    first = np.cumsum(n) - n
    if first[-1] + n[-1] > 65535:
        return None
    return np.stack([np.repeat(order, n), (np.arange(n.sum()) - np.repeat(first, n)) * queries], 1).astype(np.int32)


class BertModel:
    def __init__(self, cfg: BertConfig, device="cpu"):
        self.cfg = cfg
        self.device = torch.device(device)
        self.dtype = ACT_DTYPE if self.device.type == "cuda" else torch.float32
        self.w: dict[str, torch.Tensor] = {}
        # tensors in the order encoder.hip takes them: the embeddings', then 12 a layer
        H, d, f32 = cfg.hidden, self.dtype, torch.float32
        mats = [("qkv", (3 * H, H), d), ("attn_output", (H, H), d), ("attn_output_norm", (H,), f32), ("ffn_up", (cfg.ffn, H), d),
                ("ffn_down", (H, cfg.ffn), d), ("layer_output_norm", (H,), f32)]
        self._names = ["token_embd.weight", "position_embd.weight", "token_types.weight", "token_embd_norm.weight",
                       "token_embd_norm.bias"] + [f"blk.{i}.{n}.{x}" for i in range(cfg.n_layers) for n, _, _ in mats
                                                  for x in ("weight", "bias")]
        self._want = [(torch.Size(s if x == 0 else s[:1]), t, x == 0) for _, s, t in mats for x in (0, 1)]
        self.has_cls_head = False

    # ------------------------------------------------------------------ loading
    @classmethod
    def load(cls, cfg: BertConfig, get_tensor, device="cpu") -> "BertModel":
        """get_tensor(name) -> np.float32 array (or None). llama.cpp bert tensor names."""
        m = cls(cfg, device)
        dt = m.dtype

        def put(name, key=None, f32=False):
            a = get_tensor(name)
            if a is None:
                return None
            t = torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(m.device)
            m.w[key or name] = t if f32 else t.to(dt)
            return m.w[key or name]
        put("token_embd.weight", f32=True)
        put("position_embd.weight", f32=True)
        put("token_types.weight", f32=True)
        put("token_embd_norm.weight", f32=True)
        put("token_embd_norm.bias", f32=True)
        for i in range(cfg.n_layers):
            p = f"blk.{i}."
            q, k, v = (get_tensor(p + f"attn_{x}.weight") for x in "qkv")
            if q is not None:
                m.w[p + "qkv.weight"] = torch.from_numpy(np.concatenate([q, k, v], 0).astype(np.float32)).to(
                    m.device).to(dt)
                bs = [get_tensor(p + f"attn_{x}.bias") for x in "qkv"]
                if bs[0] is not None:
                    m.w[p + "qkv.bias"] = torch.from_numpy(np.concatenate(bs, 0).astype(np.float32)).to(m.device).to(dt)
            else:  # fused qkv (nomic-bert / jina)
                put(p + "attn_qkv.weight", p + "qkv.weight")
                put(p + "attn_qkv.bias", p + "qkv.bias")
            for n in ("attn_output", "ffn_up", "ffn_down", "ffn_gate"):
                put(p + n + ".weight")
                put(p + n + ".bias")
            for n in ("attn_output_norm", "layer_output_norm"):
                put(p + n + ".weight", f32=True)
                put(p + n + ".bias", f32=True)
        # cross-encoder head (rerankers): cls.weight/bias (+ optional cls.output)
        if put("cls.weight") is not None:
            put("cls.bias")
            put("cls.output.weight")
            put("cls.output.bias")
            m.has_cls_head = True
        return m

    # ------------------------------------------------------------------ forward
    def _linear(self, x, name, act: str | None = None):
        W = self.w[name + ".weight"]
        b = self.w.get(name + ".bias")
        y = torch.addmm(b, x, W.t()) if b is not None else x @ W.t()
        if act == "gelu":
            y = F.gelu(y)
        return y

    def _ln(self, h: torch.Tensor, name: str, out: torch.Tensor, residual: torch.Tensor | None = None):
        K.layernorm(h, self.w[name + ".weight"], self.w.get(name + ".bias"), self.cfg.eps, out, residual=residual)
        return out

    # ---- packed rows (GPU) ----
    def _packed_weights(self, ids):
        """(tensors, addresses) in the order encoder.hip takes them, or None where the batch runs padded: encoder.hip wants
        16-bit weights on the GPU, head dims 64 / 128, widths in whole 16-byte pieces and 16-byte aligned rows."""
        cfg, w = self.cfg, self.w
        H = cfg.hidden
        if self.device.type != "cuda" or not any(map(len, ids)) or H % 32 or H > 4096 or cfg.ffn % 32 or H % cfg.n_heads \
                or H // cfg.n_heads not in (64, 128) or len(ids) > 65535:
            return None
        ts = [w.get(n) for n in self._names]
        for (shape, dtype, need), t in zip(self._want * cfg.n_layers, ts[5:]):
            if t is None:
                if need:
                    return None
            elif t.shape != shape or t.dtype != dtype or not t.is_contiguous() or not t.is_cuda:
                return None
        for t, need in zip(ts, (1, 1, 0, 1, 0)):
            if t is None:
                if need:
                    return None
            elif t.shape[-1] != H or t.dtype != torch.float32 or not t.is_contiguous() or not t.is_cuda:
                return None
        ptrs = [None if t is None else t.data_ptr() for t in ts]
        return None if any(p is not None and p & 15 for p in ptrs) else (ts, ptrs)

    def _encode_packed(self, ts, ids, types=None, last=False):
        """-> (16-bit rows [R, H] of the texts one after another, first rows [B + 1], lengths [B], both int32 on the device).
        An empty text keeps one row that sees no key, as a padded batch has it: its first one or (last) the batch's last position,
        which is what the row before the first is there."""
        cfg, dev = self.cfg, self.device
        B, H, Fd = len(ids), cfg.hidden, cfg.ffn
        ts, ptrs = ts
        tokens, positions, kinds = ts[:3]
        lens = np.fromiter((len(x) for x in ids), np.int64, B)
        rows = np.maximum(lens, 1)
        cu = np.zeros(B + 1, np.int64)
        np.cumsum(rows, out=cu[1:])
        R, S = int(cu[-1]), int(rows.max())
        tiled = H % 64 == 0 and Fd % 64 == 0 and R > few_rows(H, Fd)
        blocks = attn_blocks(rows, 64 if H // cfg.n_heads == 64 else 128) if tiled and B > 1 else None
        nb = 0 if blocks is None else blocks.shape[0]
        # pinned, so that the copy is queued and the host goes on to the next call while this one runs (one text of 19 tokens after
        # another 374 -> 347 us a call: before, each copy waited for the call before it). A capture refuses pageable memory as it did: its
        # graph would read the image again.
        queued = not torch.cuda.is_current_stream_capturing()
        host = torch.zeros(3 * R + 2 * B + 1 + 2 * nb, dtype=torch.int32, pin_memory=queued)
        img = host.numpy()
        tok, pos, typ = img[:R], img[R:2 * R], img[2 * R:3 * R]
        pos[:] = np.arange(R) - np.repeat(cu[:-1], rows)
        if last:
            pos[cu[:-1][lens == 0]] = S - 1

        def pack(dst, lists, limit, what):
            for i, n in enumerate(lens.tolist()):
                if n:
                    dst[cu[i]:cu[i] + n] = lists[i]
            lo, hi = int(dst.min()), int(dst.max())
            if lo < 0:  # (an index from the end, as tensors take it)
                dst[dst < 0] += limit
                lo = int(dst.min())
            if lo < 0 or hi >= limit:
                raise IndexError(f"{what} outside the table of {limit}")
        pack(tok, ids, tokens.shape[0], "token")
        if types is not None and kinds is not None:
            pack(typ, types, kinds.shape[0], "token type")
        if S > positions.shape[0]:
            raise IndexError(f"text of {S} tokens, {positions.shape[0]} positions")
        img[3 * R:3 * R + B + 1] = cu
        img[3 * R + B + 1:3 * R + 2 * B + 1] = lens
        if nb:
            img[3 * R + 2 * B + 1:] = blocks.reshape(-1)
        img = host.to(dev, non_blocking=queued)
        cu_d, len_d = img[3 * R:3 * R + B + 1], img[3 * R + B + 1:3 * R + 2 * B + 1]
        x = torch.empty(R, H, dtype=self.dtype, device=dev)
        attn = torch.empty(R, H, dtype=self.dtype, device=dev)
        N.ensure_act(self.dtype)
        st = N.stream_ptr()
        N.kcall("mxk_enc_embed", img.data_ptr(), R, *ptrs[:5], H, float(cfg.eps), x.data_ptr(), st)
        scale = 1.0 / math.sqrt(H // cfg.n_heads)
        if tiled:
            plan, keep = encoder_plan(R, H, Fd), R <= small_rows(H, Fd)
            plan = [n if i not in (2, 5) or n > 1 or keep else 0 for i, n in enumerate(plan)]  # 0 parts: 16-bit sums
            most = max(plan[2], plan[5])
            qkv, up = (torch.empty(R, n, dtype=self.dtype, device=dev) for n in (3 * H, Fd))
            try:
                parts = torch.empty(most, R, H, dtype=torch.float32, device=dev) if most else None
            except torch.cuda.OutOfMemoryError:  # (up to 128 MB; undivided products need one part or none)
                plan[2] = plan[5] = int(keep)
                parts = torch.empty(R, H, dtype=torch.float32, device=dev) if keep else None
            N.kcall("mxk_enc_layers_tiled", (ctypes.c_void_p * (12 * cfg.n_layers))(*ptrs[5:]), cfg.n_layers, x.data_ptr(), R, B, S, cu_d.data_ptr(), len_d.data_ptr(), H,
                    cfg.n_heads, Fd, scale, float(cfg.eps), qkv.data_ptr(), attn.data_ptr(), N.ptr(parts), up.data_ptr(), (ctypes.c_int * 6)(*plan),
                    img.data_ptr() + 4 * (3 * R + 2 * B + 1) if nb else None, nb, st)
            return x, cu_d, len_d
        if R <= small_rows(H, Fd):
            parts = torch.empty(5, R, H, dtype=torch.float32, device=dev)  # fp32 sums of up to four parts of K, and a norm's rows
            qkv, up = (torch.empty(R, n, dtype=self.dtype, device=dev) for n in (3 * H, Fd))
            N.kcall("mxk_enc_layers", (ctypes.c_void_p * (12 * cfg.n_layers))(*ptrs[5:]), cfg.n_layers, x.data_ptr(), R, B, S, cu_d.data_ptr(), len_d.data_ptr(), H,
                    cfg.n_heads, Fd, scale, float(cfg.eps), qkv.data_ptr(), attn.data_ptr(), parts.data_ptr(), up.data_ptr(), st)
            return x, cu_d, len_d

        def linear(a, W, b):
            return torch.addmm(b, a, W.t()) if b is not None else a @ W.t()

        def add_ln(a, g, b):  # x = LN(a + x)
            N.kcall("mxk_enc_add_ln", a.data_ptr(), x.data_ptr(), R, g.data_ptr(), N.ptr(b), H, float(cfg.eps), st)
        for i in range(5, len(ts), 12):
            wq, bq, wo, bo, g1, b1, wu, bu, wd, bd, g2, b2 = ts[i:i + 12]
            qkv = linear(x, wq, bq)
            q = qkv.data_ptr()
            N.kcall("mxk_attn_dense_ragged", q, 3 * H, q + 2 * H, 3 * H, q + 4 * H, 3 * H, attn.data_ptr(), H, B, S,
                    cfg.n_heads, H // cfg.n_heads, cu_d.data_ptr(), len_d.data_ptr(), scale, None, 0, st)
            add_ln(linear(attn, wo, bo), g1, b1)
            up = linear(x, wu, bu)
            N.kcall("mxk_enc_gelu", up.data_ptr(), up.numel(), st)
            add_ln(linear(up, wd, bd), g2, b2)
        return x, cu_d, len_d

    def encode(self, ids: list[list[int]], types: list[list[int]] | None = None) -> tuple[torch.Tensor, torch.Tensor]:
        """-> (hidden [B, S, H] fp32 after the final layer, lengths [B]). Rows past a text's length hold nothing of it."""
        cfg = self.cfg
        ts = self._packed_weights(ids)
        if ts is not None:
            x, cu, lens = self._encode_packed(ts, ids, types)
            S = max(map(len, ids))
            live = (torch.arange(S, device=x.device)[None] < (cu[1:] - cu[:-1])[:, None]).reshape(-1)
            out = torch.zeros(len(ids) * S, cfg.hidden, dtype=torch.float32, device=x.device)
            out[live] = x.float()
            return out.view(len(ids), S, cfg.hidden), torch.tensor([len(t) for t in ids], dtype=torch.int32)
        B = len(ids)
        S = max(len(x) for x in ids)
        dev = self.device
        tok = torch.zeros(B, S, dtype=torch.long)
        typ = torch.zeros(B, S, dtype=torch.long)
        lens = torch.tensor([len(x) for x in ids], dtype=torch.int32)
        for b, x in enumerate(ids):
            tok[b, :len(x)] = torch.tensor(x)
            if types is not None:
                typ[b, :len(x)] = torch.tensor(types[b])
        tok, typ = tok.to(dev), typ.to(dev)
        pos = torch.arange(S, device=dev)[None].expand(B, S)
        h = self.w["token_embd.weight"][tok] + self.w["position_embd.weight"][pos]
        if "token_types.weight" in self.w:
            h = h + self.w["token_types.weight"][typ]
        h = h.reshape(B * S, cfg.hidden).contiguous().float()
        x = torch.empty(B * S, cfg.hidden, dtype=self.dtype, device=dev)
        self._ln(h, "token_embd_norm", x)
        hd = cfg.hidden // cfg.n_heads
        lens_d = lens.to(dev)
        attn = torch.empty(B * S, cfg.hidden, dtype=self.dtype, device=dev)
        for i in range(cfg.n_layers):
            p = f"blk.{i}."
            qkv = self._linear(x, p + "qkv")
            H = cfg.hidden
            K.attn_dense(qkv[:, :H], qkv[:, H:2 * H], qkv[:, 2 * H:], attn, B, S, S, cfg.n_heads, cfg.n_heads, hd,
                         1.0 / math.sqrt(hd), causal=False, klen=lens_d)
            o = self._linear(attn, p + "attn_output")
            # post-LN BERT: h = LN(x + attn_out); the fp32 residual sum is formed inside the norm kernel
            h = o.float()
            self._ln(h, p + "attn_output_norm", x, residual=x.float())
            up = self._linear(x, p + "ffn_up", act="gelu")
            down = self._linear(up, p + "ffn_down")
            h = down.float()
            self._ln(h, p + "layer_output_norm", x, residual=x.float())
        return x.float().view(B, S, cfg.hidden), lens

    def embed(self, ids: list[list[int]], normalize: bool = True) -> torch.Tensor:
        ts = self._packed_weights(ids)
        if ts is not None:
            mode = {"cls": 1, "rank": 1, "last": 2}.get(self.cfg.pooling, 0)
            x, cu, lens = self._encode_packed(ts, ids, last=mode == 2)
            e = torch.empty(len(ids), self.cfg.hidden, dtype=torch.float32, device=x.device)
            N.kcall("mxk_enc_pool", x.data_ptr(), cu.data_ptr(), lens.data_ptr(), len(ids), self.cfg.hidden, mode,
                    int(normalize), e.data_ptr(), N.stream_ptr())
            return e
        hid, lens = self.encode(ids)
        B, S, H = hid.shape
        pool = self.cfg.pooling
        if pool == "cls" or pool == "rank":
            e = hid[:, 0]
        elif pool == "last":
            e = hid[torch.arange(B), (lens - 1).long().to(hid.device)]
        else:  # mean over valid tokens
            mask = (torch.arange(S, device=hid.device)[None] < lens.to(hid.device)[:, None]).float()
            e = (hid * mask[..., None]).sum(1) / mask.sum(1, keepdim=True).clamp_min(1)
        if normalize:
            e = e / e.norm(dim=-1, keepdim=True).clamp_min(1e-12)
        return e

    def rerank_scores(self, pairs_ids: list[list[int]], types: list[list[int]]) -> torch.Tensor:
        """Cross-encoder relevance: classification head on the [CLS] state."""
        hid, _ = self.encode(pairs_ids, types)
        c = hid[:, 0].to(self.dtype)
        y = self._linear(c, "cls")
        if "cls.output.weight" in self.w:
            y = self._linear(torch.tanh(y), "cls.output")
        return y.float()[:, 0]


def synthetic_bert(cfg: BertConfig, seed: int = 0, rerank: bool = False):
    rng = np.random.default_rng(seed)
    H, Fd = cfg.hidden, cfg.ffn
    t = {"token_embd.weight": (cfg.vocab, H), "position_embd.weight": (cfg.max_pos, H),
         "token_types.weight": (cfg.type_vocab, H), "token_embd_norm.weight": (H,), "token_embd_norm.bias": (H,)}
    for i in range(cfg.n_layers):
        p = f"blk.{i}."
        for x in "qkv":
            t[p + f"attn_{x}.weight"] = (H, H)
            t[p + f"attn_{x}.bias"] = (H,)
        t.update({p + "attn_output.weight": (H, H), p + "attn_output.bias": (H,),
                  p + "attn_output_norm.weight": (H,), p + "attn_output_norm.bias": (H,),
                  p + "ffn_up.weight": (Fd, H), p + "ffn_up.bias": (Fd,), p + "ffn_down.weight": (H, Fd),
                  p + "ffn_down.bias": (H,), p + "layer_output_norm.weight": (H,), p + "layer_output_norm.bias": (H,)})
    if rerank:
        t.update({"cls.weight": (H, H), "cls.bias": (H,), "cls.output.weight": (1, H), "cls.output.bias": (1,)})
    cache = {}

    def get(name):
        if name not in t:
            return None
        if name not in cache:
            shape = t[name]
            if name.endswith("norm.weight"):
                cache[name] = np.ones(shape, np.float32)
            elif name.endswith(".bias"):
                cache[name] = np.zeros(shape, np.float32)
            else:
                cache[name] = (rng.standard_normal(shape) * 0.02).astype(np.float32)
        return cache[name]
    return get


def gguf_tensor_source(reader):
    from ..ops.quant import dequantize

    def get(name):
        ti = reader.tensors.get(name)
        if ti is None:
            return None
        a = dequantize(reader.tensor_bytes(name), ti.qtype, ti.shape)  # numpy shape = reversed(ggml shape)
        return a if len(ti.shape) > 1 else a.reshape(-1)
    return get
