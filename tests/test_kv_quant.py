"""llama.cpp quantised KV-cache types (cache_type_k / cache_type_v = q8_0 / q4_0 / q4_1 / q5_0 / q5_1 / iq4_nl,
grpc-server.cpp:2338-2341) stored as real blocks (ops/kvq.py, csrc/kernels/kvq.h): bytes per token equal llama.cpp's
block sizes, the reference quantiser round-trips within each format's error, the CPU engine runs on quantised caches,
and on the GPU the quantiser kernel matches the host reference and the decode / prefill attention kernels match the
fp32 oracle on the dequantised cache."""
import numpy as np
import pytest
import torch

from localai_tfp_amd.ops import kvq as KQ

FMTS = ["q8_0", "q4_0", "q4_1", "q5_0", "q5_1", "iq4_nl"]
# relative RMS error bound of one quantise -> dequantise round trip on Gaussian rows
TOL = {"q8_0": 0.01, "q4_0": 0.12, "q4_1": 0.1, "q5_0": 0.06, "q5_1": 0.05, "iq4_nl": 0.1}


@pytest.mark.parametrize("fmt", FMTS)
def test_row_bytes_match_llamacpp_blocks(fmt):
    f = KQ.FORMATS[fmt]
    for D in (64, 128, 256):
        assert KQ.row_bytes(f, D) == KQ.BLOCK_BYTES[f] * D // 32


@pytest.mark.parametrize("fmt", FMTS)
def test_quantise_round_trip(fmt):
    f = KQ.FORMATS[fmt]
    x = np.random.default_rng(0).standard_normal((64, 128)).astype(np.float32)
    u = KQ.quantize_rows(x, f)
    y = KQ.dequantize_rows(u, f, 128)
    err = np.sqrt(((y - x) ** 2).mean() / (x ** 2).mean())
    assert err < TOL[fmt], err
    if fmt == "q8_0":  # exact llama.cpp numerics: d = amax / 127 (f16), q = round(x / d)
        d = np.abs(x.reshape(64, 4, 32)).max(-1) / 127
        q = np.clip(np.round(x.reshape(64, 4, 32) / d[..., None]), -127, 127)
        assert np.abs(q * d.astype(np.float16).astype(np.float32)[..., None] - y.reshape(64, 4, 32)).max() < 1e-6


@pytest.mark.parametrize("fmt", ["q8_0", "q4_0", "iq4_nl"])
def test_engine_cpu_runs_on_quantised_cache(fmt):
    from localai_tfp_amd.engine.engine import EngineConfig, LLMEngine
    from localai_tfp_amd.models.config import tiny_config
    from localai_tfp_amd.models.llama import LlamaModel
    from localai_tfp_amd.models.synthetic import synthetic_source
    from localai_tfp_amd.ops.sampling import SamplingParams
    from localai_tfp_amd.tokenizer import ByteTokenizer
    cfg = tiny_config(n_layers=2)
    m = LlamaModel.load(cfg, synthetic_source(cfg, "Q8_0", seed=4), "cpu")
    tok = ByteTokenizer(cfg.vocab)
    outs = {}
    for kv in ("bf16", fmt):
        eng = LLMEngine(m, tok, EngineConfig(num_blocks=64, max_num_seqs=4, max_batched_tokens=32, max_model_len=256,
                                             kv_dtype=kv))
        if kv != "bf16":
            assert eng.kv.k.dtype == torch.uint8 and eng.kv.k.shape[-1] == KQ.row_bytes(KQ.FORMATS[fmt], cfg.head_dim)
        o = eng.generate(tok.encode("quantised kv cache test prompt"), SamplingParams(temperature=0.0), max_tokens=8)
        outs[kv] = o.token_ids
    assert len(outs[fmt]) == 8
    if fmt == "q8_0":
        assert outs[fmt] == outs["bf16"]


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", FMTS)
def test_kvq_kernels_gpu(fmt):
    """kvq_append (quantiser) vs the host reference, then decode and prefill attention on the quantised cache vs the
    fp32 attention over the dequantised cache."""
    from localai_tfp_amd import _native as N
    from localai_tfp_amd.ops import core as K
    f = KQ.FORMATS[fmt]
    dev = torch.device("cuda")
    rng = np.random.default_rng(1)
    Hq, Hkv, D, bs, nb = 8, 2, 128, 16, 32
    RB = KQ.row_bytes(f, D)
    T = 80
    kc = torch.zeros(nb, Hkv, bs, RB, dtype=torch.uint8, device=dev)
    vc = torch.zeros_like(kc)
    ks = torch.from_numpy(rng.standard_normal((T, Hkv, D)).astype(np.float32)).to(torch.bfloat16).to(dev)
    vs = torch.from_numpy(rng.standard_normal((T, Hkv, D)).astype(np.float32)).to(torch.bfloat16).to(dev)
    blocks = [3, 7, 1, 12, 20]  # one sequence's block table
    slots = torch.tensor([blocks[t // bs] * bs + t % bs for t in range(T)], dtype=torch.int32, device=dev)
    N.kcall("mxk_kvq_append", f, ks.data_ptr(), vs.data_ptr(), slots.data_ptr(), T, Hkv, D, bs, kc.data_ptr(),
            vc.data_ptr(), N.stream_ptr())
    torch.cuda.synchronize()
    ref = KQ.quantize_rows(ks.float().cpu().reshape(-1, D), f).reshape(T, Hkv, RB)
    got = np.stack([kc[blocks[t // bs], :, t % bs].cpu().numpy() for t in range(T)])
    # codes may differ by one step where x / d lands within rounding of a boundary (fma vs mul + add)
    gd = KQ.dequantize_rows(got.reshape(-1, RB), f, D)
    rd = KQ.dequantize_rows(ref.reshape(-1, RB), f, D)
    assert np.abs(gd - rd).max() <= 0.02 * np.abs(rd).max() and (gd != rd).mean() < 0.01
    kc.kvf = vc.kvf = f
    # decode: one query per sequence (the same sequence twice, lengths 80 and 57)
    bt = torch.tensor([blocks + [0] * 3] * 2, dtype=torch.int32, device=dev)
    lens = torch.tensor([T, 57], dtype=torch.int32, device=dev)
    q = torch.randn(2, Hq, D, device=dev).to(torch.bfloat16)
    out = torch.empty_like(q)
    K.attn_decode(q, kc, vc, bt, lens, D ** -0.5, out, part_size=64)
    kd = torch.from_numpy(KQ.dequantize_rows(kc.cpu().reshape(-1, RB), f, D)).view(nb, Hkv, bs, D)
    vd = torch.from_numpy(KQ.dequantize_rows(vc.cpu().reshape(-1, RB), f, D)).view(nb, Hkv, bs, D)
    for b in range(2):
        L = int(lens[b])
        r = K._attn_ref_one(q[b:b + 1].cpu().float(), kd, vd, bt[b].cpu(), L, L - 1, D ** -0.5, bs)[0]
        assert float((out[b].float().cpu() - r).norm() / r.norm()) < 2e-2
    # prefill: the last 24 positions of the sequence as a chunk over the cached prefix
    ql = 24
    qp = torch.randn(ql, Hq, D, device=dev).to(torch.bfloat16)
    op = torch.empty_like(qp)
    cu = torch.tensor([0, ql], dtype=torch.int32, device=dev)
    ctx = torch.tensor([T], dtype=torch.int32, device=dev)
    K.attn_prefill(qp, kc, vc, bt[:1], cu, ctx, D ** -0.5, op, [ql], [T])
    r = K._attn_ref_one(qp.cpu().float(), kd, vd, bt[0].cpu(), T, T - ql, D ** -0.5, bs)
    assert float((op.float().cpu() - r).norm() / r.norm()) < 2e-2


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["q8_0", "q4_0", "q5_1"])
def test_engine_gpu_quantised_cache(fmt):
    """The GPU engine (graphs) on a quantised cache generates like the CPU engine on the same cache type (short
    greedy continuation), and q8_0 matches bf16 greedily."""
    from localai_tfp_amd.engine.engine import EngineConfig, LLMEngine
    from localai_tfp_amd.models.config import tiny_config
    from localai_tfp_amd.models.llama import LlamaModel
    from localai_tfp_amd.models.synthetic import synthetic_source
    from localai_tfp_amd.ops.sampling import SamplingParams
    from localai_tfp_amd.tokenizer import ByteTokenizer
    cfg = tiny_config(n_layers=2, hidden=512, ffn=1024, n_heads=8, n_kv_heads=2, head_dim=64, rope_dim=64)
    src = synthetic_source(cfg, "Q4_K_M", seed=5)
    mg = LlamaModel.load(cfg, src, "cuda")
    tok = ByteTokenizer(cfg.vocab)
    eng = LLMEngine(mg, tok, EngineConfig(num_blocks=256, max_num_seqs=4, max_batched_tokens=64, max_model_len=512,
                                          kv_dtype=fmt))
    outs = [eng.generate(tok.encode(f"quantised kv {i} " * 6), SamplingParams(temperature=0.0, ignore_eos=True),
                         max_tokens=16) for i in range(3)]
    assert all(len(o.token_ids) == 16 for o in outs)
    assert eng.kv.k.dtype == torch.uint8


@pytest.mark.gpu
@pytest.mark.parametrize("D,neox,bias,norm", [(128, False, False, False), (128, True, True, True), (64, False, True, True), (64, True, False, False)])
@pytest.mark.parametrize("T,Hq,Hkv", [(1, 4, 1), (9, 6, 3), (700, 5, 5)])
def test_rotation_quantises_q8_0_rows(D, neox, bias, norm, T, Hq, Hkv):
    """Rotation into a q8_0 cache against rotation into bf16 rows that are then quantised: the same rounding to bf16 and the same codes
    (a product and sum that the two fuse differently may move a code by one), rows without a slot left alone."""
    from localai_tfp_amd import _native as N
    from localai_tfp_amd.ops import core as K
    f, bs, g = KQ.FORMATS["q8_0"], 16, torch.Generator().manual_seed(T + D)
    qkv = torch.randn(T, (Hq + 2 * Hkv) * D, generator=g)
    qkv[0, (Hq + Hkv) * D:(Hq + Hkv) * D + 32] = 0.0  # a block of zeros
    b = torch.randn((Hq + 2 * Hkv) * D, generator=g).cuda() if bias else None
    qk = (torch.rand(D, generator=g).cuda() + 0.5, torch.rand(D, generator=g).cuda() + 0.5, 1e-6) if norm else None
    pos, nb = torch.randint(0, 5000, (T,), generator=g, dtype=torch.int32).cuda(), -(-T // bs) + 1
    slots = torch.randperm(nb * bs, generator=g)[:T].to(torch.int32)
    slots[T // 2:T // 2 + T // 8] = -1
    slots = slots.cuda()
    inv = (10000.0 ** (-torch.arange(0, D, 2).double() / D)).float().cuda()
    q = [torch.zeros(T, Hq, D, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    kc, vc, kr, vr = (torch.full((nb, Hkv, bs, KQ.row_bytes(f, D)), 77, dtype=torch.uint8, device="cuda") for _ in range(4))
    ks, vs = (torch.zeros(T, Hkv, D, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    x = qkv.cuda()
    K.rope_kv(x, b, pos, slots, inv, 1.0, Hq, Hkv, D, D, neox, q[0], KQ.tag(kc, f), KQ.tag(vc, f), bs, qk_norm=qk, zero_after=True)
    assert not x.any()
    K.rope_kv(qkv.cuda(), b, pos, torch.arange(T, dtype=torch.int32, device="cuda"), inv, 1.0, Hq, Hkv, D, D, neox, q[1], ks, vs, 1, qk_norm=qk)
    N.kcall("mxk_kvq_append", f, ks.data_ptr(), vs.data_ptr(), slots.data_ptr(), T, Hkv, D, bs, kr.data_ptr(), vr.data_ptr(), N.stream_ptr())
    assert torch.equal(q[0], q[1])
    for got, want in ((kc, kr), (vc, vr)):
        codes = (got[..., :D].view(torch.int8).int() - want[..., :D].view(torch.int8).int()).abs()
        scales = (got[..., D:].contiguous().view(torch.float16).float() - want[..., D:].contiguous().view(torch.float16).float()).abs()
        assert codes.max() <= 1 and (codes > 0).float().mean() < 0.01 and (scales <= 2 ** -8 * want[..., D:].contiguous().view(torch.float16).float().abs()).all()
