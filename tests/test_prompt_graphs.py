"""Mixed steps of short prompts replay graphs captured with a bound on their contexts (engine/engine.py PROMPT_CTX): their prompt
attention runs the plan that known contexts get."""
import types

import numpy as np
import pytest
import torch

from localai_tfp_amd.engine.engine import EngineConfig, LLMEngine


def _engine(max_model_len=8192, head_dim=128):
    e = LLMEngine.__new__(LLMEngine)
    e.cfg = EngineConfig(max_model_len=max_model_len)
    e.use_graphs, e.recurrent, e._bounds, e.max_blocks_per_seq = True, False, {}, max_model_len // 16
    e.ws = types.SimpleNamespace(max_tokens=2048)
    e.model = types.SimpleNamespace(prefill_rows=lambda: 16, n_heads=32, n_kv=8, cfg=types.SimpleNamespace(head_dim=head_dim, attn_softcap=0.0))
    return e


def _plan(nd, rows, ctx, dec=700):
    p = {"nd": nd, "keep_hidden": False, "pf_cu": np.cumsum([0] + rows), "pf_ctx": np.asarray(ctx, np.int32)}
    return {**p, "dec_lens": np.full(nd, dec, np.int32)} if nd else p


def test_bucket_follows_the_longest_context():
    key = _engine()._graph_key
    assert key(_plan(0, [37], [37])) == (0, 64, 4, 0, 64) and key(_plan(0, [64], [65])) == (0, 64, 4, 0, 1280)
    assert key(_plan(0, [333], [1280])) == (0, 352, 4, 0, 1280) and key(_plan(0, [333], [1281])) == (0, 352, 4, 0)
    assert key(_plan(0, [30, 30], [30, 30])) == (0, 64, 4, 0, 64) and key(_plan(0, [30, 30], [30, 4000])) == (0, 64, 4, 0)
    assert key(_plan(0, [60, 60], [60, 60])) == (0, 128, 4, 0, 1280)
    assert key(_plan(127, [289], [289])) == (128, 320, 4, 1024, 1280) and key(_plan(127, [289], [9000], 2000)) == (128, 320, 4, 0)
    assert key(_plan(3, [100], [800], 5000)) == (4, 128, 4, 0, 1280)


def test_no_bound_where_the_plan_is_the_same():
    assert _engine(head_dim=256)._graph_key(_plan(0, [37], [37])) == (0, 64, 4, 0)  # another kernel, which knows no parts
    assert _engine(max_model_len=1024)._graph_key(_plan(0, [100], [100])) == (0, 128, 4, 0)  # tables too short for parts
    assert _engine(max_model_len=1024)._graph_key(_plan(0, [37], [37])) == (0, 64, 4, 0, 64)


@pytest.mark.gpu
def test_bounded_graphs_serve_the_same_tokens(monkeypatch):
    """Short, middle and long prompts through the engine's graphs against its eager steps, step by step under the eager steps' tokens, and
    the plans their captures ran.

    The paths may differ in the order of their sums (parts of K meet by atomics, in no fixed order on either path), which the 8-bit
    activations of one-row steps widen: a rounding is off by up to half a step of a block's largest number / 127, 0.0057 of the numbers' rms where
    that is 2.5 of it, sqrt 2 of that between two runs and sqrt 9 for two layers' products and the head's: 0.024 of the logits' deviation. A
    path against itself is 0.009 off, and 467 and 816 of the 60-token prompt's second step are 0.027 apart in fp32: either may win. So logits
    are compared within 0.03, and tokens where five times as much between two logits does not change the winner."""
    from localai_tfp_amd.engine import engine as E
    from localai_tfp_amd.models.config import tiny_config
    from localai_tfp_amd.models.llama import LlamaModel
    from localai_tfp_amd.models.synthetic import synthetic_source
    from localai_tfp_amd.ops import core as K
    from localai_tfp_amd.ops.sampling import SamplingParams
    from localai_tfp_amd.tokenizer import ByteTokenizer
    cfg = tiny_config(hidden=1024, ffn=1024, n_heads=8, n_kv_heads=2, head_dim=128, rope_dim=128, vocab=1024, n_layers=2)
    model = LlamaModel.load(cfg, synthetic_source(cfg, "Q4_K_M"), torch.device("cuda", 0))
    tok = ByteTokenizer(cfg.vocab)
    plans, real = [], K.flash_plan

    def spy(*a, **k):
        plans.append((a[8] if len(a) > 8 else k.get("ctx_lens_host"), real(*a, **k)))
        return plans[-1][1]
    got = {}
    for graphs in (False, True):
        eng = LLMEngine(model, tok, EngineConfig(num_blocks=400, max_num_seqs=4, max_batched_tokens=256, max_model_len=4096, use_graphs=graphs))
        monkeypatch.setattr(K, "flash_plan", spy)
        got[graphs] = []
        execute, steps = eng._execute, []

        def recorded(plan):
            lg, am = execute(plan)
            if lg.shape[0]:  # (else a chunk that is not the prompt's last)
                steps.append((lg[0].float().clone(), None if am is None else am.clone()))
                if am is not None and len(steps) <= 6:
                    am.fill_(got[False][len(got[True])][0][len(steps) - 1])
            return lg, am
        monkeypatch.setattr(eng, "_execute", recorded)
        for n in (20, 60, 200, 1400):
            ids = [(7 * i + n) % 900 + 1 for i in range(n)]
            steps.clear()
            t = eng.generate(ids, SamplingParams(temperature=0.0), max_tokens=6).token_ids
            got[graphs].append((t, [x.cpu() for x, _ in steps[:6]], [int(a[0]) for _, a in steps[:6] if a is not None]))
        if graphs:
            bounded = [p for c, p in plans if c in ([64], [1280])]
            assert bounded and all(p is None or p[1] == 1 for p in bounded) and any(p and p[1] > 1 for c, p in plans if not c)
            keys = set(eng.graphs)
            assert any(k[4:] == (64,) for k in keys) and any(k[4:] == (1280,) for k in keys) and any(k[1] and len(k) == 4 for k in keys)
        monkeypatch.setattr(K, "flash_plan", real)
        plans.clear()
        eng.shutdown()
    clear = 0
    for (t0, lg0, _), (t1, lg1, won) in zip(got[False], got[True]):
        assert t0 == t1 and len(t0) == len(lg0) == len(lg1) == len(won) == 6
        for tok, a, b, w in zip(t0, lg0, lg1, won):
            assert (a - b).norm() <= 0.03 * (a - a.mean()).norm() and w == int(b.argmax()) and tok == int(a.argmax())
            top = a.topk(2).values
            if top[0] - top[1] > 5 * 2 ** 0.5 * 0.03 * a.std():
                clear += 1
                assert w == tok
    assert clear >= 12  # of 24; 16 in fp32
    assert E.flash_plan is real
