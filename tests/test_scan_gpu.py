"""Rounds of the recurrence kernel (csrc/kernels/hybrid/hybrid_scan.hip) on the GPU against the same steps on the CPU."""
import types

import pytest
import torch

from localai_tfp_amd.ops import hybrid as HY

pytestmark = pytest.mark.gpu


def _rag(n_dec, chunks, at, slots, dev):
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)  # noqa: E731
    cu = [0]
    for c in chunks:
        cu.append(cu[-1] + c)
    pos = [p for p, c in zip(at, [1] * n_dec + chunks) for p in range(p, p + c)]
    return HY.Ragged(types.SimpleNamespace(
        T=len(pos), n_decode=n_dec, positions=i32(pos), seq_state=i32(slots), slots=i32([-1] * len(pos)), pf_cu_q=i32(cu),
        pf_q_lens_host=chunks, pf_ctx_lens_host=[p + c for p, c in zip(at[n_dec:], chunks)], pf_block_tables=None, pf_ctx_lens=None,
        dec_block_tables=None, dec_seq_lens=None, dec_max_len=0))


@pytest.mark.parametrize("N,P", [(16, 64), (32, 5), (33, 16), (64, 17), (128, 16), (100, 33), (256, 20)])
@pytest.mark.parametrize("delta,channel,nout", [(True, False, False), (False, False, True), (False, True, False), (True, True, False)])
def test_rounds_of_tokens(N, P, delta, channel, nout):
    """Chunks that end just before, at and after a round of 8 or 16 tokens, beside decode rows, with and without padding of N.
    Both sides sum in fp32, in another order: a share of 2^-24 per step and term of sums whose terms shrink with the decay, some
    40 steps of up to 256 terms, stays below 2e-5 of the largest output."""
    g = torch.Generator().manual_seed(N)
    H, G, chunks = 2, 1, [1, 7, 8, 9, 15, 16, 17, 33, 48]
    n_dec, T = 2, 2 + sum(chunks)
    k = torch.randn(T, G * N, generator=g) * N ** -0.5
    q, v = torch.randn(T, G * N, generator=g), torch.randn(T, H * P, generator=g)
    decay = torch.rand(T, H * N if channel else H, generator=g)
    coef = torch.rand(T, H, generator=g)
    skip = None if delta or nout else torch.randn(H, generator=g)  # (no caller has a skip term beside a normaliser)
    slots = list(range(n_dec + len(chunks)))
    at = [3, 0] + [0, 5] * 5
    start = torch.randn(len(slots), H, P + nout, N, generator=g)
    got = {}
    for dev in ("cpu", "cuda"):
        state, out = start.clone().to(dev), torch.zeros(T, H * P, device=dev)
        no = torch.zeros(T, H, device=dev) if nout else None
        HY.state_scan(k.to(dev), q.to(dev), v.to(dev), decay.to(dev), coef.to(dev), None if skip is None else skip.to(dev), state,
                      _rag(n_dec, chunks, at[:len(slots)], slots, dev), out, H, G, N, P, delta, channel, 0.5, False, no)
        got[dev] = [t.cpu() for t in (out, state, no) if t is not None]
    for a, b in zip(got["cuda"], got["cpu"]):
        assert (a - b).abs().max() <= 2e-5 * b.abs().max()
