"""Load-time GEMM autotuner for the quantised-weight kernels (qmm2.hip, qmm3.hip, qmm4.hip, qmmr.hip).

The K-quant GEMMs run one workgroup per CU (up to 150 KB of LDS each), so a launch's time is set by how its
(row tile x column tile x K split) grid quantises onto the 256 CUs — a hand-written M -> tile rule mispicks
badly between its breakpoints (qkv 6144 x 4096: 55 us at M = 384 against 41 us at M = 512 with the rule's picks,
profiles/r5_gemm_curve.md). Instead, every distinct (N, K, block format, epilogue class) of a loaded model is
timed on the GPU it runs on, for each M bucket the engine produces, over every compiled tile / split
candidate; the fastest plan per bucket is kept in TUNED and ops/linear.py dispatches from it. A plan is
("q2", wm, ks, wn, splits) | ("q3", wm, splits) | ("qr", wm, gw, kw, splits) | ("q4", blocks, splits) | ("rows", chunk) (row chunks of
`chunk`, each dispatched by its own bucket). Only kernel choice is tuned: every candidate computes the same product
(the GPU tests check every tile / split / epilogue against the fp32 reference).

A shape has 12 to 33 candidates a bucket where K cannot be split and 48 to 129 where it can, 17 launches each: 10 s for
Llama-3-8B in Q4_K_M. Results are
cached per device in $MX_TUNE_CACHE (default ~/.cache/localai_tfp_amd/gemm_tune.json) and reused.
"""
from __future__ import annotations

import json
import logging
import os
import time

import torch

log = logging.getLogger("localai_tfp_amd.autotune")

# M buckets the engine's steps fall into: decode-only batches (graph buckets) and mixed decode + prompt-chunk steps
BUCKETS = (16, 32, 64, 96, 128, 160, 192, 224, 256, 320, 384, 448, 512)
SPLITS = (1, 2, 4, 8)
# (N, K, qtype, epi, can_split) -> [(bucket, plan)] sorted by bucket
TUNED: dict[tuple, list] = {}
TUNED_PAIRS: dict[tuple, list] = {}  # (Na, Nb, K, qa, qb) -> [(bucket, plan of qmmp.hip, () where two launches are faster)]
TIMES: dict[tuple, list] = {}  # key -> [(bucket, plan, us)] of the plans tuned in this process (reports)
ENABLED = os.environ.get("MX_GEMM_TUNE", "1") != "0"


def _key(N: int, K: int, qtype: int, epi: int, can_split: bool) -> tuple:
    return (int(N), int(K), int(qtype), int(epi), bool(can_split))


def lookup(N: int, K: int, qtype: int, epi: int, can_split: bool, M: int):
    """Tuned plan for this GEMM at M rows, or None (untuned shape, or M beyond the largest bucket)."""
    ent = TUNED.get(_key(N, K, qtype, epi, can_split))
    if not ent:
        return None
    for b, plan in ent:
        if M <= b:
            return plan
    return None


def lookup_pair(Na: int, Nb: int, K: int, qa: int, qb: int, M: int):
    """Tuned plan of two weights in one launch, () where two launches won, or None (untuned, or M beyond the largest bucket)."""
    for b, plan in TUNED_PAIRS.get((int(Na), int(Nb), int(K), int(qa), int(qb)), ()):
        if M <= b:
            return plan
    return None


def candidates(M: int, N: int, K: int, qtype: int, can_split: bool) -> list[tuple]:
    from . import linear as L
    nsb = K // 256
    sp = [s for s in SPLITS if (s == 1 or can_split) and nsb // s >= 2]
    out = []
    for wm, ks, wn in L.QMM2_CONFIGS:
        bm = 32 * wm * wn
        if bm > 2 * max(M, 32) and bm > 64:  # a row tile more than twice the rows: never faster
            continue
        for s in sp:
            out.append(("q2", wm, ks, wn, s))
    if M >= 32:
        for wm in (1, 2, 3, 4):
            if 64 * wm > 2 * max(M, 64):
                continue
            for s in sp:
                out.append(("q3", wm, s))
    if M >= L.QMM4_MIN_M and not (L.NORM_FUSE or L.ROPE_FUSE):  # (nor has qmm4; it refuses accumulating products in one part)
        top, step, _ = L._QMM4_TILES[qtype]
        tiles = {-(-(-(-M // 16)) // b): b for b in range(top // step * step, 7, -step)}  # the fewest blocks for each number of tiles
        out += [("q4", b, 1) for b in tiles.values()]
        if can_split:  # parts that make one round of workgroups
            out += [("q4", b, s) for t, b in tiles.items() if (s := min(L.CU_COUNT // (t * -(-N // 256)), nsb // 2)) >= 2 and s * M * N <= L.QMM4_PARTS]
    if M <= L.QMMR_MAX_M and not (L.NORM_FUSE or L.ROPE_FUSE):  # (qmmr has no fused instances)
        for wm, gw, kw in L.QMMR_CONFIGS:
            if 32 * wm <= max(32, M):
                for s in sp:
                    out.append(("qr", wm, gw, kw, s))
    for c in (128, 256):
        if c < M:
            out.append(("rows", c))
    return out


def _time(fn, iters: int) -> float:
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(iters):
        fn()
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / iters * 1e3


def tune_weight(W, epi: int, can_split: bool, buckets=BUCKETS, iters: int = 8) -> list:
    """Time every candidate plan of `W` (a t32 K-quant QWeight on the GPU) at each bucket; -> [(bucket, plan)]."""
    from . import linear as L
    dev = W.data.device
    Mmax = max(buckets)
    x = (torch.randn(Mmax, W.K, device=dev) * 0.5).to(torch.float16)
    if epi in L.GLU_EPIS:
        out = torch.empty(Mmax, W.N // 2, device=dev, dtype=torch.float16)
    elif epi == L.EPI_BF16:  # 16-bit activation out: the plan runner requires out.dtype == x.dtype
        out = torch.empty(Mmax, W.N, device=dev, dtype=x.dtype)
    else:
        out = torch.zeros(Mmax, W.N, device=dev, dtype=torch.float32)
    res = []
    key = _key(W.N, W.K, int(W.qtype), epi, can_split)
    TUNED[key] = res  # "rows" plans of a bucket dispatch their chunks through the buckets tuned before it
    for b in sorted(buckets):
        xb, ob = x[:b], out[:b]
        best, best_t = None, float("inf")
        for plan in candidates(b, W.N, W.K, int(W.qtype), can_split):
            if plan[0] == "rows" and not any(bb >= plan[1] for bb, _ in res):
                continue

            def run(p=plan):
                L.run_plan(p, W, xb, epi, ob, True)
            try:
                run()
            except Exception as ex:  # a candidate the library refuses (shape limits): skip it
                log.debug("tune %s M=%d %s: %s", key, b, plan, ex)
                continue
            t = min(_time(run, iters), _time(run, iters))
            if t < best_t:
                best, best_t = plan, t
        if best is not None:
            res.append((b, best))
            TIMES.setdefault(key, []).append((b, best, round(best_t, 2)))
            log.debug("tune %s M=%d -> %s %.1f us", key, b, best, best_t)
    return res


def tune_pair(a, b, buckets=BUCKETS, iters: int = 8) -> list:
    """Time the plans of two weights in one launch beside a launch each by their own plans; -> [(bucket, plan or ())]."""
    from . import linear as L
    dev, Mmax = a.data.device, max(buckets)
    x = (torch.randn(Mmax, a.K, device=dev) * 0.5).to(torch.float16)
    out = torch.zeros(Mmax, a.N + b.N, device=dev, dtype=torch.float32)
    res = []
    for m in sorted(buckets):
        xb, ob = x[:m], out[:m]

        def apart():
            L.qmatmul(a, xb, L.EPI_F32, ob[:, :a.N], out_zeroed=True)
            L.qmatmul(b, xb, L.EPI_F32, ob[:, a.N:], out_zeroed=True)
        apart()
        best, best_t = (), min(_time(apart, iters), _time(apart, iters))
        for p in L.PAIR_PLANS:
            if 32 * p[1] > 2 * max(m, 32) or p[0] == "qr" and m > L.QMMR_MAX_M:
                continue
            for s in (s for s in SPLITS if s == 1 or a.K // 256 // s >= 2):
                def run(plan=(*p, s)):
                    L.run_pair(plan, a, b, xb, ob)
                run()
                t = min(_time(run, iters), _time(run, iters))
                if t < best_t:
                    best, best_t = (*p, s), t
        res.append((m, best))
        log.debug("tune pair %s M=%d -> %s %.1f us", (a.N, b.N, a.K), m, best, best_t)
    return res


def report() -> list[dict]:
    """The plans tuned in this process with their times (bench / profiles)."""
    return [{"N": k[0], "K": k[1], "qtype": k[2], "epi": k[3], "split": k[4],
             "plans": [[b, list(p), us] for b, p, us in v]} for k, v in TIMES.items()]


def _cache_path() -> str:
    return os.environ.get("MX_TUNE_CACHE") or os.path.join(os.path.expanduser("~"), ".cache", "localai_tfp_amd",
                                                           "gemm_tune.json")


_LIB_TAG = None


def _lib_tag() -> str:
    """Hash of the kernel library: plans tuned against another build of the kernels are not reused."""
    global _LIB_TAG
    if _LIB_TAG is None:
        import hashlib
        from .. import _native as N
        try:
            with open(N.kernel_lib_path(), "rb") as f:
                _LIB_TAG = hashlib.sha1(f.read()).hexdigest()[:12]
        except (OSError, AttributeError):
            _LIB_TAG = "unknown"
    return _LIB_TAG


def _device_tag() -> str:
    p = torch.cuda.get_device_properties(torch.cuda.current_device())
    return f"{p.name}|{getattr(p, 'gcnArchName', '')}|{p.multi_processor_count}|{_lib_tag()}"


def load_cache() -> dict:
    try:
        with open(_cache_path()) as f:
            d = json.load(f)
        return d.get(_device_tag(), {})
    except (OSError, ValueError):
        return {}


def save_cache(entries: dict):
    path = _cache_path()
    try:
        os.makedirs(os.path.dirname(path), exist_ok=True)
        try:
            with open(path) as f:
                d = json.load(f)
        except (OSError, ValueError):
            d = {}
        d.setdefault(_device_tag(), {}).update(entries)
        tmp = path + ".tmp"
        with open(tmp, "w") as f:
            json.dump(d, f)
        os.replace(tmp, path)
    except OSError as ex:
        log.warning("gemm tune cache not written (%s)", ex)


def tune_gemms(specs, buckets=BUCKETS) -> float:
    """specs: iterable of (QWeight, epi, can_split). Tunes each distinct GEMM once (cache first); -> seconds spent."""
    from . import linear as L
    if not ENABLED or not torch.cuda.is_available():
        return 0.0
    t0 = time.time()
    cache = load_cache()
    new = {}
    seen = set()
    pairs = {}
    for W, epi, can_split in specs:
        if isinstance(W, tuple):  # two weights by the same rows, tuned when each of them is
            if L.pair_ok(W):
                pairs.setdefault((W[0].N, W[1].N, W[0].K, int(W[0].qtype), int(W[1].qtype)), W)
            continue
        if (not isinstance(W, L.QWeight) or W.layout != "t32" or not W.data.is_cuda
                or int(W.qtype) not in L.QMM2_QTYPES):
            continue
        key = _key(W.N, W.K, int(W.qtype), epi, can_split)
        if key in seen:
            continue
        seen.add(key)
        ck = ",".join(map(str, key)) + "|" + ",".join(map(str, buckets)) + ("|fused" if L.NORM_FUSE or L.ROPE_FUSE else "")
        if ck in cache:
            TUNED[key] = [(b, tuple(p)) for b, p in cache[ck]]
            continue
        res = tune_weight(W, epi, can_split, buckets)
        if res:  # an empty result (every candidate refused) is not cached: the next load tunes it again
            new[ck] = [(b, list(p)) for b, p in res]
        else:
            log.warning("gemm autotune: no plan ran for %s; the untuned fallback rule serves it", key)
    for key, (a, b) in pairs.items():
        ck = "pair," + ",".join(map(str, key)) + "|" + ",".join(map(str, buckets))
        if ck in cache:
            TUNED_PAIRS[key] = [(b_, tuple(p)) for b_, p in cache[ck]]
            continue
        TUNED_PAIRS[key] = tune_pair(a, b, buckets)
        new[ck] = [(b_, list(p)) for b_, p in TUNED_PAIRS[key]]
    if new:
        save_cache(new)
    dt = time.time() - t0
    log.info("gemm autotune: %d shapes (%d tuned now) in %.1f s", len(seen), len(new), dt)
    return dt
