// attention.hip — paged GQA attention for the LLM worker (K4/K5 of SURVEY §2.6).
//
// KV cache layout (written by rope_kv.hip): [num_blocks][Hkv][block_size][D] bf16, or fp8 e4m3
// (KV8: half the bytes per position; widened to fp32 in registers / to bf16 while staging to LDS), or rows of the
// llama.cpp block formats q8_0 / q4_0 / q4_1 / q5_0 / q5_1 / iq4_nl (kvq.h; written by kvq.hip, dequantised to bf16
// in registers like fp8 — the decode-MFMA and prefill kernels take the format as template KVF).
//
// decode  (one query token per sequence): memory-bound split-K over context partitions. A 256-thread
//   workgroup owns (sequence, kv-head, partition); D/8 lanes cover one cached position with 16-byte
//   loads, so a wave streams 64*16 B of K (then V) per step; all G = Hq/Hkv query heads of the kv
//   head are scored from the same K/V bytes (GQA packing: K/V are read once per kv head, not per q
//   head). Online softmax in the log2 domain; partitions merge in attn_decode_reduce.
// prefill (varlen, causal, paged context incl. cached prefix): attention_flash.hip; here the form for head dim 256 and for
//   contexts of one key tile (ops/core.py flash_plan): flash-attention forward on MFMA 16x16x32 bf16. A workgroup holds 16 query
//   rows x up to 8 query heads of one kv head (one wave per head) so every K/V tile staged in LDS is reused by all heads of the group. K is stored
//   XOR-swizzled for conflict-free ds_read_b128 B-fragments; V is read with ds_read_b64_tr_b16
//   (hardware transpose) from a region-swizzled image; P goes register -> LDS -> A-fragment.
#include <type_traits>

#include "kvq.h"

#define LOG2E 1.4426950408889634f

// Pages a decode partition lists in LDS. A partition that starts inside a page touches part_size / bs + 2 of them at most: 257
// where the launchers' limit of part_size / bs + 1 <= 256 is met.
constexpr int DEC_MAXB = 257;

// ------------------------------------------------------------------------------------------------
template <int D, int G, bool F16, bool KV8>
__global__ __launch_bounds__(256) void attn_decode_kernel(const bf16_t* __restrict__ q, int q_stride,
                                                          const void* __restrict__ kcv,
                                                          const void* __restrict__ vcv,
                                                          const int* __restrict__ block_tables, int bt_stride,
                                                          const int* __restrict__ seq_lens, int Hkv, int bs,
                                                          float scale, int window, float softcap, int part_size,
                                                          int n_parts, bf16_t* __restrict__ out, int out_stride,
                                                          float2* __restrict__ part_ml, float* __restrict__ part_o) {
    // window > 0: sliding-window attention, keys p >= L - window only (Gemma 2/3 local layers);
    // softcap > 0: scores s -> softcap * tanh(s / softcap) before the softmax (Gemma 2).
    constexpr int LPP = D / 8;        // lanes per position
    constexpr int PPW = 64 / LPP;     // positions per wave step
    constexpr int PPB = 4 * PPW;      // positions per workgroup step
    __shared__ float sm_m[4][G], sm_l[4][G];
    __shared__ float sm_o[4][G][D];
    const int kvh = blockIdx.x, b = blockIdx.y, part = blockIdx.z;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int pg = lane / LPP, dl = lane % LPP;
    const int L = seq_lens[b];
    const int p0 = part * part_size;
    const int p1 = min(L, p0 + part_size);
    const int Hq = Hkv * G;
    // partitions past the end of this sequence do nothing (the reduce kernel reads only the
    // ceil(L / part_size) live ones); graphs launch a fixed partition count for max_model_len.
    if (p0 >= L && part > 0) return;

    float qf[G][8];
    const float qs = scale * LOG2E;
    const float sc_l2 = softcap * LOG2E, sc_inv = softcap > 0.f ? 1.f / (softcap * LOG2E) : 0.f;
    const int p_start = window > 0 ? max(p0, L - window) : p0;
#pragma unroll
    for (int h = 0; h < G; ++h) {
        const uint4 raw = *(const uint4*)(q + (size_t)b * q_stride + (size_t)(kvh * G + h) * D + dl * 8);
        const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            qf[h][2 * j] = __uint_as_float(w[j] << 16) * qs;
            qf[h][2 * j + 1] = __uint_as_float(w[j] & 0xFFFF0000u) * qs;
        }
    }
    float m[G], l[G], o[G][8];
#pragma unroll
    for (int h = 0; h < G; ++h) {
        m[h] = -INFINITY;
        l[h] = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) o[h][j] = 0.f;
    }
    // The partition's block ids are staged in LDS once (no dependent global load in front of every
    // K/V fetch), and K/V are double-buffered in registers: the loads of step i+1 are in flight
    // while step i is scored, so each lane keeps 2*U 16-byte loads outstanding (memory-level
    // parallelism is what bounds this kernel, not VALU).
    __shared__ int sbt[DEC_MAXB];
    const int* bt = block_tables + (size_t)b * bt_stride;
    using kvec = typename KVVec<KV8>::T;
    constexpr int ES = KV8 ? 1 : 2;  // bytes per cached element
    const char* kc = (const char*)kcv;
    const char* vc = (const char*)vcv;
    const int blk0 = p0 / bs;
    const int nblk = p1 > p0 ? (p1 - 1) / bs - blk0 + 1 : 0;
    for (int i = threadIdx.x; i < nblk; i += 256) sbt[i] = bt[blk0 + i];
    __syncthreads();
    constexpr int U = 2;
    constexpr int STEP = PPB * U;
    // two register buffers with compile-time names (a runtime buffer index, or arrays passed by
    // reference to helpers, would put them in scratch): the step is a macro over (K, V)
    kvec ka[U], va[U], kb[U], vb[U];
#define DEC_LOAD(K, V, BASE)                                                                  \
    _Pragma("unroll") for (int u = 0; u < U; ++u) {                                           \
        const int p = (BASE) + u * PPB + wave * PPW + pg;                                     \
        if (p < p1) {                                                                         \
            const int blk = sbt[p / bs - blk0], off = p % bs;                                 \
            const size_t eo = (((size_t)blk * Hkv + kvh) * bs + off) * D + dl * 8;            \
            K[u] = __builtin_nontemporal_load((const kvec*)(kc + eo * ES));                   \
            V[u] = __builtin_nontemporal_load((const kvec*)(vc + eo * ES));                   \
        } else {                                                                              \
            K[u] = V[u] = kvec{};                                                             \
        }                                                                                     \
    }
#define DEC_CONSUME(K, V, BASE)                                                               \
    _Pragma("unroll") for (int h = 0; h < G; ++h) {                                           \
        float s[U];                                                                           \
        _Pragma("unroll") for (int u = 0; u < U; ++u) {                                       \
            float acc = 0.f, kf[8];                                                           \
            kv_unpack8<KV8>(K[u], kf);                                                        \
            _Pragma("unroll") for (int j = 0; j < 8; ++j) acc = fmaf(qf[h][j], kf[j], acc);   \
            s[u] = group_sum<LPP>(acc);                                                       \
            if (softcap > 0.f) s[u] = sc_l2 * tanhf(s[u] * sc_inv);                           \
            if ((BASE) + u * PPB + wave * PPW + pg >= p1) s[u] = -INFINITY;                   \
        }                                                                                     \
        float mx = m[h];                                                                      \
        _Pragma("unroll") for (int u = 0; u < U; ++u) mx = fmaxf(mx, s[u]);                  \
        if (mx != -INFINITY) {                                                                \
            const float a = exp2f(m[h] - mx);                                                 \
            l[h] *= a;                                                                        \
            _Pragma("unroll") for (int j = 0; j < 8; ++j) o[h][j] *= a;                       \
            _Pragma("unroll") for (int u = 0; u < U; ++u) {                                   \
                const float pr = exp2f(s[u] - mx);                                            \
                l[h] += pr;                                                                   \
                float vf[8];                                                                  \
                kv_unpack8<KV8>(V[u], vf);                                                    \
                _Pragma("unroll") for (int j = 0; j < 8; ++j) o[h][j] = fmaf(pr, vf[j], o[h][j]); \
            }                                                                                 \
            m[h] = mx;                                                                        \
        }                                                                                     \
    }
    if (p_start < p1) { DEC_LOAD(ka, va, p_start) }
    for (int base = p_start; base < p1; base += 2 * STEP) {
        if (base + STEP < p1) { DEC_LOAD(kb, vb, base + STEP) }
        DEC_CONSUME(ka, va, base)
        if (base + STEP >= p1) break;
        if (base + 2 * STEP < p1) { DEC_LOAD(ka, va, base + 2 * STEP) }
        DEC_CONSUME(kb, vb, base + STEP)
    }
#undef DEC_LOAD
#undef DEC_CONSUME
    // merge the PPW position groups of the wave (xor over lane offsets LPP, 2LPP, ...)
#pragma unroll
    for (int off = LPP; off < 64; off <<= 1) {
#pragma unroll
        for (int h = 0; h < G; ++h) {
            const float m2 = __shfl_xor(m[h], off, 64), l2 = __shfl_xor(l[h], off, 64);
            const float mn = fmaxf(m[h], m2);
            const float a1 = mn == -INFINITY ? 0.f : exp2f(m[h] - mn);
            const float a2 = mn == -INFINITY ? 0.f : exp2f(m2 - mn);
            l[h] = l[h] * a1 + l2 * a2;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float o2 = __shfl_xor(o[h][j], off, 64);
                o[h][j] = o[h][j] * a1 + o2 * a2;
            }
            m[h] = mn;
        }
    }
    if (pg == 0) {
#pragma unroll
        for (int h = 0; h < G; ++h) {
            if (dl == 0) { sm_m[wave][h] = m[h]; sm_l[wave][h] = l[h]; }
#pragma unroll
            for (int j = 0; j < 8; ++j) sm_o[wave][h][dl * 8 + j] = o[h][j];
        }
    }
    __syncthreads();
    // combine the 4 waves: thread -> (h, d)
    for (int idx = threadIdx.x; idx < G * D; idx += 256) {
        const int h = idx / D, d = idx % D;
        float mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < 4; ++w) mx = fmaxf(mx, sm_m[w][h]);
        float ls = 0.f, os = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float a = mx == -INFINITY ? 0.f : exp2f(sm_m[w][h] - mx);
            ls += sm_l[w][h] * a;
            os += sm_o[w][h][d] * a;
        }
        const int hq = kvh * G + h;
        // one partition holds the whole sequence: final output here (attn_decode_reduce skips it)
        if (n_parts == 1 || (part == 0 && L <= part_size)) {
            out[(size_t)b * out_stride + (size_t)hq * D + d] = f32_to_act<F16>(ls > 0.f ? os / ls : 0.f);
        } else {
            const size_t pi = ((size_t)b * Hq + hq) * n_parts + part;
            if (d == 0) part_ml[pi] = make_float2(mx, ls);
            part_o[pi * D + d] = os;
        }
    }
}

constexpr int DEC_RED_MAXP = 512;  // partitions whose merge weights fit the reduce kernel's LDS table

// One (sequence, query head) per workgroup. Wave 0 reads the partitions' (m, l) with all its lanes at once and publishes the
// merge weights through LDS; then groups of D / 4 threads take every n-th partition, four dims a thread and four partitions in
// flight, and their sums meet in LDS. A chain of memory latencies bounds it: 9 contexts of 3001-24001 in 256-key partitions 9.9 us
// with one group of D threads, 5.7 with eight of 32; the first four partitions of a group are asked for ahead of the weights
// (attention and merge of one context of 711 in 48-key partitions 8.65 -> 8.0 us, of 32 of 97-3879 in 128-key ones 48.9
// -> 47.8, of 192 of 300-491 in 256-key ones, head dim 64, 37.6 -> 35.6).
template <bool F16>
__global__ __launch_bounds__(256) void attn_decode_reduce_kernel(const float2* __restrict__ part_ml,
                                                                  const float* __restrict__ part_o, int n_parts,
                                                                  int Hq, int D, const int* __restrict__ seq_lens,
                                                                  int part_size, bf16_t* __restrict__ out,
                                                                  int out_stride) {
    __shared__ float wts[DEC_RED_MAXP];
    __shared__ __attribute__((aligned(16))) float sums[1024];  // [groups][D]
    __shared__ float s_mx, s_ls;
    const int bh = blockIdx.x;
    const int b = bh / Hq, h = bh % Hq;
    const int np = min(n_parts, (seq_lens[b] + part_size - 1) / part_size);
    if (np <= 1) return;  // the attention workgroup wrote this sequence's output directly
    const size_t pb = (size_t)bh * n_parts;
    const int nq = D / 4, groups = 256 / nq, grp = threadIdx.x / nq, d = threadIdx.x % nq * 4;  // (D 64, 128 or 256)
    auto at = [&](int p) { return *(const float4*)(part_o + (pb + p) * D + d); };
    float2 ml0 = make_float2(-INFINITY, 0.f);
    if (threadIdx.x < 64) ml0 = part_ml[pb + min((int)threadIdx.x, np - 1)];
    float4 o[4] = {};
#pragma unroll
    for (int u = 0; u < 4; ++u)
        if (grp + u * groups < np) o[u] = at(grp + u * groups);
    if (threadIdx.x < 64) {
        float m = ml0.x;
        for (int p = threadIdx.x + 64; p < np; p += 64) m = fmaxf(m, part_ml[pb + p].x);
        m = wave_max_all(m);
        float l = 0.f;
        for (int p = threadIdx.x; p < np; p += 64) {
            const float2 ml = p < 64 ? ml0 : part_ml[pb + p];
            const float a = m == -INFINITY ? 0.f : exp2f(ml.x - m);
            l += ml.y * a;
            if (p < DEC_RED_MAXP) wts[p] = a;
        }
        l = wave_sum_all(l);
        if (threadIdx.x == 0) { s_mx = m; s_ls = l; }
    }
    __syncthreads();
    const float mx = s_mx, L = s_ls;
    float4 os = make_float4(0.f, 0.f, 0.f, 0.f);
    auto add = [&](const float4& o, float a) {
        os.x += o.x * a;
        os.y += o.y * a;
        os.z += o.z * a;
        os.w += o.w * a;
    };
#pragma unroll
    for (int u = 0; u < 4; ++u)
        if (grp + u * groups < np) add(o[u], wts[grp + u * groups]);
    int p = grp + 4 * groups;
    for (; p + 3 * groups < min(np, DEC_RED_MAXP); p += 4 * groups) {
        const float4 o0 = at(p), o1 = at(p + groups), o2 = at(p + 2 * groups), o3 = at(p + 3 * groups);
        add(o0, wts[p]);
        add(o1, wts[p + groups]);
        add(o2, wts[p + 2 * groups]);
        add(o3, wts[p + 3 * groups]);
    }
    for (; p < np; p += groups) add(at(p), p < DEC_RED_MAXP ? wts[p] : (mx == -INFINITY ? 0.f : exp2f(part_ml[pb + p].x - mx)));
    *(float4*)(sums + grp * D + d) = os;
    __syncthreads();
    for (int e = threadIdx.x; e < D; e += 256) {
        float v = 0.f;
        for (int k = 0; k < groups; ++k) v += sums[k * D + e];
        out[(size_t)b * out_stride + (size_t)h * D + e] = f32_to_act<F16>(L > 0.f ? v / L : 0.f);
    }
}

template <int D, int G>
static int launch_decode(const bf16_t* q, int q_stride, const void* kc, const void* vc, const int* bt,
                         int bt_stride, const int* seq_lens, int B, int Hkv, int bs, float scale, int window,
                         float softcap, int part_size, int n_parts, bf16_t* out, int out_stride, float2* part_ml,
                         float* part_o, int kv8, hipStream_t st) {
    dim3 grid(Hkv, B, n_parts);
    MX_ACT_DISPATCH({
        if (kv8)
            attn_decode_kernel<D, G, F16, true><<<grid, 256, 0, st>>>(q, q_stride, kc, vc, bt, bt_stride, seq_lens,
                                                                      Hkv, bs, scale, window, softcap, part_size,
                                                                      n_parts, out, out_stride, part_ml, part_o);
        else
            attn_decode_kernel<D, G, F16, false><<<grid, 256, 0, st>>>(q, q_stride, kc, vc, bt, bt_stride, seq_lens,
                                                                       Hkv, bs, scale, window, softcap, part_size,
                                                                       n_parts, out, out_stride, part_ml, part_o);
        if (n_parts > 1)
            attn_decode_reduce_kernel<F16><<<B * Hkv * G, 256, 0, st>>>(part_ml, part_o, n_parts, Hkv * G, D, seq_lens,
                                                                        part_size, out, out_stride);
    });
#undef DQK
    MXK_CHECK_LAUNCH();
}

extern "C" int mxk_attn_decode(const bf16_t* q, int q_stride, const void* kc, const void* vc, const int* bt,
                               int bt_stride, const int* seq_lens, int B, int Hq, int Hkv, int D, int bs,
                               float scale, int window, float softcap, int part_size, int n_parts, bf16_t* out,
                               int out_stride, float2* part_ml, float* part_o, int kv8, hipStream_t st) {
    if (B <= 0) return 0;
    if (Hq % Hkv || kv8 > KVF_FP8) return (int)hipErrorInvalidValue;  // block-quantised caches: the MFMA kernel only
    const int G = Hq / Hkv;
    if (n_parts > 1 && (!part_ml || !part_o)) return (int)hipErrorInvalidValue;
    if (bs <= 0 || part_size / bs + 1 > 256) return (int)hipErrorInvalidValue;  // LDS block-id stage
#define DEC(D_, G_) \
    if (D == D_ && G == G_) return launch_decode<D_, G_>(q, q_stride, kc, vc, bt, bt_stride, seq_lens, B, Hkv, bs, scale, window, softcap, part_size, n_parts, out, out_stride, part_ml, part_o, kv8, st);
    DEC(128, 1) DEC(128, 2) DEC(128, 3) DEC(128, 4) DEC(128, 5) DEC(128, 6) DEC(128, 7) DEC(128, 8)
    DEC(64, 1) DEC(64, 2) DEC(64, 4) DEC(64, 8) DEC(256, 1) DEC(256, 2) DEC(256, 4) DEC(256, 8)
#undef DEC
    return (int)hipErrorInvalidValue;
}

// ------------------------------------------------------------------------------------------------
// prefill: MFMA flash attention over the paged cache.
// K image: row p (64 per tile) holds D/8 16-byte chunks; chunk c lives at slot c ^ fk(p).
template <int D>
MX_DEV int k_lds_off(int p, int c) {
    const int r = p & 15;
    int f;
    if constexpr (D == 128) f = r ^ (((r + 4) >> 3) & 1);
    else f = ((r >> 1) & 7) ^ (((r + 4) >> 3) & 1);
    return p * (D * 2) + ((c ^ (f & (D / 8 - 1))) << 4);
}
// V image: row p holds D/16 32-byte regions (16 dims each); region nt lives at nt ^ sv(p).
template <int D>
MX_DEV int v_lds_off(int p, int nt) {
    int sv;
    if constexpr (D == 128) sv = (p & 3) | (((p >> 3) & 1) << 2);
    else sv = ((p >> 1) & 1) | (((p >> 3) & 1) << 1);
    return p * (D * 2) + ((nt ^ sv) << 5);
}

// ------------------------------------------------------------------------------------------------
// decode on MFMA. The VALU kernel above spends its time on the per-position dot products and the
// 16-lane shuffle reductions (~30% of HBM bandwidth at B=128); here the G query heads of a kv head are
// the columns of a 16x16x32 bf16 MFMA tile, so QK^T and PV run on the matrix cores and the softmax
// happens once per 32-key tile.
//   workgroup = (kv head, sequence, partition), 4 waves; wave w takes the partition's 32-key tiles
//   w, w+4, ...: K fragments come straight from the paged cache into MFMA A operands (16-byte loads,
//   one cached position x 8 dims per lane) and S^T = K Q^T leaves a head's scores in four lanes: two lane
//   swaps give its maximum, the rest is lane-local, and the probabilities are already the B operand of
//   O^T = V^T P^T when V^T's keys are read in the order S^T's layout has them. V is staged in the wave's LDS
//   slice and read with the hardware-transposing ds_read_b64_tr_b16 (same V image as the prefill kernel). The 4
//   waves' (m, l, O) merge through LDS at the end, in the same partial-result format as attn_decode_kernel
//   (attn_decode_reduce merges partitions).
// Against the form with heads as rows (4 rows a lane, two 16-lane shuffle reductions per row and tile, P through LDS) and
// caches widened load by load: bf16 B=128 ctx 65-1021 53.1 -> 49.2 us at 512-key partitions (44.9 at 1024: 4.1 TB/s), B=9 ctx
// 3001-24001 95 -> 85; q8_0 B=9 155 -> 64 us (3.2 TB/s), fp8 147 -> 59, q4_0 151 -> 60 (1.8 TB/s, bound by the widening's
// vector work). Three waves per SIMD instead of two gave the quantised caches 73 -> 64 of that.
// A key's pool row is worked out once, by one lane, and passed to the lanes that load its numbers (a division by the page size for
// each of a lane's ten loads was half of a bf16 tile's vector instructions), masks and score caps stand in branches of their own:
// 700 -> 600 vector instructions a tile in q8_0 (320 of them the widening), 570 -> 370 in fp8. With the merge launch, us: 128 rows of
// 65-1021 keys in one partition q8_0 30.0 -> 28.6, fp8 25.5 -> 23.1; 9 rows of 3001-24001 in partitions of 256 63.0 -> 61.9, 58.5 ->
// 56.7; 32 rows of 97-4003 30.0 -> 28.8, 29.1 -> 27.3. bf16 of head dim 64 the same way 22.2 -> 20.9.
// bf16 of head dim 128, four waves, keeps mask and cap in one pass, which measures faster (why, no counter shows; fewer instructions
// between a tile's loads are no gain there: with all ten rows fetched ahead of the first load 32 rows of 97-4003 took 45.4). Before /
// with branches / so, us: 32 rows of 97-4003 39.3 / 39.7 / 39.2; 20 rows of 2000-6000 in partitions of 128 72.3 / 75.7 / 73.2; 12 rows
// of 30-200 9.4 / 9.1 / 9.0; 128 rows of 65-1021 in one 44.5 / 42.9 / 42.9. What is left of the loss is 1 % for long contexts in many
// partitions, 2 % for 32 x 1000 in four, 3 % for 48 x 100-500 in two; rows worked out by each lane again give it back, at 4 to 8 % for
// short contexts (32 rows of 30-400 13.0 / 14.1), and the host does not know which they are.
// Occupancy, not register double buffering, hides HBM latency: 8 KB of LDS per wave lets 4
// workgroups (16 waves) share a CU, each with one tile's 16 KB of K/V loads in flight.
template <int D>
constexpr int dec_wave_lds() { return 32 * D * 2; }

// maximum / sum over the lanes l, l ^ 16, l ^ 32, l ^ 48 in each of them
MX_DEV float quarters_max(float x) {
    const u32x2 a = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false));
    x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const u32x2 b = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false));
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
MX_DEV float quarters_sum(float x) {
    const u32x2 a = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false));
    x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const u32x2 b = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false));
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// NW = 16 (1024 threads, one workgroup per CU): the small-batch form — a 512-key partition per workgroup, so a
// context of <= 512 keys is ONE partition whose workgroup writes the final output (no reduce work for it).
// TS: debug instantiation writing wall-clock stamps of workgroup (0, 0, 0) wave 0 to ts[0..7] (tools/prof_attn_decode.py)
// DPF: the K-prefetch form (below; 2 waves / SIMD for its registers, MX_DECODE_PF=0 selects the 4-wave form)
// The bytes of one tile of an 8-bit or block-quantised cache as a lane holds them (16 + 16 keys of K, a half row of V),
// requested one tile ahead: wide loads (8 bytes of K, 16 of V) and one load for all of a row's block scales, not two loads
// per eight elements. Rows are 4-byte aligned.
struct __attribute__((packed, aligned(4))) DecU4 { uint32_t x[4]; };
struct __attribute__((packed, aligned(4))) DecU2 { uint32_t x[2]; };
template <int KVF, int D>
struct DecRaw {
    using Q = KVQ<KVF, D>;
    static constexpr bool KVQ_ = KVF >= KVF_Q8_0;
    static constexpr bool B8 = KVF == KVF_FP8 || Q::Q8;              // one byte per element, else four bits
    static constexpr int ROWB = KVQ_ ? Q::ROWB : D;
    static constexpr int SB = KVQ_ ? (Q::MIN ? 4 : 2) : 0;           // scale bytes per block of 32
    static constexpr int KS = D / 32;
    uint32_t kc[2][KS][B8 ? 2 : 1];
    uint32_t ks[2][KVQ_ ? (KS * SB + 3) / 4 : 1], kh[2][KVQ_ && Q::HB ? KS : 1];
    uint32_t vc[D / 2 / (B8 ? 4 : 8)];
    uint32_t vs[KVQ_ ? (KS / 2 * SB + 3) / 4 : 1], vh[KVQ_ && Q::HB ? D / 64 : 1];

    static MX_DEV void copy(uint32_t* to, const uint8_t* from, int bytes) {
        int i = 0;
        for (; i + 16 <= bytes; i += 16) {
            const DecU4 w = *(const DecU4*)(from + i);
            for (int j = 0; j < 4; ++j) to[i / 4 + j] = w.x[j];
        }
        for (; i + 8 <= bytes; i += 8) {
            const DecU2 w = *(const DecU2*)(from + i);
            to[i / 4] = w.x[0];
            to[i / 4 + 1] = w.x[1];
        }
        for (; i + 4 <= bytes; i += 4) to[i / 4] = *(const uint32_t*)(from + i);
        if (i < bytes) to[i / 4] = *(const uint16_t*)(from + i);
    }
    // K row `row`, chunks 32 ks + 8 g
    MX_DEV void load_k(int t, const void* base, size_t row, int g) {
        const uint8_t* r = (const uint8_t*)base + row * ROWB;
#pragma unroll
        for (int k = 0; k < KS; ++k) copy(kc[t][k], r + (B8 ? 32 * k + 8 * g : 16 * k + 4 * g), B8 ? 8 : 4);
        if constexpr (KVQ_) copy(ks[t], r + Q::CB + Q::HBB, KS * SB);
        if constexpr (KVQ_ && Q::HB) copy(kh[t], r + Q::CB, 4 * KS);
    }
    // half hf of V row `row`
    MX_DEV void load_v(const void* base, size_t row, int hf) {
        const uint8_t* r = (const uint8_t*)base + row * ROWB;
        constexpr int HC = D / 2 / (B8 ? 1 : 2);
        copy(vc, r + hf * HC, HC);
        if constexpr (KVQ_) copy(vs, r + Q::CB + Q::HBB + hf * (KS / 2 * SB), KS / 2 * SB);
        if constexpr (KVQ_ && Q::HB) copy(vh, r + Q::CB + hf * (D / 16), D / 16);
    }
    static MX_DEV uint4 widen(uint32_t c0, uint32_t c1, const uint32_t* sw, int blk, uint32_t hb) {
        if constexpr (KVF == KVF_FP8) return fp8x8_to_bf16x8(make_uint2(c0, c1));
        else if constexpr (KVQ_) {
            KVQRaw w;
            w.c = make_uint2(c0, c1);
            w.s = Q::MIN ? sw[blk] : (sw[blk >> 1] >> (16 * (blk & 1))) & 0xFFFF;
            w.hb = hb;
            return kvq_to_bf16x8<KVF>(w);
        } else return make_uint4(0, 0, 0, 0);
    }
    MX_DEV bf16x8 k(int t, int k_, int g) const {
        return __builtin_bit_cast(bf16x8, widen(kc[t][k_][0], B8 ? kc[t][k_][B8 ? 1 : 0] : 0u, ks[t], k_,
                                                KVQ_ && Q::HB ? (kh[t][KVQ_ && Q::HB ? k_ : 0] >> (8 * g)) & 0xFF : 0u));
    }
    MX_DEV uint4 v(int j) const {  // elements 8 j .. of the half row
        return widen(vc[B8 ? 2 * j : j], B8 ? vc[B8 ? 2 * j + 1 : 0] : 0u, vs, j >> 2,
                     KVQ_ && Q::HB ? (vh[KVQ_ && Q::HB ? j >> 2 : 0] >> (8 * (j & 3))) & 0xFF : 0u);
    }
};
// waves per SIMD: what the registers of each cache format allow without spilling
template <int KVF, int NW, bool TS, bool DPF>
constexpr int dec_waves() {
    return KVF == KVF_IQ4_NL || (KVF == KVF_BF16 && DPF && !TS && NW <= 8) ? 2 : KVF != KVF_BF16 ? 3 : 4;
}
template <int D, bool F16, int KVF, int NW = 4, bool TS = false, bool DPF = false>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(
    dec_waves<KVF, NW, TS, DPF>(), dec_waves<KVF, NW, TS, DPF>()))) void attn_decode_mfma_kernel(
    const bf16_t* __restrict__ q, int q_stride, const void* __restrict__ kcv, const void* __restrict__ vcv,
    const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ seq_lens, int Hkv, int G, int bs,
    float scale, int window, float softcap, int part_size, int n_parts, bf16_t* __restrict__ out, int out_stride,
    float2* __restrict__ part_ml, float* __restrict__ part_o, int* __restrict__ part_cnt,
    unsigned long long* __restrict__ ts = nullptr) {
    const bool ts_on = TS && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0 && threadIdx.x == 0;
#define DEC_TS(k)                                    \
    if constexpr (TS) {                              \
        __builtin_amdgcn_s_waitcnt(0);               \
        if (ts_on) ts[k] = wall_clock64();           \
    }
    DEC_TS(0)
    constexpr int KT = 32;                      // keys per wave tile
    constexpr int WB = dec_wave_lds<D>();
    constexpr int NVC = KT * D / 8 / 64;        // 16-byte V chunks per lane per tile
    constexpr bool KV8 = KVF != KVF_BF16;       // a cache widened in registers (fp8 or block-quantised)
    constexpr int ES = KV8 ? 1 : 2;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    __shared__ int sbt[DEC_MAXB];
    const int kvh = blockIdx.x, b = blockIdx.y, part = blockIdx.z;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int g = lane >> 4, col = lane & 15;
    const int p0 = part * part_size;
    const int* bt = block_tables + (size_t)b * bt_stride;
    const int blk0 = p0 / bs;
    // the partition's block-table entries (its last page's is (p0 + part_size - 1) / bs: a partition may start inside a page) are
    // requested before the sequence length and wait in a register: a partition past the context ends as soon as the length is here
    static_assert(64 * NW >= DEC_MAXB - 1, "one entry a thread, the last one apart");
    const int nbt = min((p0 + part_size - 1) / bs - blk0 + 1, bt_stride - blk0);
    const int bt_entry = (int)threadIdx.x < nbt ? bt[blk0 + threadIdx.x] : 0;
    const int L = seq_lens[b];
    const int p1 = min(L, p0 + part_size);
    if (p0 >= L && part > 0) return;  // uniform: graphs launch n_parts for max_model_len
    if ((int)threadIdx.x < nbt) sbt[threadIdx.x] = bt_entry;
    if (64 * NW < DEC_MAXB && nbt == DEC_MAXB && threadIdx.x == 0) sbt[DEC_MAXB - 1] = bt[blk0 + DEC_MAXB - 1];
    DEC_TS(1)
    const int Hq = Hkv * G;
    const int p_start = window > 0 ? max(p0, L - window) : p0;
    const float qs = scale * LOG2E;
    const float sc_l2 = softcap * LOG2E, sc_inv = softcap > 0.f ? 1.f / (softcap * LOG2E) : 0.f;
    // Q^T as the B operand: column = head (lane col), k = dims 32 ks + 8 g — requested before the block-table
    // barrier so its latency overlaps the table read
    bf16x8 qf[D / 32];
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) {
        if (col < G) qf[ks] = *(const bf16x8*)(q + (size_t)b * q_stride + (size_t)(kvh * G + col) * D + 32 * ks + 8 * g);
        else qf[ks] = (bf16x8){};
    }
    __syncthreads();
    DEC_TS(2)
    f32x4 oacc[D / 16];
#pragma unroll
    for (int i = 0; i < D / 16; ++i) oacc[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float mrow = -INFINITY, lrow = 0.f;  // of head `col`; lrow: this lane's keys
    char* v_lds = smem + wave * WB;
    const char* kc = (const char*)kcv;
    const char* vc = (const char*)vcv;

    // PF (bf16 caches): the next tile's K fragments are requested while this tile computes. Every K load is then
    // issued unconditionally (keys past the end repeat the last key's row, the mask alone makes their weights 0), and V comes
    // through registers (plain loads, stored to the LDS image after QK^T) instead of LDS-DMA: the explicit vmcnt
    // waits below count exactly NK K loads and NVC V loads per tile, which holds only for loads that complete in
    // issue order (LDS-DMA completions are not ordered against plain loads).
    constexpr bool PF = DPF && !KV8 && !TS && NW <= 8;  // (16-wave form: 128 VGPRs, no room for a second K tile)
    constexpr int NK = 2 * (D / 32);
    // lane l holds the pool row of the tile's key l % 32 (past the end: the last key's, P = 0 there); the lanes that load a key's
    // numbers fetch its row from that lane: one division by the page size a tile
    auto rows_of = [&](int kt) {
        const unsigned key = min(kt + (lane & 31), p1 - 1), bi = key / (unsigned)bs;
        return ((unsigned)sbt[bi - blk0] * Hkv + kvh) * bs + (key - bi * bs);
    };
    auto row_at = [&](unsigned rows, int key) { return (size_t)(unsigned)__builtin_amdgcn_ds_bpermute(4 * key, (int)rows); };
    auto load_k = [&](unsigned rows, bf16x8(&kf_)[2][D / 32]) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const char* r = kc + (row_at(rows, 16 * t + col) * D + 8 * g) * ES;
#pragma unroll
            for (int ks = 0; ks < D / 32; ++ks) kf_[t][ks] = *(const bf16x8*)(r + 32 * ks * ES);
        }
    };
    // 8-bit and block-quantised caches: a tile's bytes wait in registers (keys past the end: the last one again, P = 0)
    [[maybe_unused]] DecRaw<KVF, D> raw;
    auto load_raw = [&](unsigned rows) {
#pragma unroll
        for (int t = 0; t < 2; ++t) raw.load_k(t, kc, row_at(rows, 16 * t + col), g);
        raw.load_v(vc, row_at(rows, lane >> 1), lane & 1);
    };
    unsigned rows = 0;  // of the tile whose loads come next
    if (p_start + wave * KT < p1) rows = rows_of(p_start + wave * KT);
    if constexpr (KV8) {
        if (p_start + wave * KT < p1) load_raw(rows);
    }
    [[maybe_unused]] bf16x8 knext[2][D / 32];
    if constexpr (PF) {
        if (p_start + wave * KT < p1) load_k(rows, knext);
    }
    for (int kt0 = p_start + wave * KT; kt0 < p1; kt0 += NW * KT) {
        // ---- the tile's K fragments (PF: requested during the previous tile) and V chunk loads ----
        bf16x8 kf[2][D / 32];
        if constexpr (PF) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int ks = 0; ks < D / 32; ++ks) kf[t][ks] = knext[t][ks];
        } else if constexpr (KV8) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int ks = 0; ks < D / 32; ++ks) kf[t][ks] = raw.k(t, ks, g);
        } else {
            load_k(rows, kf);
        }
        // V: bf16 caches go HBM -> LDS by DMA (global_load_lds, no VGPR staging): instruction j fills
        // bytes [1024 j, 1024 j + 1024) of the slice linearly by lane, so each lane fetches the chunk
        // that the swizzled V image (v_lds_off) places at its slot; 8-bit caches widen in registers.
        [[maybe_unused]] uint4 vv[PF ? NVC : 1];
        if constexpr (KV8) {
#pragma unroll
            for (int j = 0; j < NVC; ++j) {
                const int p = lane >> 1, c = (lane & 1) * (D / 16) + j;
                *(uint4*)(v_lds + v_lds_off<D>(p, c >> 1) + 16 * (c & 1)) = raw.v(j);
            }
            if (kt0 + NW * KT < p1) load_raw(rows_of(kt0 + NW * KT));
        }
#pragma unroll
        for (int j = 0; j < (KV8 ? 0 : NVC); ++j) {
            int p, c;
            if constexpr (PF) {
                const int id = lane + 64 * j;
                p = id / (D / 8);
                c = id % (D / 8);
            } else {
                // slot 1024 j + 16 lane of the V image
                constexpr int CPR = D / 8;  // chunks a row
                const int sv = D == 128 ? (lane / CPR) & 3 : (lane / CPR) >> 1 & 1;
                p = 512 / D * j + lane / CPR;
                c = (2 * ((lane % CPR >> 1) ^ sv) + (lane & 1)) ^ (D == 128 ? (j >> 1 & 1) * 8 : (j & 1) * 4);
            }
            const size_t eo = row_at(rows, p) * D + c * 8;
            if constexpr (PF) {
                vv[j] = *(const uint4*)(vc + eo * ES);  // rows past the end: a valid row, P = 0 there
            } else {
                __builtin_amdgcn_global_load_lds((const void*)(vc + eo * ES), (MX_LDS void*)(v_lds + 1024 * j), 16, 0, 0);
            }
        }
        [[maybe_unused]] const bool more = kt0 + NW * KT < p1;  // wave-uniform
        if constexpr (PF) {
            __builtin_amdgcn_sched_barrier(0);
            if (more) load_k(rows = rows_of(kt0 + NW * KT), knext);
            __builtin_amdgcn_sched_barrier(0);
            // this tile's K (issued before its V DMAs and the next tile's K) has landed
            if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NVC + NK) : "memory");
            else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NVC) : "memory");
        } else if constexpr (!KV8) {
            if (more) rows = rows_of(kt0 + NW * KT);
        }
        // ---- S^T = K Q^T: 2 x 16 keys x 16 head columns; a lane holds keys 16 t + 4 g + i of head `col` ----
        f32x4 sacc[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            sacc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < D / 32; ++ks)
                sacc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t][ks], qf[ks], sacc[t], 0, 0, 0);
        }
        if constexpr (TS) {
            if (kt0 == p_start) DEC_TS(3)  // the K tile has landed (first tile of wave 0)
        }
        if constexpr (PF) {  // V -> this wave's LDS slice (the previous tile's reads have returned)
#pragma unroll
            for (int j = 0; j < NVC; ++j) {
                const int id = lane + 64 * j, p = id / (D / 8), c = id % (D / 8);
                *(uint4*)(v_lds + v_lds_off<D>(p, c >> 1) + 16 * (c & 1)) = vv[j];
            }
        }
        // ---- online softmax over the tile: the head's maximum over its four lanes, everything else lane-local ----
        float mx = -INFINITY;
        // the mask and the cap: in one pass over the scores, or in branches of their own that most tiles skip (see above)
        if constexpr (!KV8 && D == 128 && NW == 4) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float v = sacc[t][i] * qs;
                    if (softcap > 0.f) v = sc_l2 * tanhf(v * sc_inv);
                    if (kt0 + 16 * t + 4 * g + i >= p1) v = -INFINITY;
                    sacc[t][i] = v;
                    mx = fmaxf(mx, v);
                }
        } else {
            if (softcap > 0.f) {
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) sacc[t][i] = sc_l2 * tanhf(sacc[t][i] * qs * sc_inv);
            } else {
#pragma unroll
                for (int t = 0; t < 2; ++t) sacc[t] *= qs;
            }
            if (kt0 + KT > p1) {
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (kt0 + 16 * t + 4 * g + i >= p1) sacc[t][i] = -INFINITY;
            }
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sacc[t][i]);
        }
        const float mn = fmaxf(mrow, quarters_max(mx));
        if (__any(mn > mrow)) {
            const float alpha = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(mrow - mn);
            lrow *= alpha;
#pragma unroll
            for (int nt = 0; nt < D / 16; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i) oacc[nt][i] *= alpha;
            mrow = mn;
        }
        u32x4 pw;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            float pv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                pv[i] = mn == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(sacc[t][i] - mn);
                lrow += pv[i];
            }
            pw[2 * t] = pack_bf16x2(pv[0], pv[1]);
            pw[2 * t + 1] = pack_bf16x2(pv[2], pv[3]);
        }
        // P^T as B operand: k slot (g, e) is key 16 (e / 4) + 4 g + e % 4, and V^T's rows are read in that order
        const bf16x8 pb = __builtin_bit_cast(bf16x8, pw);
        // the V DMA has landed and the V writes are visible (PF, 8-bit caches: the next tile's loads may stay in flight)
        if constexpr (PF) {
            if (more) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NK) : "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        } else if constexpr (KV8) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        } else {
            __builtin_amdgcn_s_waitcnt(0);
        }
        __builtin_amdgcn_wave_barrier();
        // ---- O^T += V^T P^T ----
        const int r0 = 4 * g, q4 = col >> 2, p4 = col & 3;
#pragma unroll
        for (int nt = 0; nt < D / 16; ++nt) {
            const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (MX_LDS s16x4*)(v_lds + v_lds_off<D>(r0 + q4, nt) + 8 * p4));
            const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (MX_LDS s16x4*)(v_lds + v_lds_off<D>(r0 + 16 + q4, nt) + 8 * p4));
            const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
            const u32x4 w4 = {l2[0], l2[1], h2[0], h2[1]};
            oacc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w4), pb, oacc[nt], 0, 0, 0);
        }
        __builtin_amdgcn_s_waitcnt(0xc07f);  // the transposed reads have returned before V is rewritten
        __builtin_amdgcn_wave_barrier();
    }
    // ---- merge the NW waves: (m, l) per row and O rows through the (now free) LDS slices ----
    DEC_TS(4)
    __syncthreads();
    DEC_TS(5)
    float* wo = (float*)(smem + wave * WB);        // [16 rows][D] fp32 (8 KB for D=128 <= WB)
    float* wml = (float*)(smem + NW * WB) + wave * 32;  // [16 rows] m, [16 rows] l
    // waves past the context's last tile hold nothing (m = -inf, l = 0): neither written nor read
    const int nwa = p1 > p_start ? min(NW, (p1 - p_start + KT - 1) / KT) : 0;
    lrow = quarters_sum(lrow);
    if (wave < nwa && col < G) {  // only the G real heads of the 16 columns
#pragma unroll
        for (int nt = 0; nt < D / 16; ++nt)
            *(float4*)(wo + col * D + 16 * nt + 4 * g) = make_float4(oacc[nt][0], oacc[nt][1], oacc[nt][2], oacc[nt][3]);
        if (g == 0) { wml[col] = mrow; wml[16 + col] = lrow; }
    }
    __syncthreads();
    DEC_TS(6)
    const float* ml = (const float*)(smem + NW * WB);
    // a sequence that fits this one partition: the final output here, no partials (the reduce skips it)
    const bool single = n_parts == 1 || (p0 == 0 && L <= part_size);
    // per head row: the waves' merge weights exp2(m_w - mx) and the row's (mx, l) — once per row in 16-lane
    // groups, not once per output element (the output loop below is then one FMA per wave)
    __shared__ float s_wt[16 * 16];
    __shared__ float2 s_rml[16];
    if (threadIdx.x < G * 16) {  // whole 16-lane groups (G * 16 is a multiple of 16)
        const int h = threadIdx.x >> 4, w = threadIdx.x & 15;
        const float m = w < nwa ? ml[w * 32 + h] : -INFINITY;
        const float mx = group_max<16>(m);
        const float a = (w < nwa && mx != -INFINITY) ? exp2f(m - mx) : 0.f;
        const float ls = group_sum<16>(w < nwa ? ml[w * 32 + 16 + h] * a : 0.f);
        s_wt[threadIdx.x] = a;
        if (w == 0) s_rml[h] = make_float2(mx, ls);
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < G * D; idx += 64 * NW) {
        const int h = idx / D, d = idx % D;
        const float mx = s_rml[h].x, ls = s_rml[h].y;
        float os = 0.f;
#pragma unroll 4
        for (int w = 0; w < nwa; ++w) os += ((const float*)(smem + w * WB))[h * D + d] * s_wt[h * 16 + w];
        const int hq = kvh * G + h;
        if (single) {
            out[(size_t)b * out_stride + (size_t)hq * D + d] = f32_to_act<F16>(ls > 0.f ? os / ls : 0.f);
        } else {
            const size_t pi = ((size_t)b * Hq + hq) * n_parts + part;
            // sc1 stores (agent-scope relaxed atomics): the fused merge below reads them from another CU / XCD with
            // sc1 loads, so no L2 write-back fence is needed (MI355X_MICROARCH.md inter-workgroup hand-off, row 1)
            if (d == 0)
                __hip_atomic_store((unsigned long long*)(part_ml + pi),
                                   __builtin_bit_cast(unsigned long long, make_float2(mx, ls)), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(part_o + pi * D + d, os, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    DEC_TS(7)
#undef DEC_TS
    if (single || !part_cnt) return;
    // fused split-K merge: the last of the (b, kvh) partition workgroups to finish merges all of them,
    // instead of a separate reduce launch (at batch 1 that launch costs as much as the attention itself).
    // The counter is left at zero for the next launch / graph replay.
    // hand-off without fences: every storing wave waits for its sc1 stores, a barrier, then ONE agent-scope atomic add
    // per workgroup; the workgroup whose add came last reads the partials with sc1 loads (no buffer_wbl2 / buffer_inv:
    // an agent fence costs ~3.5 us per workgroup here and made this merge lose to a separate launch in round 5)
    __shared__ int s_last;
    const int np = min(n_parts, (L + part_size - 1) / part_size);  // partitions that did not return early
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        const int old = __hip_atomic_fetch_add(&part_cnt[b * Hkv + kvh], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = old == np - 1;
        if (old == np - 1) __hip_atomic_store(&part_cnt[b * Hkv + kvh], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!s_last) return;
    auto ml_at = [&](size_t i) {
        return __builtin_bit_cast(float2, __hip_atomic_load((unsigned long long*)(part_ml + i), __ATOMIC_RELAXED,
                                                            __HIP_MEMORY_SCOPE_AGENT));
    };
    for (int idx = threadIdx.x; idx < G * D; idx += 64 * NW) {
        const int h = idx / D, d = idx % D, hq = kvh * G + h;
        const size_t pb = ((size_t)b * Hq + hq) * n_parts;
        float mx = -INFINITY;
        for (int p = 0; p < np; ++p) mx = fmaxf(mx, ml_at(pb + p).x);
        float ls = 0.f, os = 0.f;
        for (int p = 0; p < np; ++p) {
            const float2 pm = ml_at(pb + p);
            const float a = mx == -INFINITY ? 0.f : exp2f(pm.x - mx);
            ls += pm.y * a;
            os += __hip_atomic_load(part_o + (pb + p) * D + d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) * a;
        }
        out[(size_t)b * out_stride + (size_t)hq * D + d] = f32_to_act<F16>(ls > 0.f ? os / ls : 0.f);
    }
}

static bool decode_pf() {
    // off by default: at c128 the 2-wave prefetch form measured 1.5 % slower end to end than the 4-wave form
    // (profiles/r5_step_composition.md); MX_DECODE_PF=1 selects it
    static const bool on = getenv("MX_DECODE_PF") && atoi(getenv("MX_DECODE_PF")) != 0;
    return on;
}

template <int D>
static int launch_decode_mfma(const bf16_t* q, int q_stride, const void* kc, const void* vc, const int* bt,
                              int bt_stride, const int* seq_lens, int B, int Hkv, int G, int bs, float scale,
                              int window, float softcap, int part_size, int n_parts, bf16_t* out, int out_stride,
                              float2* part_ml, float* part_o, int* part_cnt, int kv8, hipStream_t st) {
    dim3 grid(Hkv, B, n_parts);
    static_assert(16 * D * 4 <= dec_wave_lds<D>(), "merge buffer");
    // 512-key partitions run 16 waves per workgroup (one 32-key tile each), 256-key ones 8, smaller ones 4
    const bool wide = part_size >= 512 && !kv8 && B < 8;  // (large batches keep 4-wave workgroups)
    const bool mid = !wide && part_size >= 256 && !kv8 && B < 8;
    const int NWs = wide ? 16 : mid ? 8 : 4;
    const size_t lds = NWs * dec_wave_lds<D>() + NWs * 32 * 4;
#define DQK(F_)                                                                                                   \
    attn_decode_mfma_kernel<D, F16, F_><<<grid, 256, lds, st>>>(q, q_stride, kc, vc, bt, bt_stride, seq_lens, Hkv, G, \
                                                               bs, scale, window, softcap, part_size, n_parts, out,   \
                                                               out_stride, part_ml, part_o, part_cnt)
    MX_ACT_DISPATCH({
        if (kv8 == KVF_FP8) DQK(KVF_FP8);
        else if (kv8 == KVF_Q8_0) DQK(KVF_Q8_0);
        else if (kv8 == KVF_Q4_0) DQK(KVF_Q4_0);
        else if (kv8 == KVF_Q4_1) DQK(KVF_Q4_1);
        else if (kv8 == KVF_Q5_0) DQK(KVF_Q5_0);
        else if (kv8 == KVF_Q5_1) DQK(KVF_Q5_1);
        else if (kv8 == KVF_IQ4_NL) DQK(KVF_IQ4_NL);
        else if (wide) {
            static bool attr = false;
            if (!attr) {
                (void)hipFuncSetAttribute((const void*)attn_decode_mfma_kernel<D, F16, KVF_BF16, 16>,
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
                attr = true;
            }
            attn_decode_mfma_kernel<D, F16, KVF_BF16, 16><<<grid, 1024, lds, st>>>(
                q, q_stride, kc, vc, bt, bt_stride, seq_lens, Hkv, G, bs, scale, window, softcap, part_size, n_parts,
                out, out_stride, part_ml, part_o, part_cnt);
        } else if (mid) {
            static bool attr8 = false;
            if (!attr8) {
                (void)hipFuncSetAttribute((const void*)attn_decode_mfma_kernel<D, F16, KVF_BF16, 8>,
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
                attr8 = true;
            }
            attn_decode_mfma_kernel<D, F16, KVF_BF16, 8><<<grid, 512, lds, st>>>(
                q, q_stride, kc, vc, bt, bt_stride, seq_lens, Hkv, G, bs, scale, window, softcap, part_size, n_parts,
                out, out_stride, part_ml, part_o, part_cnt);
        } else if (decode_pf())
            attn_decode_mfma_kernel<D, F16, KVF_BF16, 4, false, true><<<grid, 256, lds, st>>>(
                q, q_stride, kc, vc, bt, bt_stride, seq_lens, Hkv, G, bs, scale, window, softcap, part_size, n_parts,
                out, out_stride, part_ml, part_o, part_cnt);
        else
            attn_decode_mfma_kernel<D, F16, KVF_BF16><<<grid, 256, lds, st>>>(q, q_stride, kc, vc, bt, bt_stride,
                                                                          seq_lens, Hkv, G, bs, scale, window, softcap,
                                                                          part_size, n_parts, out, out_stride, part_ml,
                                                                          part_o, part_cnt);
        if (n_parts > 1 && !part_cnt)
            attn_decode_reduce_kernel<F16><<<B * Hkv * G, 256, 0, st>>>(part_ml, part_o, n_parts, Hkv * G, D, seq_lens,
                                                                        part_size, out, out_stride);
    });
    MXK_CHECK_LAUNCH();
}

// debug: the 16-wave single-pass decode (bf16 activations and cache, D = 128) with phase stamps of workgroup 0's
// wave 0 in ts[0..7] (s_memrealtime, 100 MHz): entry, past the seq-len check, block table in LDS, first K tile
// landed, tiles done, merge barrier 1, merge barrier 2, output stored
extern "C" int mxk_attn_decode_ts(const bf16_t* q, int q_stride, const void* kc, const void* vc, const int* bt,
                                  int bt_stride, const int* seq_lens, int B, int Hq, int Hkv, int bs, float scale,
                                  int part_size, bf16_t* out, int out_stride, unsigned long long* ts, hipStream_t st) {
    if (Hq % Hkv || Hq / Hkv > 16 || part_size < 512 || bs <= 0 || part_size / bs + 1 > 256)
        return (int)hipErrorInvalidValue;
    const size_t lds = 16 * dec_wave_lds<128>() + 16 * 32 * 4;
    (void)hipFuncSetAttribute((const void*)attn_decode_mfma_kernel<128, false, KVF_BF16, 16, true>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    attn_decode_mfma_kernel<128, false, KVF_BF16, 16, true><<<dim3(Hkv, B, 1), 1024, lds, st>>>(
        q, q_stride, kc, vc, bt, bt_stride, seq_lens, Hkv, Hq / Hkv, bs, scale, 0, 0.f, part_size, 1, out, out_stride,
        nullptr, nullptr, nullptr, ts);
    MXK_CHECK_LAUNCH();
}

// MFMA decode for D in {64, 128} and up to 16 query heads per kv head; other shapes return
// hipErrorInvalidValue (the caller falls back to mxk_attn_decode). part_cnt: B x Hkv zero-initialised
// counters for the in-kernel partition merge (nullptr: a separate reduce launch).
extern "C" int mxk_attn_decode_mfma(const bf16_t* q, int q_stride, const void* kc, const void* vc, const int* bt,
                                    int bt_stride, const int* seq_lens, int B, int Hq, int Hkv, int D, int bs,
                                    float scale, int window, float softcap, int part_size, int n_parts, bf16_t* out,
                                    int out_stride, float2* part_ml, float* part_o, int kv8, int* part_cnt,
                                    hipStream_t st) {
    if (B <= 0) return 0;
    if (Hq % Hkv || Hq / Hkv > 16) return (int)hipErrorInvalidValue;
    if (n_parts > 1 && (!part_ml || !part_o)) return (int)hipErrorInvalidValue;
    if (bs <= 0 || part_size / bs + 1 > 256) return (int)hipErrorInvalidValue;
    const int G = Hq / Hkv;
    if (D == 128) return launch_decode_mfma<128>(q, q_stride, kc, vc, bt, bt_stride, seq_lens, B, Hkv, G, bs, scale, window, softcap, part_size, n_parts, out, out_stride, part_ml, part_o, part_cnt, kv8, st);
    if (D == 64) return launch_decode_mfma<64>(q, q_stride, kc, vc, bt, bt_stride, seq_lens, B, Hkv, G, bs, scale, window, softcap, part_size, n_parts, out, out_stride, part_ml, part_o, part_cnt, kv8, st);
    return (int)hipErrorInvalidValue;
}

// What attention_flash.hip does not take (ops/core.py flash_plan): head dim 256, with V as rows or (VT = 1, `vmode`) transposed in
// LDS, and short contexts of head dims 64 / 128 where its wider workgroups lose.
template <int D, int GW, int VT, bool F16, int KVF>
__global__ __launch_bounds__(512) void attn_prefill_kernel(const bf16_t* __restrict__ q,
                                                           const void* __restrict__ kc,
                                                           const void* __restrict__ vc,
                                                           const int* __restrict__ block_tables, int bt_stride,
                                                           const int* __restrict__ tile_seq,
                                                           const int* __restrict__ tile_q0,
                                                           const int* __restrict__ cu_q,
                                                           const int* __restrict__ ctx_lens, int Hq, int Hkv,
                                                           int G, int bs, float scale, int window, float softcap,
                                                           bf16_t* __restrict__ out) {
    constexpr int NW = GW >= 3 ? GW : 4;      // waves per workgroup
    constexpr int RT = NW / GW;               // 16-row query tiles per workgroup
    constexpr int KT = 64;                    // keys per tile
    constexpr int KBYTES = KT * D * 2;
    constexpr int PSTRIDE = (KT + 8) * 2;     // bytes per P row (padded)
    constexpr int VTSTRIDE = (KT + 8) * 2;    // VT=1: bytes per transposed V row (one dim)
    constexpr int VBYTES = VT ? D * VTSTRIDE : KBYTES;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    char* k_lds = smem;
    char* v_lds = k_lds + KBYTES;
    char* p_lds = v_lds + VBYTES;
    constexpr int NT_C = NW * 64;              // threads staging a tile
    const int tid = threadIdx.x;
    const int g = lane >> 4, col = lane & 15;
    const int tile = blockIdx.x;
    const int s = tile_seq[tile], q0 = tile_q0[tile];
    if (s < 0) return;  // padding tile of a graph-captured step (uniform across the workgroup)
    const int hq = blockIdx.y * GW + (wave % GW);
    const int kvh = (blockIdx.y * GW) / G;
    const int rt = wave / GW;
    const int qbeg = cu_q[s], qlen = cu_q[s + 1] - qbeg;
    const int ctx = ctx_lens[s];
    const int pos_off = ctx - qlen;  // position of query 0
    const int* bt = block_tables + (size_t)s * bt_stride;
    const int row_q0 = q0 + rt * 16;        // first query index of this wave
    const int wg_rows = RT * 16;
    const int kv_end = min(ctx, pos_off + min(qlen, q0 + wg_rows));
    const float qs = scale * LOG2E;
    const float sc_l2 = softcap * LOG2E, sc_inv = softcap > 0.f ? 1.f / (softcap * LOG2E) : 0.f;
    // sliding window: key tiles entirely before the earliest query's window are skipped
    const int kt_begin = window > 0 ? (max(0, pos_off + q0 - window + 1) / 64) * 64 : 0;

    // Q fragments: lane row = col, dims 32ks + 8g
    bf16x8 qf[D / 32];
    {
        const int qi = row_q0 + col;
#pragma unroll
        for (int ks = 0; ks < D / 32; ++ks) {
            if (qi < qlen) qf[ks] = *(const bf16x8*)(q + ((size_t)(qbeg + qi) * Hq + hq) * D + 32 * ks + 8 * g);
            else qf[ks] = (bf16x8){};
        }
    }
    f32x4 oacc[D / 16];
#pragma unroll
    for (int i = 0; i < D / 16; ++i) oacc[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float mrow[4], lrow[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) { mrow[i] = -INFINITY; lrow[i] = 0.f; }
    char* pw = p_lds + wave * 16 * PSTRIDE;

    // K / V tiles are software-pipelined one tile deep: tile t + 1's global loads (block-table entry, then the
    // 16-byte chunks) are issued right after tile t is staged in LDS, so their latency hides behind tile t's
    // MFMAs and softmax instead of opening every tile (short prompt chunks run only a few tiles per workgroup)
    constexpr int CH = KT * D / 8;              // 16-byte chunks per tile
    constexpr int NCH = (CH + NT_C - 1) / NT_C;  // chunks per thread
    constexpr bool KV8 = KVF == KVF_FP8;
    constexpr bool KVQ_ = KVF >= KVF_Q8_0;  // block-quantised rows (kvq.h): raw codes + scales kept in flight
    using KRaw = typename std::conditional<KVQ_, KVQRaw, typename std::conditional<KV8, uint2, uint4>::type>::type;
    KRaw kr[NCH], vr[NCH];
    auto load_tile = [&](int kt0) {
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
            const int id = tid + j * NT_C;
            const int p = id / (D / 8), c = id % (D / 8);
            const int pos = kt0 + p;
            kr[j] = KRaw{};
            vr[j] = KRaw{};
            if (id < CH && pos < kv_end) {
                const int blk = bt[pos / bs], off = pos % bs;
                const size_t eo = (((size_t)blk * Hkv + kvh) * bs + off) * D + c * 8;
                if constexpr (KVQ_) {
                    kr[j] = kvq_load<KVF, D>(kc, eo);
                    vr[j] = kvq_load<KVF, D>(vc, eo);
                } else if constexpr (KV8) {
                    kr[j] = *(const uint2*)((const uint8_t*)kc + eo);
                    vr[j] = *(const uint2*)((const uint8_t*)vc + eo);
                } else {
                    kr[j] = *(const uint4*)((const bf16_t*)kc + eo);
                    vr[j] = *(const uint4*)((const bf16_t*)vc + eo);
                }
            }
        }
    };
    auto store_tile = [&]() {
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
            const int id = tid + j * NT_C;
            if (id >= CH) continue;
            const int p = id / (D / 8), c = id % (D / 8);
            uint4 kv, vv;
            if constexpr (KVQ_) {
                kv = kvq_to_bf16x8<KVF>(kr[j]);
                vv = kvq_to_bf16x8<KVF>(vr[j]);
            } else if constexpr (KV8) {
                kv = fp8x8_to_bf16x8(kr[j]);
                vv = fp8x8_to_bf16x8(vr[j]);
            } else {
                kv = kr[j];
                vv = vr[j];
            }
            *(uint4*)(k_lds + k_lds_off<D>(p, c)) = kv;
            if constexpr (VT == 0) {
                *(uint4*)(v_lds + v_lds_off<D>(p, c >> 1) + 16 * (c & 1)) = vv;
            } else {
                const uint32_t w[4] = {vv.x, vv.y, vv.z, vv.w};
#pragma unroll
                for (int jj = 0; jj < 8; ++jj)
                    *(bf16_t*)(v_lds + (8 * c + jj) * VTSTRIDE + 2 * p) = (bf16_t)(w[jj >> 1] >> (16 * (jj & 1)));
            }
        }
    };
    if (kt_begin < kv_end) load_tile(kt_begin);
    for (int kt0 = kt_begin; kt0 < kv_end; kt0 += KT) {
        // ---- stage this K and V tile (64 keys x D), then request the next one ----
        store_tile();
        if (kt0 + KT < kv_end) load_tile(kt0 + KT);
        __syncthreads();
        // ---- S = Q K^T : 16 rows x 64 keys ----
        f32x4 sacc[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            sacc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < D / 32; ++ks) {
                const bf16x8 kf = *(const bf16x8*)(k_lds + k_lds_off<D>(16 * t + col, 4 * ks + g));
                sacc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qf[ks], kf, sacc[t], 0, 0, 0);
            }
        }
        // ---- mask + online softmax (rows 4g+i, keys 16t+col) ----
        float rmax[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int qi = row_q0 + 4 * g + i;
            const int qpos = pos_off + qi;
            float mx = -INFINITY;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int kp = kt0 + 16 * t + col;
                float v = sacc[t][i] * qs;
                if (softcap > 0.f) v = sc_l2 * tanhf(v * sc_inv);
                if (kp > qpos || kp >= ctx || qi >= qlen || (window > 0 && kp <= qpos - window)) v = -INFINITY;
                sacc[t][i] = v;
                mx = fmaxf(mx, v);
            }
            rmax[i] = group_max<16>(mx);
        }
        float alpha[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float mn = fmaxf(mrow[i], rmax[i]);
            alpha[i] = mn == -INFINITY ? 1.f : exp2f(mrow[i] - mn);
            float rs = 0.f;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float pv = mn == -INFINITY ? 0.f : exp2f(sacc[t][i] - mn);
                sacc[t][i] = pv;
                rs += pv;
            }
            rs = group_sum<16>(rs);
            lrow[i] = lrow[i] * alpha[i] + rs;
            mrow[i] = mn;
        }
#pragma unroll
        for (int nt = 0; nt < D / 16; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) oacc[nt][i] *= alpha[i];
        // ---- P -> LDS (bf16) ----
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *(bf16_t*)(pw + (4 * g + i) * PSTRIDE + (16 * t + col) * 2) = f32_to_bf16(sacc[t][i]);
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): P visible to the wave (same wave reads)
        __builtin_amdgcn_wave_barrier();
        // ---- O += P V ----
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const bf16x8 pa = *(const bf16x8*)(pw + col * PSTRIDE + (32 * ks + 8 * g) * 2);
            const int r0 = 32 * ks + 8 * g;
            const int q4 = col >> 2, p4 = col & 3;
#pragma unroll
            for (int nt = 0; nt < D / 16; ++nt) {
                bf16x8 vb;
                if constexpr (VT == 0) {
                    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (MX_LDS s16x4*)(v_lds + v_lds_off<D>(r0 + q4, nt) + 8 * p4));
                    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (MX_LDS s16x4*)(v_lds + v_lds_off<D>(r0 + 4 + q4, nt) + 8 * p4));
                    // whole-vector reinterpretation: per-element bf16 bit_casts of the v4i16 result were
                    // miscompiled (hipcc dropped elements 2,3 of each transposed read)
                    const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
                    const u32x4 w4 = {l2[0], l2[1], h2[0], h2[1]};
                    vb = __builtin_bit_cast(bf16x8, w4);
                } else {
                    vb = *(const bf16x8*)(v_lds + (16 * nt + col) * VTSTRIDE + r0 * 2);
                }
                oacc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa, vb, oacc[nt], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    // ---- write O / l ----
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int qi = row_q0 + 4 * g + i;
        if (qi >= qlen) continue;
        const float inv = lrow[i] > 0.f ? 1.f / lrow[i] : 0.f;
#pragma unroll
        for (int nt = 0; nt < D / 16; ++nt)
            out[((size_t)(qbeg + qi) * Hq + hq) * D + 16 * nt + col] = f32_to_act<F16>(oacc[nt][i] * inv);
    }
}

template <int D, int GW, int VT, int KVF>
static void launch_prefill_t(dim3 grid, int threads, size_t lds, const bf16_t* q, const void* kc, const void* vc,
                             const int* bt, int bt_stride, const int* tile_seq, const int* tile_q0, const int* cu_q,
                             const int* ctx_lens, int Hq, int Hkv, int bs, float scale, int window, float softcap,
                             bf16_t* out, hipStream_t st) {
    MX_ACT_DISPATCH({
        if (lds > 65536) {  // D=256 tiles (73-82 KB): opt in to the large LDS allocation once
            static bool opted = false;
            if (!opted) {
                (void)hipFuncSetAttribute((const void*)attn_prefill_kernel<D, GW, VT, F16, KVF>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
                opted = true;
            }
        }
        attn_prefill_kernel<D, GW, VT, F16, KVF><<<grid, threads, lds, st>>>(
            q, kc, vc, bt, bt_stride, tile_seq, tile_q0, cu_q, ctx_lens, Hq, Hkv, Hq / Hkv, bs, scale, window,
            softcap, out);
    });
}

template <int D, int GW>
static int launch_prefill(const bf16_t* q, const void* kc, const void* vc, const int* bt, int bt_stride,
                          const int* tile_seq, const int* tile_q0, int n_tiles, const int* cu_q,
                          const int* ctx_lens, int Hq, int Hkv, int bs, float scale, int window, float softcap,
                          bf16_t* out, int vmode, int kv8, hipStream_t st) {
    constexpr int NW = GW >= 3 ? GW : 4;
    dim3 grid(n_tiles, Hq / GW);
    const size_t lds0 = 2 * 64 * D * 2 + NW * 16 * (64 + 8) * 2;
    const size_t lds1 = 64 * D * 2 + D * (64 + 8) * 2 + NW * 16 * (64 + 8) * 2;
#define PFL(VT_, K8_)                                                                                          \
    launch_prefill_t<D, GW, VT_, K8_>(grid, NW * 64, VT_ ? lds1 : lds0, q, kc, vc, bt, bt_stride, tile_seq,    \
                                      tile_q0, cu_q, ctx_lens, Hq, Hkv, bs, scale, window, softcap, out, st)
#define PFK(VT_)                                                                                                \
    {                                                                                                           \
        if (kv8 == KVF_FP8) PFL(VT_, KVF_FP8);                                                                  \
        else if (kv8 == KVF_Q8_0) PFL(VT_, KVF_Q8_0);                                                           \
        else if (kv8 == KVF_Q4_0) PFL(VT_, KVF_Q4_0);                                                           \
        else if (kv8 == KVF_Q4_1) PFL(VT_, KVF_Q4_1);                                                           \
        else if (kv8 == KVF_Q5_0) PFL(VT_, KVF_Q5_0);                                                           \
        else if (kv8 == KVF_Q5_1) PFL(VT_, KVF_Q5_1);                                                           \
        else if (kv8 == KVF_IQ4_NL) PFL(VT_, KVF_IQ4_NL);                                                       \
        else PFL(VT_, KVF_BF16);                                                                                \
    }
    if constexpr (D == 256) {
        if (vmode == 0) PFK(0) else PFK(1)
    } else PFK(0)
#undef PFK
#undef PFL
    MXK_CHECK_LAUNCH();
}

// rows per workgroup for the host-side tile map: 16 * (NW / GW)
extern "C" int mxk_attn_prefill_rows(int Hq, int Hkv) {
    const int G = Hq / Hkv;
    const int GW = G <= 8 ? G : 8;
    const int NW = GW >= 3 ? GW : 4;
    return 16 * (NW / GW);
}

extern "C" int mxk_attn_prefill(const bf16_t* q, const void* kc, const void* vc, const int* bt, int bt_stride,
                                const int* tile_seq, const int* tile_q0, int n_tiles, const int* cu_q,
                                const int* ctx_lens, int Hq, int Hkv, int D, int bs, float scale, int window,
                                float softcap, bf16_t* out, int vmode, int kv8, hipStream_t st) {
    if (n_tiles <= 0) return 0;
    if (Hq % Hkv) return (int)hipErrorInvalidValue;
    const int G = Hq / Hkv;
    const int GW = G <= 8 ? G : 8;
    if (G > 8 && G % 8) return (int)hipErrorInvalidValue;
#define PF(D_, GW_) \
    if (D == D_ && GW == GW_) return launch_prefill<D_, GW_>(q, kc, vc, bt, bt_stride, tile_seq, tile_q0, n_tiles, cu_q, ctx_lens, Hq, Hkv, bs, scale, window, softcap, out, vmode, kv8, st);
    PF(128, 1) PF(128, 2) PF(128, 3) PF(128, 4) PF(128, 5) PF(128, 6) PF(128, 7) PF(128, 8)
    PF(64, 1) PF(64, 2) PF(64, 4) PF(64, 8)
    PF(256, 1) PF(256, 2) PF(256, 4)
#undef PF
    return (int)hipErrorInvalidValue;
}

// debug probe: semantics of ds_read_b64_tr_b16 on this device. LDS holds value r*16+c at row r
// (16 rows), column c (16 cols), 32-byte rows; lane l supplies row (l&15)>>2 (+4*(l>>4)),
// columns 4*(l&3). out[l*4 + e] = element e returned to lane l.
__global__ void probe_tr16_kernel(short* out) {
    __shared__ __attribute__((aligned(16))) short lds[16 * 16];
    for (int i = threadIdx.x; i < 256; i += 64) lds[i] = (short)i;
    __syncthreads();
    const int l = threadIdx.x;
    const int row = ((l & 15) >> 2) + 4 * (l >> 4);
    const int colg = 4 * (l & 3);
    s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((MX_LDS s16x4*)(lds + row * 16 + colg));
    for (int e = 0; e < 4; ++e) out[l * 4 + e] = v[e];
}
extern "C" int mxk_probe_tr16(short* out, hipStream_t st) {
    probe_tr16_kernel<<<1, 64, 0, st>>>(out);
    MXK_CHECK_LAUNCH();
}
