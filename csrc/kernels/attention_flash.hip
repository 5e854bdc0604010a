// attention_flash.hip: prompt attention over the paged cache on 32x32x16 MFMA (bf16, fp8 and block-quantised caches),
// head dims 64 and 128, except for contexts of one key tile where attention.hip is the faster (ops/core.py flash_plan).
//
// A workgroup owns one KV head, RQ consecutive queries of one sequence and a range of key tiles. Its G query heads are
// packed with the queries into 32-column groups, column = query * G + head: whatever G is, a wave holds 32 of them and
// every K / V tile in LDS serves them all. The scores are computed transposed (attn_tile.h), so that a column is one lane's (two
// half-waves hold the even and odd 4-key groups): maximum, sum and rescaling are lane-local but for one exchange between the
// half-waves per tile, and the probabilities are already where the next product's B operand wants them. Nothing goes through LDS
// but K and V.
//
// Tiles of 64 keys are double-buffered: a tile's 16-byte chunks are requested one tile ahead, wait in registers (where
// fp8 and block formats are widened to bf16) and are stored to the other buffer, one barrier per tile. The next tile is stored, and
// the one after it requested, a piece beside each pair of the scores' products, while the matrix unit is busy: as a stretch of its
// own before or after the tile it took a seventh of the time (8191 rows 576 -> 548 us, 2000 57 -> 55).
// A wave requests 4 (head dim 128) or 8 rows with one instruction, which lie in one page where its size is a multiple of that: each
// lane looks up one such group's row, for 16 tiles or more at once, and the address is a readlane away. (A division, a load of the
// block table and 64-bit products for each 16 bytes were 100 of an fp8 tile's 400 vector instructions: 416 rows behind 12000 keys
// 128 -> 120 us with 4 waves.)
//
// A short chunk behind a long context has too few workgroups (7 x 8 for 416 rows of a 32 / 8-head model), so the key
// range is split over grid.z: parts of MIN_TILES tiles or more, the last one of what is left (17 tiles: 16 + 1), write (m, l, O)
// unnormalised in fp32 and attn_flash_merge_kernel combines them; a block of queries that only one part has keys for is
// finished by that part.
//
// Measured, 32 / 8 heads of 128, against the 16-row kernel this replaced (which read each K / V fragment for one 16x16x32
// product and moved P through LDS): an 8191-token prompt 2400 -> 560 us (980 TFLOP/s), 2048 233 -> 58, 333 18.5 -> 14.0;
// 416 rows behind 12000 keys 498 -> 110 us in bf16, 788 -> 110 in fp8. Heads of 64, 8191 rows: 1253 -> 360 us. Bound by
// the vector unit beside the matrix unit (32 exponentials and ~170 other vector operations a lane and tile against 32
// products: counters show each busy for 40 % of the time and little of both at once); short prompts by the chain of one tile
// (~1.3 us) times their tiles.
#include <type_traits>

#include "attn_tile.h"
#include "kvq.h"

#define LOG2E 1.4426950408889634f

namespace {

constexpr int FT = AT_KEYS;
constexpr int MIN_TILES = 16;  // fewest key tiles of a part that is not a block's last

// c tanh(v / c) for c = softcap * log2(e), k = 2 / softcap: (1 - e) / (1 + e) with e = exp2(-k |v|). tanhf took half of a capped
// prompt's time (416 rows behind 100 tokens, 32 / 8 heads of 128: 35.4 us).
MX_DEV float f_cap(float v, float c, float k) {
    const float e = __builtin_amdgcn_exp2f(-k * fabsf(v));
    return copysignf(c * (1.f - e) * __builtin_amdgcn_rcpf(1.f + e), v);
}

template <int CTRL, int ROWS>
MX_DEV int scan_step(int v) { return v + __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, false); }
MX_DEV int wave_scan(int v) {  // sum over the lanes up to this one: row_shr 1, 2, 4, 8, then the rows' last lanes
    v = scan_step<0x111, 0xF>(v);
    v = scan_step<0x112, 0xF>(v);
    v = scan_step<0x114, 0xF>(v);
    v = scan_step<0x118, 0xF>(v);
    v = scan_step<0x142, 0xA>(v);  // row_bcast 15 into rows 1 and 3
    return scan_step<0x143, 0xC>(v);  // row_bcast 31 into rows 2 and 3
}

template <int KVF>
struct FRaw {
    using T = typename std::conditional<(KVF >= KVF_Q8_0), KVQRaw, typename std::conditional<KVF == KVF_FP8, uint2, uint4>::type>::type;
};
template <int KVF, int D>
MX_DEV typename FRaw<KVF>::T f_load(const void* base, size_t eo) {
    if constexpr (KVF >= KVF_Q8_0) return kvq_load<KVF, D>(base, eo);
    else if constexpr (KVF == KVF_FP8) return *(const uint2*)((const uint8_t*)base + eo);
    else return *(const uint4*)((const bf16_t*)base + eo);
}
template <int KVF, int D>
constexpr uint32_t f_row_bytes() {  // of the cache
    if constexpr (KVF >= KVF_Q8_0) return KVQ<KVF, D>::ROWB;
    else return D * (KVF == KVF_FP8 ? 1 : 2);
}
template <int KVF, int D>
MX_DEV typename FRaw<KVF>::T f_load_row(const uint8_t* base, uint32_t v, uint32_t e) {  // row v, elements e .. e + 7
    const uint32_t r = v * f_row_bytes<KVF, D>();
    if constexpr (KVF >= KVF_Q8_0) return kvq_load_row<KVF, D>(base, r, e);
    else return *(const typename FRaw<KVF>::T*)(base + (r + e * (KVF == KVF_FP8 ? 1 : 2)));
}
template <int KVF>
MX_DEV uint4 f_widen(const typename FRaw<KVF>::T& w) {
    if constexpr (KVF >= KVF_Q8_0) return kvq_to_bf16x8<KVF>(w);
    else if constexpr (KVF == KVF_FP8) return fp8x8_to_bf16x8(w);
    else return w;
}

// GEN: sliding window, soft cap, or a scale that is not positive; without it the scale is one FMA with the maximum.
// UNI: the rows that a wave requests with one instruction (4 of head dim 128, 8 of 64, beginning at a multiple of that) lie in
// one page: their address is scalar but for the lane's place in them.
template <int D, int NW, int KVF, bool GEN, bool UNI>
__global__ __launch_bounds__(64 * NW, NW == 8 ? 1 : 2) void attn_flash_kernel(const bf16_t* __restrict__ q, const void* __restrict__ kc,
                                                             const void* __restrict__ vc, const int* __restrict__ block_tables,
                                                             int bt_stride, const int* __restrict__ cu_q,
                                                             const int* __restrict__ ctx_lens, int n_seqs, int T, int Hq, int Hkv,
                                                             int G, int bs, int bs_sh, float scale, int window, float softcap,
                                                             bf16_t* __restrict__ out, int f16, float* __restrict__ part_o,
                                                             float2* __restrict__ part_ml) {
    constexpr int NT = 64 * NW;
    constexpr int IMG = FT * D * 2;              // one K or V image
    constexpr int CH = FT * D / 8;               // 8-element chunks per image
    constexpr int NCH = CH / NT;                 // per thread
    static_assert(CH % NT == 0, "whole chunks per thread");
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int h = lane >> 5, col = lane & 31;
    const int RQ = 32 * NW / G;                  // queries per workgroup
    const int kvh = blockIdx.x, part = blockIdx.z, n_parts = gridDim.z;

    // ---- which queries: blocks of RQ of the sequences, counted from the last one (it sees the most keys) ----
    // 64 sequences a round, lane = sequence from the end: one scan over the lanes finds the block's, whose numbers its lane holds.
    int qbeg = 0, qlen = 0, ctx = 0, s = -1, want = blockIdx.y;
    for (int b = n_seqs - 1; b >= 0; b -= 64) {
        const int i = max(b - lane, 0);
        const int c0 = cu_q[i], c1 = cu_q[i + 1], cl = ctx_lens[i];
        const int n = lane <= b ? (c1 - c0 + RQ - 1) / RQ : 0, acc = wave_scan(n);
        const unsigned long long m = __ballot(acc > want);
        if (m) {
            const int l = __builtin_amdgcn_readfirstlane(__ffsll(m) - 1);
            s = b - l;
            want = __builtin_amdgcn_readlane(acc, l) - 1 - want;  // block of the sequence, from its first
            qbeg = __builtin_amdgcn_readlane(c0, l);
            qlen = __builtin_amdgcn_readlane(c1, l) - qbeg;
            ctx = __builtin_amdgcn_readlane(cl, l);
            break;
        }
        want -= __builtin_amdgcn_readlane(acc, 63);
    }
    if (s < 0) return;  // uniform: the grid is sized for the most blocks that n_seqs sequences can have
    const int q0 = __builtin_amdgcn_readfirstlane(want) * RQ;
    const int pos_off = ctx - qlen;
    const int* bt = block_tables + (size_t)s * bt_stride;

    // ---- which keys ----
    const int kv_end = min(ctx, pos_off + min(qlen, q0 + RQ));
    const int kt_begin = GEN && window > 0 ? max(0, pos_off + q0 - window + 1) / FT * FT : 0;
    const int n_tiles = kv_end > kt_begin ? (kv_end - kt_begin + FT - 1) / FT : 0;
    const int per = max(MIN_TILES, (n_tiles + n_parts - 1) / n_parts);
    const int live = max(1, (n_tiles + per - 1) / per);
    const int r = wave * 32 + col;               // this lane's column
    const int qi = q0 + r / G, hq = kvh * G + r % G;
    const bool real = r < RQ * G && qi < qlen;
    const size_t orow = (size_t)(qbeg + (real ? qi : 0)) * Hq + hq;  // row of out / of a part's results
    if (part >= live) {
        if (real && h == 0) part_ml[(size_t)part * T * Hq + orow] = make_float2(-INFINITY, 0.f);
        return;
    }
    const int t0 = part * per, t1 = min(n_tiles, t0 + per);

    // Q^T as B operand: lane = column, 8 dims 16 ks + 8 h (columns past the end repeat a real one, never stored)
    u32x4 qf[D / 16];
    {
        const bf16_t* qp = q + ((size_t)(qbeg + min(qi, qlen - 1)) * Hq + kvh * G + r % G) * D + 8 * h;
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks) qf[ks] = *(const u32x4*)(qp + 16 * ks);
    }
    f32x16 o[D / 32];
#pragma unroll
    for (int i = 0; i < D / 32; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) o[i][j] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;
    const float qs = scale * LOG2E;
    const float sc_l2 = softcap * LOG2E, cap_k = softcap > 0.f ? 2.f / softcap : 0.f;
    const int qpos = pos_off + qi;
    // the wave's smallest query position (uniform): tiles that end before it need no mask
    const int wq0 = pos_off + min(q0 + wave * 32 / G, qlen - 1);
    const int wq1 = pos_off + min(q0 + min(RQ - 1, (wave * 32 + 31) / G), qlen - 1);

    // A tile's chunks: rows one tile before they are stored. Rows past the last key repeat it: no column sees them.
    typename FRaw<KVF>::T kr[NCH], vr[NCH];
    constexpr int RPW = 512 / D;                 // rows that a wave requests at a time
    // UNI: a lane looks up one chunk of the wave's, lane = tile * NCH + chunk of GT tiles, and the next GT tiles' block id
    constexpr int GT = 64 / NCH;
    uint32_t place = 0;                          // its first row / RPW
    int next = 0;
    // else, for each of the thread's chunks, the block id and the row in it, one tile before the rows
    int blk[NCH], off[NCH];
    const size_t page = (size_t)Hkv * bs * D;
    auto first_key = [&](int t, int j) {         // of the wave's chunk j of tile t; past the end: the last key's rows
        return min(kt_begin + t * FT + j * (NT * 8 / D) + wave * RPW, (kv_end - 1) & -RPW);
    };
    auto page_of = [&](int key) { return bs_sh >= 0 ? key >> bs_sh : key / bs; };
    auto lane_key = [&](int t) { return first_key(t + lane / NCH, lane % NCH); };
    auto find_rows = [&](int t) {
        if constexpr (UNI) return;
#pragma unroll
        for (int j = 0; j < NCH; ++j) off[j] = min(kt_begin + t * FT + (int)(threadIdx.x + j * NT) / (D / 8), kv_end - 1);
        int bi[NCH];
        if (bs_sh >= 0) {
#pragma unroll
            for (int j = 0; j < NCH; ++j) bi[j] = off[j] >> bs_sh;
        } else {
#pragma unroll
            for (int j = 0; j < NCH; ++j) bi[j] = off[j] / bs;
        }
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
            blk[j] = bt[bi[j]];
            off[j] -= bi[j] * bs;
        }
    };
    auto look_up = [&](int t) {                  // before tile t's rows, tiles in turn from t0
        if constexpr (!UNI) return;
        if ((t - t0) % GT) return;
        const int key = lane_key(t), bi = page_of(key);
        place = (uint32_t)(next * Hkv + kvh) * (uint32_t)(bs / RPW) + (uint32_t)((key - bi * bs) / RPW);
        next = bt[page_of(lane_key(t + GT))];
    };
    auto load_chunk = [&](int t, int j) {
        if constexpr (UNI) {
            const size_t at = (size_t)(uint32_t)__builtin_amdgcn_readlane(place, (t - t0) % GT * NCH + j) * (RPW * f_row_bytes<KVF, D>());
            const uint32_t v = min(lane / (D / 8), kv_end - 1 - first_key(t, j)), e = lane % (D / 8) * 8;
            kr[j] = f_load_row<KVF, D>((const uint8_t*)kc + at, v, e);
            vr[j] = f_load_row<KVF, D>((const uint8_t*)vc + at, v, e);
        } else {
            const size_t eo = blk[j] * page + (size_t)((kvh * bs + off[j]) * D + (int)(threadIdx.x + j * NT) % (D / 8) * 8);
            kr[j] = f_load<KVF, D>(kc, eo);
            vr[j] = f_load<KVF, D>(vc, eo);
        }
    };
    auto store_k = [&](int buf, int j) {
        const int id = threadIdx.x + j * NT;
        *(uint4*)(smem + buf * (2 * IMG) + at_k_off<D>(id / (D / 8), id % (D / 8))) = f_widen<KVF>(kr[j]);
    };
    auto store_v = [&](int buf, int j) {
        const int id = threadIdx.x + j * NT, p = id / (D / 8), c = id % (D / 8);
        *(uint4*)(smem + buf * (2 * IMG) + IMG + at_v_off<D>(p, c >> 1) + 16 * (c & 1)) = f_widen<KVF>(vr[j]);
    };
    constexpr int KB = UNI || NW == 8 || D == 64 ? D / 64 : 1;  // k-steps whose K fragments are read together
    int vo[D / 32];
    at_v_lane<D>(lane, vo);
    // tile t + 1 from the registers to the other buffer, tile t + 2's rows requested: a piece beside each pair of products
    auto piece = [&](int t, int i) {
        if (i >= 2 * NCH) return;
        if (i % 2 == 0) store_k((t + 1) & 1, i / 2);
        else {
            store_v((t + 1) & 1, i / 2);
            load_chunk(min(t + 2, t1 - 1), i / 2);
        }
    };
    // the last tile has nothing to stage (storing it once more, 33 rows, us before / now: q5_1 9.3 / 8.0, q8_0 8.5 / 7.7, bf16 in pages of 10 8.3 / 7.5)
    auto work = [&](int t, auto more) {
        const char* kb = smem + (t & 1) * (2 * IMG);
        const char* vb = kb + IMG;
        const int kt0 = kt_begin + t * FT;
        f32x16 sc[2];
        if constexpr (decltype(more)::value) at_scores<D, false, KB>(kb, h, col, qf, sc, [&](int ks) { piece(t, ks); });
        else at_scores<D, false, KB>(kb, h, col, qf, sc);
        if (kt0 > wq1) return;  // (uniform per wave) tiles past the wave's last query carry nothing
        u32x4 vf[4][D / 32];
        __builtin_amdgcn_sched_barrier(0);
        at_read_v<D>(vb, vo, 0, vf);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (GEN) {
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    const float v = sc[u][j] * qs;
                    sc[u][j] = softcap > 0.f ? f_cap(v, sc_l2, cap_k) : v;
                }
        }
        if (kt0 + FT - 1 > wq0 || (GEN && window > 0 && kt0 <= wq1 - window)) {
            const int d = qpos - kt0 - 4 * h;  // (a real column's position is below ctx: later keys hide there too)
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    const int kp = 32 * u + 8 * (j >> 2) + (j & 3);
                    if (kp > d || (GEN && window > 0 && kp <= d - window)) sc[u][j] = -INFINITY;
                }
        }
        at_softmax_v<D, false>(vb, vo, sc, GEN ? 1.f : qs, vf, o, m_run, l_run);
    };

    if (t0 < t1) {
        if constexpr (UNI) next = bt[page_of(lane_key(t0))];
        look_up(t0);
        find_rows(t0);
#pragma unroll
        for (int j = 0; j < NCH; ++j) load_chunk(t0, j);
        find_rows(min(t0 + 1, t1 - 1));
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
            store_k(t0 & 1, j);
            store_v(t0 & 1, j);
        }
        if (t0 + 1 < t1) {
            look_up(t0 + 1);
#pragma unroll
            for (int j = 0; j < NCH; ++j) load_chunk(t0 + 1, j);
            find_rows(min(t0 + 2, t1 - 1));
        }
        __syncthreads();
        for (int t = t0; t < t1 - 1; ++t) {
            // the other buffer was last read while tile t - 1 was worked on, before the barrier that ended that round
            if (t + 2 < t1) look_up(t + 2);
            work(t, std::true_type{});
            find_rows(min(t + 3, t1 - 1));
            __syncthreads();
        }
        work(t1 - 1, std::false_type{});
    }
    l_run = at_half_sum(l_run);
    auto pack2 = [f16](float a, float b) { return f16 ? pack_act2<true>(a, b) : pack_act2<false>(a, b); };
    if (live == 1) {
        if (!real) return;
        if (n_parts > 1 && h == 0) part_ml[orow] = make_float2(0.f, -1.f);  // finished here: the merge leaves the row alone
        const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
#pragma unroll
        for (int mt = 0; mt < D / 32; ++mt)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *(uint2*)(out + orow * D + 32 * mt + 8 * g + 4 * h) =
                    make_uint2(pack2(o[mt][4 * g] * inv, o[mt][4 * g + 1] * inv),
                               pack2(o[mt][4 * g + 2] * inv, o[mt][4 * g + 3] * inv));
        return;
    }
    if (!real) return;
    const size_t pr = (size_t)part * T * Hq + orow;
    if (h == 0) part_ml[pr] = make_float2(m_run, l_run);
#pragma unroll
    for (int mt = 0; mt < D / 32; ++mt)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *(float4*)(part_o + pr * D + 32 * mt + 8 * g + 4 * h) =
                make_float4(o[mt][4 * g], o[mt][4 * g + 1], o[mt][4 * g + 2], o[mt][4 * g + 3]);
}

// out rows from the parts' (m, l, O): D / 8 lanes a row, 8 dims each. A row that one part finished alone (l < 0 in part 0)
// is left as it is, parts without a visible key (m = -inf) are not read.
template <int D>
__global__ __launch_bounds__(256) void attn_flash_merge_kernel(const float* __restrict__ part_o, const float2* __restrict__ part_ml,
                                                               int n_parts, const int* __restrict__ cu_q, int n_seqs, int T, int Hq,
                                                               bf16_t* __restrict__ out, int f16) {
    constexpr int LPR = D / 8;
    const long row = (long)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
    const int d0 = threadIdx.x % LPR * 8;
    if (row >= (long)min(T, cu_q[n_seqs]) * Hq) return;  // rows past the step's last query belong to nobody
    const size_t stride = (size_t)T * Hq;
    float mx = -INFINITY;
    for (int p = 0; p < n_parts; ++p) {
        const float2 ml = part_ml[p * stride + row];
        if (p == 0 && ml.y < 0.f) return;
        mx = fmaxf(mx, ml.x);
    }
    float ls = 0.f, acc[8] = {};
    for (int p = 0; p < n_parts; ++p) {
        const float2 ml = part_ml[p * stride + row];
        if (ml.x == -INFINITY) continue;
        const float a = exp2f(ml.x - mx);
        ls += ml.y * a;
        const float4* po = (const float4*)(part_o + (p * stride + row) * D + d0);
        const float4 x = po[0], y = po[1];
        acc[0] += x.x * a;
        acc[1] += x.y * a;
        acc[2] += x.z * a;
        acc[3] += x.w * a;
        acc[4] += y.x * a;
        acc[5] += y.y * a;
        acc[6] += y.z * a;
        acc[7] += y.w * a;
    }
    const float inv = ls > 0.f ? 1.f / ls : 0.f;
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
        w[e] = f16 ? pack_act2<true>(acc[2 * e] * inv, acc[2 * e + 1] * inv) : pack_act2<false>(acc[2 * e] * inv, acc[2 * e + 1] * inv);
    *(uint4*)(out + row * D + d0) = make_uint4(w[0], w[1], w[2], w[3]);
}

template <int D, int NW, int KVF>
int launch_flash(const bf16_t* q, const void* kc, const void* vc, const int* bt, int bt_stride, const int* cu_q, const int* ctx_lens,
                 int n_seqs, int T, int Hq, int Hkv, int bs, float scale, int window, float softcap, bf16_t* out, int n_parts,
                 float* part_o, float2* part_ml, hipStream_t st) {
    const int G = Hq / Hkv, RQ = 32 * NW / G;
    // the most blocks that n sequences of T rows together can have. (One more at every whole number of blocks left as many empty workgroups as a
    // block has, among which the others do not start evenly: 128 rows of 32 / 8 heads behind 4096 keys 41 -> 39 us, 256 53 -> 41)
    const long n = min(n_seqs, T), blocks = (T - n) / RQ + n;
    if (blocks > 65535) return (int)hipErrorInvalidValue;
    const dim3 grid(Hkv, (unsigned)blocks, n_parts);
    constexpr int LDS = 4 * FT * D * 2;
    const int sh = (bs & (bs - 1)) ? -1 : __builtin_ctz(bs);
    const bool gen = window > 0 || softcap > 0.f || !(scale > 0.f);
#define FL(GEN_, UNI_)                                                                                                       \
    do {                                                                                                                     \
        static const hipError_t once = hipFuncSetAttribute((const void*)attn_flash_kernel<D, NW, KVF, GEN_, UNI_>,            \
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, LDS);                 \
        if (once != hipSuccess) return (int)once;                                                                            \
        attn_flash_kernel<D, NW, KVF, GEN_, UNI_><<<grid, 64 * NW, LDS, st>>>(q, kc, vc, bt, bt_stride, cu_q, ctx_lens, n_seqs, \
                                                                             T, Hq, Hkv, G, bs, sh, scale, window, softcap,  \
                                                                             out, g_mx_act_f16, part_o, part_ml);                          \
    } while (0)
    if (bs % (512 / D) == 0) {
        if (gen) FL(true, true);
        else FL(false, true);
    } else {
        if (gen) FL(true, false);
        else FL(false, false);
    }
    if (n_parts > 1)
        attn_flash_merge_kernel<D><<<(unsigned)(((long)T * Hq * (D / 8) + 255) / 256), 256, 0, st>>>(part_o, part_ml, n_parts, cu_q,
                                                                                               n_seqs, T, Hq, out, g_mx_act_f16);
#undef FL
    MXK_CHECK_LAUNCH();
}

template <int D, int NW>
int dispatch_flash(const bf16_t* q, const void* kc, const void* vc, const int* bt, int bt_stride, const int* cu_q, const int* ctx_lens,
                   int n_seqs, int T, int Hq, int Hkv, int bs, float scale, int window, float softcap, bf16_t* out, int n_parts,
                   float* part_o, float2* part_ml, int kvf, hipStream_t st) {
#define FD(F_)                                                                                                                \
    case F_:                                                                                                                  \
        return launch_flash<D, NW, F_>(q, kc, vc, bt, bt_stride, cu_q, ctx_lens, n_seqs, T, Hq, Hkv, bs, scale, window, softcap, \
                                       out, n_parts, part_o, part_ml, st)
    switch (kvf) {
        FD(KVF_BF16);
        FD(KVF_FP8);
        FD(KVF_Q8_0);
        FD(KVF_Q4_0);
        FD(KVF_Q4_1);
        FD(KVF_Q5_0);
        FD(KVF_Q5_1);
        FD(KVF_IQ4_NL);
    }
#undef FD
    return (int)hipErrorInvalidValue;
}

}  // namespace

// q bf16 [T, Hq, D]; sequences cu_q [n_seqs + 1] with contexts ctx_lens; keys and values from the paged caches. waves: 4 or 8
// per workgroup (the caller's plan). n_parts > 1 needs part_o fp32 [n_parts, T, Hq, D] and part_ml float2 [n_parts, T, Hq].
extern "C" int mxk_attn_flash(const bf16_t* q, const void* kc, const void* vc, const int* bt, int bt_stride, const int* cu_q,
                              const int* ctx_lens, int n_seqs, int T, int Hq, int Hkv, int D, int bs, float scale, int window,
                              float softcap, bf16_t* out, int waves, int n_parts, float* part_o, float2* part_ml, int kvf, hipStream_t st) {
    if (T <= 0 || n_seqs <= 0) return 0;
    if (Hkv <= 0 || Hq % Hkv || Hq / Hkv > 128 || bs <= 0 || n_parts < 1 || n_parts > 64) return (int)hipErrorInvalidValue;
    if (n_parts > 1 && (!part_o || !part_ml)) return (int)hipErrorInvalidValue;
#define FW(D_, W_) \
    if (D == D_ && waves == W_)  \
        return dispatch_flash<D_, W_>(q, kc, vc, bt, bt_stride, cu_q, ctx_lens, n_seqs, T, Hq, Hkv, bs, scale, window, softcap, out, n_parts, part_o, part_ml, kvf, st)
    FW(128, 4);
    FW(128, 8);
    FW(64, 4);
    FW(64, 8);
#undef FW
    return (int)hipErrorInvalidValue;
}
