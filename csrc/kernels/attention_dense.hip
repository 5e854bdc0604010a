// attention_dense.hip — fused MFMA flash attention over dense (non-paged) Q/K/V, for the encoder /
// diffusion / embedding models: BERT & cross-encoders (key padding), Whisper encoder (bidirectional)
// and decoder (causal self-attention, cross-attention to the audio states), UNet / MMDiT attention
// (SURVEY §2.6 K4 for the non-LLM workers).
//
//   O[b, i, h, :] = softmax(scale · Q[b, i, h, :] · K[b, :, h/G, :]^T  (+ masks)) · V[b, :, h/G, :]
//
// Layout: token-major rows with explicit strides (q/k/v/o[(b·S + s)·stride + head·D + d]) so fused
// QKV projections can be consumed in place. 16-bit operands in the library's act16 format (bf16 or
// f16 MFMA), fp32 softmax state, online (flash) softmax in the log2 domain.
// Head dims 64 / 128 (attn_dense_t_kernel): 4 (or 2) waves x 32 queries of one head; scores are computed transposed,
// S^T = K Q^T on 32x32x16 tiles, so that a query's softmax stays in two lanes and its probabilities are the B operand of
// O^T = V^T P^T as they lie (V^T's keys read in S^T's order); K/V staged 64 keys at a time, two tiles in LDS, one more in
// registers. Against 16 query rows a wave with P through LDS (f16, no mask): 4096 x 4096, 2 x 10 heads of 64 388 -> 138 us (622
// TFLOP/s), 1500 x 1500, 20 heads 76 -> 33, 4500 x 4500, 24 heads of 128 824 -> 343 (725 TFLOP/s), 1 x 1500, 20 heads 58 -> 22,
// 77 x 77, 8 x 12 heads 9 -> 9 (a launch). Large ones are bound by the LDS reads of K and V (each feeds one product), small
// ones by the chain of a tile. Head dim 512: 4 waves x 16 query rows, 32 keys at a time, P through LDS.
// Masks: `causal` (key position > query position + (Sk - Sq) dropped) and per-batch key lengths
// `klen` (BERT padding); rows past `qlen[b]` are not written. Optional additive relative-position bias
// `rbias[h][j - i + Sq - 1]` (fp32, T5's bucketed bias table expanded per offset; shared by the batch).
#include "attn_tile.h"

#define LOG2E_D 1.4426950408889634f

// Head dim 512. K image: row p holds D/8 16-byte chunks; chunk c lives at c ^ f(p) (f < 16: 16 consecutive rows, one chunk
// column, land in 16 different banks).
template <int D>
MX_DEV int kd_lds_off(int p, int c) {
    const int r = p & 15;
    return p * (D * 2) + ((c ^ r ^ (((r + 4) >> 3) & 1)) << 4);
}
template <int D>
MX_DEV int vd_lds_off(int p, int nt) {
    return p * (D * 2) + ((nt ^ ((p & 3) | (((p >> 3) & 1) << 2))) << 5);
}

template <bool F16>
MX_DEV f32x4 mfma16(const u32x4& a, const u32x4& b, f32x4 c) {
    if constexpr (F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                       0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                        c, 0, 0, 0);
}

template <int D, bool F16>
__global__ __launch_bounds__(256) void attn_dense_kernel(const uint16_t* __restrict__ q, int q_stride,
                                                         const uint16_t* __restrict__ k, int k_stride,
                                                         const uint16_t* __restrict__ v, int v_stride,
                                                         uint16_t* __restrict__ o, int o_stride, int Sq, int Sk,
                                                         int Hq, int Hkv, const int* __restrict__ qlen_b,
                                                         const int* __restrict__ klen_b, int causal, float scale,
                                                         int kv_rows, const float* __restrict__ rbias, int rb_ld) {
    static_assert(D == 512, "smaller head dims: attn_dense_t_kernel");
    constexpr int KT = 32;  // keys per tile (the VAE mid-block's single 512-wide head; K + V tiles 64 KB)
    constexpr int KBYTES = KT * D * 2;
    constexpr int PSTRIDE = (KT + 8) * 2;
    __shared__ __attribute__((aligned(16))) char smem[2 * KBYTES + 4 * 16 * PSTRIDE];
    char* k_lds = smem;
    char* v_lds = smem + KBYTES;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int g = lane >> 4, col = lane & 15;
    const int b = blockIdx.z, h = blockIdx.y;
    const int kvh = h / (Hq / Hkv);
    const int qlen = qlen_b ? qlen_b[b] : Sq;
    const int klen = klen_b ? klen_b[b] : Sk;
    const int row_q0 = blockIdx.x * 64 + wave * 16;
    if (blockIdx.x * 64 >= qlen) return;  // whole workgroup idle (uniform)
    const int shift = Sk - Sq;            // causal: query i sees keys <= i + shift
    int kv_end = klen;
    if (causal) kv_end = min(kv_end, blockIdx.x * 64 + 64 + shift);
    const float qs = scale * LOG2E_D;
    const uint16_t* kb = k + (size_t)b * kv_rows * k_stride + (size_t)kvh * D;
    const uint16_t* vb_ = v + (size_t)b * kv_rows * v_stride + (size_t)kvh * D;

    u32x4 qf[D / 32];
    {
        const int qi = row_q0 + col;
#pragma unroll
        for (int ks = 0; ks < D / 32; ++ks) {
            if (qi < qlen) qf[ks] = *(const u32x4*)(q + ((size_t)b * Sq + qi) * q_stride + (size_t)h * D + 32 * ks + 8 * g);
            else qf[ks] = (u32x4){0, 0, 0, 0};
        }
    }
    f32x4 oacc[D / 16];
#pragma unroll
    for (int i = 0; i < D / 16; ++i) oacc[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float mrow[4], lrow[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) { mrow[i] = -INFINITY; lrow[i] = 0.f; }
    char* pw = smem + 2 * KBYTES + wave * 16 * PSTRIDE;

    // (a tile is 8 chunks per thread and per operand: asking for the next one ahead would spill, so each loads in place)
    constexpr int CH = KT * D / 8;
    constexpr int NCH = (CH + 255) / 256;  // chunks per thread
    uint4 kr[NCH], vr[NCH];
    auto load_tile = [&](int kt0) {
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
            const int id = threadIdx.x + 256 * j;
            const int p = id / (D / 8), c = id % (D / 8);
            const int pos = kt0 + p;
            kr[j] = make_uint4(0, 0, 0, 0);
            vr[j] = make_uint4(0, 0, 0, 0);
            if (id < CH && pos < kv_end) {
                kr[j] = *(const uint4*)(kb + (size_t)pos * k_stride + c * 8);
                vr[j] = *(const uint4*)(vb_ + (size_t)pos * v_stride + c * 8);
            }
        }
    };
    for (int kt0 = 0; kt0 < kv_end; kt0 += KT) {
        load_tile(kt0);
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
            const int id = threadIdx.x + 256 * j;
            if (id >= CH) continue;
            const int p = id / (D / 8), c = id % (D / 8);
            *(uint4*)(k_lds + kd_lds_off<D>(p, c)) = kr[j];
            *(uint4*)(v_lds + vd_lds_off<D>(p, c >> 1) + 16 * (c & 1)) = vr[j];
        }
        __syncthreads();
        constexpr int NT16 = KT / 16;
        f32x4 sacc[NT16];
#pragma unroll
        for (int t = 0; t < NT16; ++t) {
            sacc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < D / 32; ++ks) {
                const u32x4 kf = *(const u32x4*)(k_lds + kd_lds_off<D>(16 * t + col, 4 * ks + g));
                sacc[t] = mfma16<F16>(qf[ks], kf, sacc[t]);
            }
        }
        float rmax[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int qi = row_q0 + 4 * g + i;
            float mx = -INFINITY;
#pragma unroll
            for (int t = 0; t < NT16; ++t) {
                const int kp = kt0 + 16 * t + col;
                float s = sacc[t][i] * qs;
                if (kp >= kv_end || qi >= qlen || (causal && kp > qi + shift)) s = -INFINITY;
                else if (rbias) s += rbias[(size_t)h * rb_ld + (kp - qi + Sq - 1)] * LOG2E_D;
                sacc[t][i] = s;
                mx = fmaxf(mx, s);
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
            for (int t = 0; t < NT16; ++t) {
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
#pragma unroll
        for (int t = 0; t < NT16; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *(uint16_t*)(pw + (4 * g + i) * PSTRIDE + (16 * t + col) * 2) = f32_to_act<F16>(sacc[t][i]);
        __builtin_amdgcn_s_waitcnt(0xc07f);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int ks = 0; ks < KT / 32; ++ks) {
            const u32x4 pa = *(const u32x4*)(pw + col * PSTRIDE + (32 * ks + 8 * g) * 2);
            const int r0 = 32 * ks + 8 * g;
            const int q4 = col >> 2, p4 = col & 3;
#pragma unroll
            for (int nt = 0; nt < D / 16; ++nt) {
                const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (MX_LDS s16x4*)(v_lds + vd_lds_off<D>(r0 + q4, nt) + 8 * p4));
                const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (MX_LDS s16x4*)(v_lds + vd_lds_off<D>(r0 + 4 + q4, nt) + 8 * p4));
                const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
                const u32x4 vv = {l2[0], l2[1], h2[0], h2[1]};
                oacc[nt] = mfma16<F16>(pa, vv, oacc[nt]);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int qi = row_q0 + 4 * g + i;
        if (qi >= qlen) continue;
        const float inv = lrow[i] > 0.f ? 1.f / lrow[i] : 0.f;
#pragma unroll
        for (int nt = 0; nt < D / 16; ++nt)
            o[((size_t)b * Sq + qi) * o_stride + (size_t)h * D + 16 * nt + col] = f32_to_act<F16>(oacc[nt][i] * inv);
    }
}

// ---- head dims 64 / 128 ----
// GEN: a position bias, or a scale that is not positive; without it the scale is one FMA with the maximum
template <int D, int NW, bool F16, bool GEN>
__global__ __launch_bounds__(64 * NW, 2) void attn_dense_t_kernel(const uint16_t* __restrict__ q, int q_stride,
                                                              const uint16_t* __restrict__ k, int k_stride,
                                                              const uint16_t* __restrict__ v, int v_stride,
                                                              uint16_t* __restrict__ o, int o_stride, int Sq, int Sk, int Hq,
                                                              int Hkv, const int* __restrict__ qlen_b,
                                                              const int* __restrict__ klen_b, int causal, float scale,
                                                              int kv_rows, const float* __restrict__ rbias, int rb_ld,
                                                              const int* __restrict__ cu, const int* __restrict__ blocks) {
    constexpr int FT = AT_KEYS, IMG = FT * D * 2;
    constexpr int NCH = FT * D / 8 / (64 * NW);  // 16-byte chunks of an image per thread
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int h = lane >> 5, col = lane & 31;
    // `blocks`: the (sequence, first query) of a block, in the order they are to start
    const int b = blocks ? blocks[2 * blockIdx.y] : blockIdx.z, head = blocks ? blockIdx.x : blockIdx.y, kvh = head / (Hq / Hkv);
    const int q0 = blocks ? blocks[2 * blockIdx.y + 1] : blockIdx.x * (32 * NW);
    // ragged batches: sequence b's rows are cu[b] .. cu[b + 1], keys and queries alike
    const size_t q_row = cu ? (size_t)cu[b] : (size_t)b * Sq, k_row = cu ? (size_t)cu[b] : (size_t)b * kv_rows;
    const int qlen = cu ? cu[b + 1] - cu[b] : qlen_b ? qlen_b[b] : Sq;
    if (q0 >= qlen) return;  // whole workgroup idle (uniform)
    const int shift = Sk - Sq;  // causal: query i sees keys <= i + shift
    int kv_end = klen_b ? klen_b[b] : Sk;
    if (causal) kv_end = min(kv_end, min(q0 + 32 * NW, qlen) + shift);
    const int n_tiles = kv_end > 0 ? (kv_end + FT - 1) / FT : 0;
    const uint16_t* kb_ = k + k_row * k_stride + (size_t)kvh * D;
    const uint16_t* vb_ = v + k_row * v_stride + (size_t)kvh * D;
    const int qi = q0 + wave * 32 + col;
    const bool real = qi < qlen;
    u32x4 qf[D / 16];  // Q^T as B operand: lane = query (past the end: the last one, not stored), 8 dims 16 ks + 8 h
    {
        const uint16_t* qp = q + (q_row + min(qi, qlen - 1)) * q_stride + (size_t)head * D + 8 * h;
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks) qf[ks] = *(const u32x4*)(qp + 16 * ks);
    }
    f32x16 acc[D / 32];
#pragma unroll
    for (int i = 0; i < D / 32; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;
    const float qs = scale * LOG2E_D;
    const int lim = causal ? min(kv_end - 1, min(qi, qlen - 1) + shift) : kv_end - 1;  // last key of this query
    const int wq0 = q0 + wave * 32, wq1 = min(wq0 + 31, qlen - 1);                     // the wave's queries
    const int wlim0 = causal ? min(kv_end - 1, wq0 + shift) : kv_end - 1;
    const int wlim1 = wq0 >= qlen ? -1 : causal ? min(kv_end - 1, wq1 + shift) : kv_end - 1;
    const float* rb = GEN && rbias ? rbias + (size_t)head * rb_ld + (Sq - 1 - min(qi, qlen - 1)) : nullptr;

    u32x4 kr[NCH], vr[NCH];  // rows past the last key repeat it: no query sees them
    auto load_rows = [&](int t) {
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
            const int id = threadIdx.x + 64 * NW * j, p = min(t * FT + id / (D / 8), kv_end - 1), c = id % (D / 8);
            kr[j] = *(const u32x4*)(kb_ + (size_t)p * k_stride + c * 8);
            vr[j] = *(const u32x4*)(vb_ + (size_t)p * v_stride + c * 8);
        }
    };
    auto store_rows = [&](int buf) {
        char* kb = smem + buf * (2 * IMG);
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
            const int id = threadIdx.x + 64 * NW * j, p = id / (D / 8), c = id % (D / 8);
            *(u32x4*)(kb + at_k_off<D>(p, c)) = kr[j];
            *(u32x4*)(kb + IMG + at_v_off<D>(p, c >> 1) + 16 * (c & 1)) = vr[j];
        }
    };
    int vo[D / 32];
    at_v_lane<D>(lane, vo);
    auto work = [&](int t) {
        const char* kb = smem + (t & 1) * (2 * IMG);
        const char* vb = kb + IMG;
        const int kt0 = t * FT;
        f32x16 sc[2];
        at_scores<D, F16, 2>(kb, h, col, qf, sc);
        u32x4 vf[4][D / 32];
        __builtin_amdgcn_sched_barrier(0);
        at_read_v<D>(vb, vo, 0, vf);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (GEN) {
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    const int kp = kt0 + 32 * u + 8 * (j >> 2) + 4 * h + (j & 3);
                    sc[u][j] *= qs;
                    if (rb) sc[u][j] += rb[min(kp, kv_end - 1)] * LOG2E_D;
                }
        }
        if (kt0 + FT - 1 > wlim0) {
            const int d = lim - kt0 - 4 * h;
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    if (32 * u + 8 * (j >> 2) + (j & 3) > d) sc[u][j] = -INFINITY;
        }
        at_softmax_v<D, F16>(vb, vo, sc, GEN ? 1.f : qs, vf, acc, m_run, l_run);
    };
    if (n_tiles > 0) {
        load_rows(0);
        store_rows(0);
        if (n_tiles > 1) load_rows(1);
        __syncthreads();
        for (int t = 0; t < n_tiles; ++t) {
            // the other buffer was last read while tile t - 1 was worked on, before the barrier that ended that round; half
            // of the waves store first and half work first, so that one's products run beside the other's loads
            auto stage = [&]() {
                if (t + 1 >= n_tiles) return;
                store_rows((t + 1) & 1);
                if (t + 2 < n_tiles) load_rows(t + 2);
            };
            const bool first = wave < NW / 2;
            if (first) stage();
            if (t * FT <= wlim1) work(t);  // (uniform per wave) tiles past the wave's last key carry nothing
            if (!first) stage();
            __syncthreads();
        }
    }
    l_run = at_half_sum(l_run);
    if (!real) return;
    const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
    uint16_t* op = o + (q_row + qi) * o_stride + (size_t)head * D + 4 * h;
    const bool wide = ((uintptr_t)o | (uintptr_t)(2 * o_stride)) % 8 == 0;
#pragma unroll
    for (int mt = 0; mt < D / 32; ++mt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const uint2 w = make_uint2(pack_act2<F16>(acc[mt][4 * g] * inv, acc[mt][4 * g + 1] * inv),
                                       pack_act2<F16>(acc[mt][4 * g + 2] * inv, acc[mt][4 * g + 3] * inv));
            uint16_t* d = op + 32 * mt + 8 * g;
            if (wide) {
                *(uint2*)d = w;
            } else {
                d[0] = (uint16_t)w.x;
                d[1] = (uint16_t)(w.x >> 16);
                d[2] = (uint16_t)w.y;
                d[3] = (uint16_t)(w.y >> 16);
            }
        }
}

template <int D, int NW, bool F16>
static int launch_dense_t(const uint16_t* q, int q_stride, const uint16_t* k, int k_stride, const uint16_t* v, int v_stride,
                          uint16_t* o, int o_stride, int B, int Sq, int Sk, int Hq, int Hkv, const int* qlen, const int* klen,
                          int causal, float scale, int kv_rows, const float* rbias, int rb_ld, const int* cu, const int* blocks, int n_blocks,
                          hipStream_t st) {
    constexpr int LDS = 4 * 64 * D * 2;
    const dim3 grid = blocks ? dim3(Hq, n_blocks) : dim3((Sq + 32 * NW - 1) / (32 * NW), Hq, B);
#define DT(GEN_)                                                                                                              \
    do {                                                                                                                      \
        static const hipError_t once = hipFuncSetAttribute((const void*)attn_dense_t_kernel<D, NW, F16, GEN_>,                \
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, LDS);                  \
        if (once != hipSuccess) return (int)once;                                                                             \
        attn_dense_t_kernel<D, NW, F16, GEN_><<<grid, 64 * NW, LDS, st>>>(q, q_stride, k, k_stride, v, v_stride, o, o_stride, \
                                                                          Sq, Sk, Hq, Hkv, qlen, klen, causal, scale, kv_rows, \
                                                                          rbias, rb_ld, cu, blocks);                          \
    } while (0)
    if (rbias || !(scale > 0.f)) DT(true);
    else DT(false);
#undef DT
    return (int)hipGetLastError();
}

static int dense_t(const uint16_t* q, int q_stride, const uint16_t* k, int k_stride, const uint16_t* v, int v_stride, uint16_t* o,
                   int o_stride, int B, int Sq, int Sk, int Hq, int Hkv, int D, const int* qlen, const int* klen, int causal,
                   float scale, int kv_rows, const float* rbias, int rb_ld, const int* cu, const int* blocks, int n_blocks, hipStream_t st) {
    // two waves for ragged heads of 64, where the last block of each sequence is part empty (48 texts of 23-401 rows, 12 heads:
    // 23.7 us against 29.8; at 401 rows each 80 against 69); four waves elsewhere, whatever the grid (1500 rows, 20 heads:
    // 32.6 against 40.5; 4500 rows of 24 heads of 128: 343 against 515)
    int rc = 0;
#define DTL(D_, NW_) launch_dense_t<D_, NW_, F16>(q, q_stride, k, k_stride, v, v_stride, o, o_stride, B, Sq, Sk, Hq, Hkv, qlen, \
                                                  klen, causal, scale, kv_rows, rbias, rb_ld, cu, blocks, n_blocks, st)
    MX_ACT_DISPATCH(rc = D == 128 ? DTL(128, 4) : cu ? DTL(64, 2) : DTL(64, 4));
#undef DTL
    return rc;
}

// q/k/v/o: 16-bit (act16 mode) token-major with row strides in elements; B batches of Sq queries /
// Sk keys; Hq query heads, Hkv key/value heads (Hq % Hkv == 0); D in {64, 128, 512}. K/V rows of batch b
// start at row b * kv_rows (kv_rows = 0 -> Sk): a fixed-capacity KV cache [B, cap, H*D] is read in
// place with Sk = valid length (causal offset Sk - Sq) or Sk = cap with per-batch klen.
extern "C" int mxk_attn_dense(const uint16_t* q, int q_stride, const uint16_t* k, int k_stride, const uint16_t* v,
                              int v_stride, uint16_t* o, int o_stride, int B, int Sq, int Sk, int Hq, int Hkv, int D,
                              const int* qlen, const int* klen, int causal, float scale, int kv_rows,
                              const float* rbias, int rb_ld, hipStream_t st) {
    if (B <= 0 || Sq <= 0) return 0;
    if (kv_rows <= 0) kv_rows = Sk;
    if (Hq % Hkv || (D != 64 && D != 128 && D != 512)) return (int)hipErrorInvalidValue;
    if ((q_stride | k_stride | v_stride) & 7) return (int)hipErrorInvalidValue;
    if (D != 512)
        return dense_t(q, q_stride, k, k_stride, v, v_stride, o, o_stride, B, Sq, Sk, Hq, Hkv, D, qlen, klen, causal, scale,
                       kv_rows, rbias, rb_ld, nullptr, nullptr, 0, st);
    MX_ACT_DISPATCH((attn_dense_kernel<512, F16><<<dim3((Sq + 63) / 64, Hq, B), 256, 0, st>>>(
        q, q_stride, k, k_stride, v, v_stride, o, o_stride, Sq, Sk, Hq, Hkv, qlen, klen, causal, scale, kv_rows, rbias, rb_ld)));
    MXK_CHECK_LAUNCH();
}

// Rows packed without padding (BERT): sequence b of B has rows cu[b] .. cu[b + 1] (at most Smax) of q, k, v and o, and sees
// its first klen[b] keys; D in {64, 128}. blocks (or null): n_blocks pairs (b, first query), one for every 64 (D 64) or 128 queries that a sequence
// has, in the order they start. A block's time is its keys', so the longest come first: in the order of 48 texts of 23 to 401 rows from the
// shortest, 12 heads, the last ones' seven key tiles ran after all else (24.1 us, so 19.9).
extern "C" int mxk_attn_dense_ragged(const uint16_t* q, int q_stride, const uint16_t* k, int k_stride, const uint16_t* v,
                                     int v_stride, uint16_t* o, int o_stride, int B, int Smax, int H, int D, const int* cu,
                                     const int* klen, float scale, const int* blocks, int n_blocks, hipStream_t st) {
    if (B <= 0 || Smax <= 0) return 0;
    if ((D != 64 && D != 128) || B > 65535 || !cu || !klen || (blocks && (n_blocks <= 0 || n_blocks > 65535))) return (int)hipErrorInvalidValue;
    if ((q_stride | k_stride | v_stride) & 7) return (int)hipErrorInvalidValue;
    return dense_t(q, q_stride, k, k_stride, v, v_stride, o, o_stride, B, Smax, Smax, H, H, D, nullptr, klen, 0, scale, 0, nullptr,
                   0, cu, blocks, n_blocks, st);
}
