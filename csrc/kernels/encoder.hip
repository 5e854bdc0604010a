// encoder.hip — post-norm text encoders (BERT) on packed rows: the texts of a batch one after another, no padding rows.
//
// A layer is four GEMMs, attention (attention_dense.hip) and two LayerNorms. Batches of few rows are bound by launches
// and by the time a workgroup waits for its first loads, large ones by the GEMMs and by the passes between them; so
//   - up to 64 rows, more of narrow layers (models/bert.py few_rows), they run from one call (mxk_enc_layers), with a GEMM that splits K over the waves of a workgroup
//     and applies bias and GELU to its fp32 sums, and with what lies before a product done inside it where that is cheaper
//     than a launch: attention of one text up to 64 rows, the norms up to 16 (8 of several texts beyond 512 columns);
//   - above, and for wider layers below, they run from one call too (mxk_enc_layers_tiled), on dense16.hip's tiles with bias and GELU in the
//     up product's epilogue, the narrow products' sums in fp32 parts that the LayerNorm adds up, or 16 bits;
//   - widths that are no whole 64s: the first up to ops/dense.py small_rows, beyond that the caller multiplies with the library and the passes
//     between are one kernel each, over 16-bit rows.
// Measured on BERT-base, against padded rows with fp32 copies around each LayerNorm and a library call per operation: one
// text of 19 tokens 2019 -> 345 us (75 launches of 4-5 us; 8 tokens 275, 51 launches), 48 texts of 23-401 tokens (6428 rows of 19248 padded) 7147 ->
// 2041 on tiles (2278 with the library's products): LayerNorm + casts 74 -> 8.3 us (30 MB: 3.6 TB/s), GELU 40 -> 16 (79 MB: 4.9 TB/s) and then none.
#include "dense16.h"
#include "mx_common.h"

#include <type_traits>

namespace {

constexpr int EW = 4;  // rows (waves) per workgroup of the row kernels
constexpr int GW = 8;  // waves per workgroup of the GEMM
constexpr int ENC_ACT = 0, ENC_GELU = 1, ENC_PART = 2;  // what the GEMM writes
__host__ constexpr int enc_parts(int K) { return K >= 2048 ? 4 : 1; }

// A row is held by a wave: lane has the 8-element chunks lane + 64 j. Chunks past H are loaded from the row's last one and count
// as zero: loads behind a branch are waited for inside it, one after another (LayerNorm of 19 rows after four parts of a product
// 6.6 -> 4.6 us, the gains and offsets asked for ahead of the sums). So a lane is given no more chunks than the row has (ENC_NC).
MX_DEV int enc_chunk(int j, int H, int lane) { return min(8 * (lane + 64 * j), H - 8); }
MX_DEV bool enc_has(int j, int H, int lane) { return 8 * (lane + 64 * j) < H; }

template <int NC>
struct LnGain {
    float4 g[NC][2], b[NC][2];
    MX_DEV void load(const float* __restrict__ gp, const float* __restrict__ bp, int H, int lane) {
#pragma unroll
        for (int j = 0; j < NC; ++j)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int c = enc_chunk(j, H, lane) + 4 * e;
                g[j][e] = *(const float4*)(gp + c);
                b[j][e] = bp ? *(const float4*)(bp + c) : make_float4(0.f, 0.f, 0.f, 0.f);
            }
    }
};

// LayerNorm of one row. Two passes over registers: the variance is a sum of squares about the mean.
template <int NC, bool F16>
MX_DEV void ln_row(float (&v)[NC][8], int H, const LnGain<NC>& gb, float eps, uint16_t* __restrict__ out, int lane) {
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < NC; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) s += v[j][e];
    const float mean = wave_sum_all(s) / H;
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NC; ++j) {
        float q = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) q += (v[j][e] - mean) * (v[j][e] - mean);
        ss += enc_has(j, H, lane) ? q : 0.f;
    }
    const float rs = rsqrtf(wave_sum_all(ss) / H + eps);
#pragma unroll
    for (int j = 0; j < NC; ++j) {
        float y[8];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float4 gv = gb.g[j][e], bv = gb.b[j][e];
            y[4 * e] = (v[j][4 * e] - mean) * rs * gv.x + bv.x;
            y[4 * e + 1] = (v[j][4 * e + 1] - mean) * rs * gv.y + bv.y;
            y[4 * e + 2] = (v[j][4 * e + 2] - mean) * rs * gv.z + bv.z;
            y[4 * e + 3] = (v[j][4 * e + 3] - mean) * rs * gv.w + bv.w;
        }
        if (enc_has(j, H, lane))
            *(uint4*)(out + 8 * (lane + 64 * j)) = make_uint4(pack_act2<F16>(y[0], y[1]), pack_act2<F16>(y[2], y[3]),
                                                              pack_act2<F16>(y[4], y[5]), pack_act2<F16>(y[6], y[7]));
    }
}
template <int NC>
MX_DEV void add_f32(float (&v)[NC][8], const float* __restrict__ p, int H, int lane) {
#pragma unroll
    for (int j = 0; j < NC; ++j) {
        const int c = enc_chunk(j, H, lane);
        const bool has = enc_has(j, H, lane);
        const float4 a = *(const float4*)(p + c), b = *(const float4*)(p + c + 4);
        v[j][0] += has ? a.x : 0.f;
        v[j][1] += has ? a.y : 0.f;
        v[j][2] += has ? a.z : 0.f;
        v[j][3] += has ? a.w : 0.f;
        v[j][4] += has ? b.x : 0.f;
        v[j][5] += has ? b.y : 0.f;
        v[j][6] += has ? b.z : 0.f;
        v[j][7] += has ? b.w : 0.f;
    }
}

template <int NC, bool F16>
MX_DEV void add_act(float (&v)[NC][8], const uint16_t* __restrict__ p, int H, int lane) {
#pragma unroll
    for (int j = 0; j < NC; ++j) {
        const uint4 w = *(const uint4*)(p + enc_chunk(j, H, lane));
        const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float lo, hi;
            unpack_act2<F16>(enc_has(j, H, lane) ? ws[e] : 0u, lo, hi);
            v[j][2 * e] += lo;
            v[j][2 * e + 1] += hi;
        }
    }
}

// x = LN(tok[id] + pos[p] + typ[t]); ids: [3][rows] token, position, type (typ null: no type table)
template <int NC, bool F16>
__global__ __launch_bounds__(64 * EW) void enc_embed_kernel(const int* __restrict__ ids, int rows, const float* __restrict__ tok,
                                                            const float* __restrict__ pos, const float* __restrict__ typ,
                                                            const float* __restrict__ g, const float* __restrict__ b, int H,
                                                            float eps, uint16_t* __restrict__ x) {
    const int row = blockIdx.x * EW + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= rows) return;
    // gains ahead of the tables' rows where there are registers for both: a wide row's three tables and gains leave a SIMD a wave or
    // two (6428 rows of 2048 36.5 us, 17.4 with the gains after them), a narrow one is bound by its rows in flight (512: 5.6 / 5.4)
    constexpr bool AHEAD = NC == 2 || NC == 3;
    LnGain<NC> gb;
    float v[NC][8] = {};
    const int ti = ids[row], pi = ids[rows + row], yi = typ ? ids[2 * rows + row] : 0;
    if constexpr (AHEAD) gb.load(g, b, H, lane);
    add_f32<NC>(v, tok + (size_t)ti * H, H, lane);
    add_f32<NC>(v, pos + (size_t)pi * H, H, lane);
    if (typ) add_f32<NC>(v, typ + (size_t)yi * H, H, lane);
    if constexpr (!AHEAD) {
        __builtin_amdgcn_sched_barrier(0);
        gb.load(g, b, H, lane);
    }
    ln_row<NC, F16>(v, H, gb, eps, x + (size_t)row * H, lane);
}

// x = LN(a + x): the residual sum in fp32, one pass over 16-bit rows
template <int NC, bool F16>
__global__ __launch_bounds__(64 * EW) void enc_add_ln_kernel(const uint16_t* __restrict__ a, uint16_t* __restrict__ x, int rows,
                                                             const float* __restrict__ g, const float* __restrict__ b, int H,
                                                             float eps) {
    const int row = blockIdx.x * EW + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= rows) return;
    LnGain<NC> gb;
    gb.load(g, b, H, lane);
    float v[NC][8] = {};
    add_act<NC, F16>(v, a + (size_t)row * H, H, lane);
    add_act<NC, F16>(v, x + (size_t)row * H, H, lane);
    ln_row<NC, F16>(v, H, gb, eps, x + (size_t)row * H, lane);
}

// y = LN(sum of parts + bias + x); parts [NP][rows][H] fp32; y may be x
template <int NC, int NP, bool F16>
__global__ __launch_bounds__(64 * EW) void enc_parts_ln_kernel(const float* __restrict__ parts, const uint16_t* __restrict__ bias,
                                                               const uint16_t* x, uint16_t* y, int rows, const float* __restrict__ g,
                                                               const float* __restrict__ b, int H, float eps) {
    const int row = blockIdx.x * EW + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= rows) return;
    LnGain<NC> gb;
    gb.load(g, b, H, lane);
    float v[NC][8] = {};
#pragma unroll
    for (int p = 0; p < NP; ++p) add_f32<NC>(v, parts + ((size_t)p * rows + row) * H, H, lane);
    if (bias) add_act<NC, F16>(v, bias, H, lane);
    add_act<NC, F16>(v, x + (size_t)row * H, H, lane);
    ln_row<NC, F16>(v, H, gb, eps, y + (size_t)row * H, lane);
}

// y = gelu(y) in place, 8 elements a thread
template <bool F16>
__global__ __launch_bounds__(256) void enc_gelu_kernel(uint16_t* __restrict__ y, long n8) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n8) return;
    uint4 w = ((uint4*)y)[i];
    uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float lo, hi;
        unpack_act2<F16>(ws[e], lo, hi);
        ws[e] = pack_act2<F16>(gelu_erf_f(lo), gelu_erf_f(hi));
    }
    ((uint4*)y)[i] = make_uint4(ws[0], ws[1], ws[2], ws[3]);
}

// One text per workgroup -> e [H] fp32. mode 0: mean over its klen rows, 1: first row, 2: last row; then / max(|e|, 1e-12).
// Groups of H / 8 threads (at most 512) take every n-th row, 16 bytes a thread; their sums meet in LDS (H <= 4096). A text of
// 401 rows x 768 (0.6 MB): 56 us with 4-byte loads of four row groups, 9 with these.
template <bool F16>
__global__ __launch_bounds__(1024) void enc_pool_kernel(const uint16_t* __restrict__ x, const int* __restrict__ cu,
                                                        const int* __restrict__ klen, int H, int mode, int norm,
                                                        float* __restrict__ e) {
    __shared__ __attribute__((aligned(16))) float part[1024 * 8];
    __shared__ float red[16];
    const int b = blockIdx.x, r0 = cu[b], n = cu[b + 1] - r0, live = klen[b];
    const int lo = mode == 2 ? n - 1 : 0, hi = mode == 0 ? live : lo + 1;
    const int nc = H / 8, ng = 1024 / nc;  // (nc <= 512)
    const int grp = threadIdx.x / nc, c = threadIdx.x - grp * nc;
    float s[8] = {};
    if (grp < ng) {
        const uint16_t* xp = x + (size_t)r0 * H + 8 * c;
        auto add = [&](const uint4& w) {
            const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float a, d;
                unpack_act2<F16>(ws[i], a, d);
                s[2 * i] += a;
                s[2 * i + 1] += d;
            }
        };
        int r = lo + grp;
        for (; r + 3 * ng < hi; r += 4 * ng) {
            uint4 w[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) w[u] = *(const uint4*)(xp + (size_t)(r + u * ng) * H);
#pragma unroll
            for (int u = 0; u < 4; ++u) add(w[u]);
        }
        for (; r < hi; r += ng) add(*(const uint4*)(xp + (size_t)r * H));
        float* p = part + grp * H + 8 * c;
        *(float4*)p = make_float4(s[0], s[1], s[2], s[3]);
        *(float4*)(p + 4) = make_float4(s[4], s[5], s[6], s[7]);
    }
    __syncthreads();
    const float cnt = mode == 0 ? (float)max(live, 1) : 1.f;
    float sq = 0.f;
    for (int i = threadIdx.x; i < H; i += 1024) {
        float v = 0.f;
        for (int k = 0; k < ng; ++k) v += part[k * H + i];
        v /= cnt;
        part[i] = v;  // (group 0's sums: this thread alone reads them)
        sq += v * v;
    }
    sq = wave_sum(sq);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sq;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) tot += red[i];
    const float nr = norm ? fmaxf(sqrtf(tot), 1e-12f) : 1.f;
    for (int i = threadIdx.x; i < H; i += 1024) e[(size_t)b * H + i] = part[i] / nr;
}

template <bool F16>
MX_DEV f32x4 enc_mfma(u32x4 a, u32x4 b, f32x4 c) {
    if constexpr (F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// element idx of a 16 MT x 16 tile whose 8 waves' sums are in red
template <int MT, bool F16, int OUT>
MX_DEV void enc_store(const float* red, int idx, const uint16_t* __restrict__ bias, void* __restrict__ y, int m0, int M, int N, int n0) {
    const int n = idx & 15, r = idx >> 4, m = m0 + r;
    if (m >= M) return;
    const int e = (r >> 4) * 256 + (((r & 15) >> 2) * 16 + n) * 4 + (r & 3);
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < GW; ++w) v += red[w * MT * 256 + e];
    if constexpr (OUT == ENC_PART) {
        ((float*)y)[(size_t)m * N + n0 + n] = v;
    } else {
        if (bias) v += act_to_f32<F16>(bias[n0 + n]);
        if constexpr (OUT == ENC_GELU) v = gelu_erf_f(v);
        ((uint16_t*)y)[(size_t)m * N + n0 + n] = f32_to_act<F16>(v);
    }
}

// y[M, N] = act(x[M, K] W[N, K]^T + bias), 16-bit in and out, fp32 sums; or, ENC_PART, the fp32 sums of gridDim.z parts of K
// one after another, which the LayerNorm that follows adds up. A workgroup has 16 columns and 16 MT rows; its 8 waves take
// every 8th 32-wide k-step and their sums meet in LDS. What bounds it is the wait for the first loads: a wave asks for U
// k-steps at once (all three of K = 768). 19 rows: K = 768 4.5 us whatever N up to 3072; K = 3072, N = 768 9.4 us with 48
// workgroups (16 waves in each: the same), 4.5 in four parts. Rows past M read row M - 1 and are not stored.
template <int MT, bool F16, int OUT>
__global__ __launch_bounds__(64 * GW) void enc_gemm_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ W,
                                                           const uint16_t* __restrict__ bias, void* __restrict__ y, int M, int N,
                                                           int K) {
    __shared__ float red[GW * MT * 256];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16, m0 = blockIdx.y * (16 * MT);
    const int KS = K / 32 * (blockIdx.z + 1) / gridDim.z;
    const uint16_t* wp = W + (size_t)(n0 + col) * K + 8 * g;
    const uint16_t* xp[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) xp[t] = x + (size_t)min(m0 + 16 * t + col, M - 1) * K + 8 * g;
    f32x4 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    auto steps = [&](int s, auto uc) {
        constexpr int U = decltype(uc)::value;
        u32x4 wf[U], xf[U][MT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            wf[u] = *(const u32x4*)(wp + 32 * (s + GW * u));
#pragma unroll
            for (int t = 0; t < MT; ++t) xf[u][t] = *(const u32x4*)(xp[t] + 32 * (s + GW * u));
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[t] = enc_mfma<F16>(xf[u][t], wf[u], acc[t]);
    };
    constexpr int U = MT <= 2 ? 6 : 3;
    int s = K / 32 * blockIdx.z / gridDim.z + wave;
    for (; s + GW * (U - 1) < KS; s += GW * U) steps(s, std::integral_constant<int, U>{});
    if (U > 3 && s + GW * 2 < KS) {
        steps(s, std::integral_constant<int, 3>{});
        s += GW * 3;
    }
    for (; s < KS; s += GW) steps(s, std::integral_constant<int, 1>{});
#pragma unroll
    for (int t = 0; t < MT; ++t)
        *(float4*)(red + ((wave * MT + t) * 64 + lane) * 4) = make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]);
    __syncthreads();
    if constexpr (OUT == ENC_PART) y = (float*)y + (size_t)blockIdx.z * M * N;
    for (int idx = threadIdx.x; idx < MT * 256; idx += 64 * GW) enc_store<MT, F16, OUT>(red, idx, bias, y, m0, M, N, n0);
}

// ---- few rows: what comes before a product is done by each of its workgroups, on rows that stay in LDS ----
// Every launch of a layer waits ~4 us for its first loads whatever it does, and the host issues one in as long: seven a layer become six
// (one text up to 64 rows: attention inside the output product), five (several texts, up to 16 rows: both norms inside) or four. A
// workgroup has all M rows and 16 columns of the weights, whose fragments (all NS k-steps of its wave) are asked for ahead of the rows.
template <int MT, int NS, bool F16>
struct EncTail {
    u32x4 wf[NS];
    int wave, lane, steps;
    MX_DEV void load(const uint16_t* __restrict__ W, int n0, int K, int k0, int k1) {  // columns n0 .. n0 + 15, K's k0 .. k1
        wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        lane = threadIdx.x & 63;
        steps = (k1 - k0) / 32;
        const uint16_t* wp = W + (size_t)(n0 + (lane & 15)) * K + k0 + 8 * (lane >> 4);
#pragma unroll
        for (int u = 0; u < NS; ++u) wf[u] = *(const u32x4*)(wp + 32 * min(wave + GW * u, steps - 1));
    }
    // y[M, N] as enc_gemm_kernel's, from rows [16 MT][ld] in LDS that are complete behind a barrier; the sums take their place. ld: 8 more
    // than the rows have, so that 16 rows' chunks lie in different banks
    template <int OUT>
    MX_DEV void store(char* smem, int ld, const uint16_t* __restrict__ bias, void* __restrict__ y, int M, int N, int n0) {
        const uint16_t* rows = (const uint16_t*)smem + (lane & 15) * ld + 8 * (lane >> 4);
        float* red = (float*)smem;
        f32x4 acc[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < NS; ++u)
            if (wave + GW * u < steps)
#pragma unroll
                for (int t = 0; t < MT; ++t) acc[t] = enc_mfma<F16>(*(const u32x4*)(rows + 16 * t * ld + 32 * (wave + GW * u)), wf[u], acc[t]);
        __syncthreads();
#pragma unroll
        for (int t = 0; t < MT; ++t) *(float4*)(red + ((wave * MT + t) * 64 + lane) * 4) = make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]);
        __syncthreads();
        for (int idx = threadIdx.x; idx < MT * 256; idx += 64 * GW) enc_store<MT, F16, OUT>(red, idx, bias, y, 0, M, N, n0);
    }
};

// y = act(LN(sum of parts + pbias + x) W^T + bias); the first workgroup stores the normalised rows, the next residual, to xn (not x). A wave
// has RW rows. Bound by reading the parts into every compute unit: with 768 x 3072 weights and four parts 9.2 us at 16 rows, 13.3 at 19, where
// norm and product are 4.1 + 4.7; whole calls, us, norms apart / inside, 12 layers: 8 rows 398 / 279, 16 rows 403 / 339, 17 rows 344 / 435.
template <int RW, int NC, int NP, bool F16, int OUT>
__global__ __launch_bounds__(64 * GW) void enc_ln_gemm_kernel(const float* __restrict__ parts, const uint16_t* __restrict__ pbias,
                                                              const uint16_t* __restrict__ x, const float* __restrict__ g, const float* __restrict__ b,
                                                              float eps, uint16_t* __restrict__ xn, const uint16_t* __restrict__ W,
                                                              const uint16_t* __restrict__ bias, void* __restrict__ y, int M, int N, int K) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int n0 = blockIdx.x * 16, ld = K + 8;
    EncTail<(RW + 1) / 2, 2 * NC, F16> tail;
    tail.load(W, n0, K, 0, K);
    const int lane = tail.lane;
    LnGain<NC> gb;
    gb.load(g, b, K, lane);
    float v[RW][NC][8] = {};  // (rows past M: the last one's again, not stored)
#pragma unroll
    for (int i = 0; i < RW; ++i) {
        const int row = min(tail.wave + GW * i, M - 1);
#pragma unroll
        for (int p = 0; p < NP; ++p) add_f32<NC>(v[i], parts + ((size_t)p * M + row) * K, K, lane);
        if (pbias) add_act<NC, F16>(v[i], pbias, K, lane);
        add_act<NC, F16>(v[i], x + (size_t)row * K, K, lane);
    }
#pragma unroll
    for (int i = 0; i < RW; ++i) ln_row<NC, F16>(v[i], K, gb, eps, (uint16_t*)smem + (tail.wave + GW * i) * ld, lane);
    __syncthreads();
    if (blockIdx.x == 0)
        for (int c = threadIdx.x; c < M * (K / 8); c += 64 * GW) {
            const int r = c / (K / 8), e = (c - r * (K / 8)) * 8;
            *(uint4*)(xn + (size_t)r * K + e) = *(const uint4*)((const uint16_t*)smem + r * ld + e);
        }
    tail.template store<OUT>(smem, ld, bias, y, M, N, n0);
}

// y = attention(qkv) W^T, fp32, of one text of M <= 16 MT rows that sees its first klen keys; heads of 64, gridDim.z parts of them, whose
// products go to as many parts of y: every workgroup computes its heads anew for its 16 columns. A wave takes every 8th pair of a head
// and 16 queries: S^T = K Q^T gives a lane its query's keys 16 t + 4 g + i, which are the next product's B operand with the k slots in
// that order; V is gathered to match. Nothing but the heads' outputs goes through LDS. 12 heads, 19 rows: 4.3 us in four parts of the
// heads (8.6 in one: three pairs a wave, one after another) where attention and product were 4.6 + 4.3.
template <int MT, int NS, bool F16>
__global__ __launch_bounds__(64 * GW) void enc_attn_gemm_kernel(const uint16_t* __restrict__ qkv, const int* __restrict__ klen, float scale, int heads,
                                                                const uint16_t* __restrict__ W, float* __restrict__ y, int M, int H) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int h0 = heads * blockIdx.z / gridDim.z, h1 = heads * (blockIdx.z + 1) / gridDim.z;
    const int n0 = blockIdx.x * 16, ld = (h1 - h0) * 64 + 8, qld = 3 * H;
    EncTail<MT, NS, F16> tail;
    tail.load(W, n0, H, 64 * h0, 64 * h1);
    const int lane = tail.lane, col = lane & 15, g = lane >> 4;
    const int live = min(klen[0], M), last = max(live, 1) - 1;
    constexpr int KS = (MT + 1) / 2;  // 32-key steps
    const float qs = scale * 1.4426950408889634f;
    for (int u = tail.wave; u < (h1 - h0) * MT; u += GW) {
        const int hd = u / MT * 64, q0 = u % MT * 16;
        const uint16_t* base = qkv + 64 * h0 + hd;
        u32x4 qf[2], kf[MT][2];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            qf[ks] = *(const u32x4*)(base + (size_t)min(q0 + col, M - 1) * qld + 32 * ks + 8 * g);
#pragma unroll
            for (int t = 0; t < MT; ++t) kf[t][ks] = *(const u32x4*)(base + H + (size_t)min(16 * t + col, last) * qld + 32 * ks + 8 * g);
        }
        uint16_t vv[4][8 * KS] = {};  // [16 dims][key]
#pragma unroll
        for (int e = 0; e < 4 * MT; ++e) {
            const uint16_t* vp = base + 2 * H + (size_t)min(16 * (e >> 2) + 4 * g + (e & 3), last) * qld + col;
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) vv[mt][e] = vp[16 * mt];
        }
        float p[8 * KS] = {}, m = -INFINITY, l = 0.f;
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            f32x4 sc = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) sc = enc_mfma<F16>(kf[t][ks], qf[ks], sc);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                p[4 * t + i] = 16 * t + 4 * g + i < live ? sc[i] * qs : -INFINITY;
                m = fmaxf(m, p[4 * t + i]);
            }
        }
        m = fmaxf(m, __shfl_xor(m, 16));
        m = fmaxf(m, __shfl_xor(m, 32));
        const float mu = m == -INFINITY ? 0.f : m;
#pragma unroll
        for (int e = 0; e < 4 * MT; ++e) {
            p[e] = __builtin_amdgcn_exp2f(p[e] - mu);
            l += p[e];
        }
        l += __shfl_xor(l, 16);
        l += __shfl_xor(l, 32);
        const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            f32x4 o = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                uint32_t a[4], w[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int k = 8 * ks + 2 * e;
                    a[e] = (uint32_t)vv[mt][k] | (uint32_t)vv[mt][k + 1] << 16;
                    w[e] = pack_act2<F16>(p[k], p[k + 1]);
                }
                o = enc_mfma<F16>((u32x4){a[0], a[1], a[2], a[3]}, (u32x4){w[0], w[1], w[2], w[3]}, o);
            }
            *(uint2*)((uint16_t*)smem + (q0 + col) * ld + hd + 16 * mt + 4 * g) =
                live > 0 ? make_uint2(pack_act2<F16>(o[0] * inv, o[1] * inv), pack_act2<F16>(o[2] * inv, o[3] * inv)) : make_uint2(0, 0);
        }
    }
    __syncthreads();
    tail.template store<ENC_PART>(smem, ld, nullptr, y + (size_t)blockIdx.z * M * H, M, H, n0);
}

template <int MT>
constexpr size_t enc_fused_lds(int K) {
    const size_t rows = (size_t)16 * MT * (K + 8) * 2, red = (size_t)GW * MT * 1024;
    return rows > red ? rows : red;
}
constexpr int ENC_NORM_ROWS = 16, ENC_ATTN_ROWS = 64, ENC_FUSED_H = 1024;
int enc_attn_parts(int M, int heads) { return heads < 2 ? 1 : heads < 4 || M <= 16 ? 2 : 4; }  // of the heads: a pair a wave or two

template <bool F16, int OUT>
int enc_ln_gemm(int np, const float* parts, const uint16_t* pbias, const uint16_t* x, const float* g, const float* b, float eps, uint16_t* xn,
                const uint16_t* W, const uint16_t* bias, void* y, int M, int N, int K, hipStream_t st) {
#define EL(RW_, NC_, NP_)                                                                                                              \
    do {                                                                                                                               \
        constexpr int MT = (RW_ + 1) / 2;                                                                                              \
        static const hipError_t once = hipFuncSetAttribute((const void*)enc_ln_gemm_kernel<RW_, NC_, NP_, F16, OUT>,                   \
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)enc_fused_lds<MT>(512 * NC_)); \
        if (once != hipSuccess) return (int)once;                                                                                      \
        enc_ln_gemm_kernel<RW_, NC_, NP_, F16, OUT><<<N / 16, 64 * GW, enc_fused_lds<MT>(K), st>>>(parts, pbias, x, g, b, eps, xn, W, bias, y, M, N, K); \
        return (int)hipGetLastError();                                                                                                 \
    } while (0)
#define ELN(RW_)                             \
    if (M <= GW * RW_) {                     \
        if (K <= 512 && np == 1) EL(RW_, 1, 1); \
        if (K <= 512) EL(RW_, 1, MP);        \
        if constexpr (RW_ == 1 || OUT == ENC_ACT) /* (9 to 16 rows so wide are one text's, whose output product has two parts) */ \
            if (np == 1) EL(RW_, 2, 1);      \
        if (np == MP) EL(RW_, 2, MP);        \
    }
    constexpr int MP = OUT == ENC_ACT ? enc_parts(1 << 20) : 2;  // behind the down product; behind the output product of heads' parts up to 16 rows
    if ((np != 1 && np != MP) || K > 1024) return (int)hipErrorInvalidValue;
    ELN(1) ELN(2)
#undef ELN
#undef EL
    return (int)hipErrorInvalidValue;
}

template <bool F16>
int enc_attn_gemm(const uint16_t* qkv, const int* klen, float scale, int heads, const uint16_t* W, float* y, int M, int H, hipStream_t st) {
    const int parts = enc_attn_parts(M, heads), K = (heads + parts - 1) / parts * 64;  // (of the largest part)
#define EA(MT_, NS_)                                                                                                                   \
    do {                                                                                                                               \
        static const hipError_t once = hipFuncSetAttribute((const void*)enc_attn_gemm_kernel<MT_, NS_, F16>,                           \
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)enc_fused_lds<MT_>(256 * NS_)); \
        if (once != hipSuccess) return (int)once;                                                                                      \
        enc_attn_gemm_kernel<MT_, NS_, F16><<<dim3(H / 16, 1, parts), 64 * GW, enc_fused_lds<MT_>(K), st>>>(qkv, klen, scale, heads, W, y, M, H); \
        return (int)hipGetLastError();                                                                                                 \
    } while (0)
    // (of at most 16 heads: two parts of up to eight to 16 rows, above four parts or two pairs)
    if (K > (M <= 16 ? 512 : 256)) return (int)hipErrorInvalidValue;
    if (M <= 16 && K > 256) EA(1, 2);
    if (M <= 16) EA(1, 1);
    if (M <= 32) EA(2, 1);
    if (M <= 48) EA(3, 1);
    if (M <= 64) EA(4, 1);
#undef EA
    return (int)hipErrorInvalidValue;
}

template <bool F16, int OUT>
int enc_gemm(const uint16_t* x, const uint16_t* W, const uint16_t* bias, void* y, int M, int N, int K, hipStream_t st) {
    const int mt = min(4, (M + 15) / 16);
#define EG(MT_)                                                                                                            \
    if (mt == MT_)                                                                                                         \
        enc_gemm_kernel<MT_, F16, OUT><<<dim3(N / 16, (M + 16 * MT_ - 1) / (16 * MT_), OUT == ENC_PART ? enc_parts(K) : 1),    \
                                         64 * GW, 0, st>>>(x, W, bias, y, M, N, K);
    EG(1) EG(2) EG(3) EG(4)
#undef EG
    return (int)hipGetLastError();
}

// Chunks a lane holds, no more than the row has: those past its end are loaded all the same. With 2 and 8 alone, x = LN(a + x) of
// 6428 rows took, us, 256 / 512 / 1536 / 2048 wide: 5.6 / 6.0 / 17.0 / 18.9, now 4.1 / 4.5 / 10.1 / 14.7; 19 rows 2.7 / 2.7 / 4.2 /
// 4.2, now 2.3 / 2.3 / 2.9 / 3.2. The sum of the embeddings, 6428 rows: 7.1 / 7.4 / 33.3 / 36.5, now 5.0 / 5.4 / 13.1 / 17.4.
#define ENC_NC(H, ...)                                          \
    do {                                                        \
        if ((H) <= 512) { constexpr int NC = 1; __VA_ARGS__; }  \
        else if ((H) <= 1024) { constexpr int NC = 2; __VA_ARGS__; } \
        else if ((H) <= 1536) { constexpr int NC = 3; __VA_ARGS__; } \
        else if ((H) <= 2048) { constexpr int NC = 4; __VA_ARGS__; } \
        else if ((H) <= 3072) { constexpr int NC = 6; __VA_ARGS__; } \
        else { constexpr int NC = 8; __VA_ARGS__; }             \
    } while (0)

int enc_add_ln(const uint16_t* a, uint16_t* x, int rows, const float* g, const float* b, int H, float eps, hipStream_t st) {
    MX_ACT_DISPATCH(ENC_NC(H, enc_add_ln_kernel<NC, F16><<<(rows + EW - 1) / EW, 64 * EW, 0, st>>>(a, x, rows, g, b, H, eps)));
    return (int)hipGetLastError();
}

bool enc_width_ok(int H) { return H > 0 && H % 8 == 0 && H <= 4096; }

}  // namespace

extern "C" int mxk_attn_dense_ragged(const uint16_t* q, int q_stride, const uint16_t* k, int k_stride, const uint16_t* v,
                                     int v_stride, uint16_t* o, int o_stride, int B, int Smax, int H, int D, const int* cu,
                                     const int* klen, float scale, const int* blocks, int n_blocks, hipStream_t st);

extern "C" int mxk_enc_embed(const int* ids, int rows, const float* tok, const float* pos, const float* typ, const float* g,
                             const float* b, int H, float eps, uint16_t* x, hipStream_t st) {
    if (rows <= 0) return 0;
    if (!enc_width_ok(H)) return (int)hipErrorInvalidValue;
    MX_ACT_DISPATCH(ENC_NC(H, enc_embed_kernel<NC, F16><<<(rows + EW - 1) / EW, 64 * EW, 0, st>>>(ids, rows, tok, pos, typ, g, b,
                                                                                                 H, eps, x)));
    MXK_CHECK_LAUNCH();
}

extern "C" int mxk_enc_add_ln(const uint16_t* a, uint16_t* x, int rows, const float* g, const float* b, int H, float eps,
                              hipStream_t st) {
    if (rows <= 0) return 0;
    if (!enc_width_ok(H)) return (int)hipErrorInvalidValue;
    return enc_add_ln(a, x, rows, g, b, H, eps, st);
}

extern "C" int mxk_enc_gelu(uint16_t* y, long long n, hipStream_t st) {
    if (n <= 0) return 0;
    if (n % 8) return (int)hipErrorInvalidValue;
    const long n8 = n / 8;
    MX_ACT_DISPATCH(enc_gelu_kernel<F16><<<(unsigned)((n8 + 255) / 256), 256, 0, st>>>(y, n8));
    MXK_CHECK_LAUNCH();
}

extern "C" int mxk_enc_pool(const uint16_t* x, const int* cu, const int* klen, int B, int H, int mode, int norm, float* e,
                            hipStream_t st) {
    if (B <= 0) return 0;
    if (!enc_width_ok(H) || mode < 0 || mode > 2) return (int)hipErrorInvalidValue;
    MX_ACT_DISPATCH(enc_pool_kernel<F16><<<B, 1024, 0, st>>>(x, cu, klen, H, mode, norm, e));
    MXK_CHECK_LAUNCH();
}

// y = LN(sum of np parts + bias + x); y may be x
int enc_parts_ln(int np, const float* parts, const uint16_t* bias, const uint16_t* x, uint16_t* y, int rows, const float* g, const float* b, int H, float eps, hipStream_t st) {
    auto go = [&](auto kern) {
        kern<<<(rows + EW - 1) / EW, 64 * EW, 0, st>>>(parts, bias, x, y, rows, g, b, H, eps);
        return (int)hipGetLastError();
    };
    int rc = (int)hipErrorInvalidValue;
#define NP_(N_) \
    if (np == N_) MX_ACT_DISPATCH(ENC_NC(H, rc = go(enc_parts_ln_kernel<NC, N_, F16>)));
    NP_(1) NP_(2) NP_(3) NP_(4) NP_(8)
#undef NP_
    return rc;
}

// w: 12 device pointers a layer: qkv W, b, output W, b, norm g, b (fp32), up W, b, down W, b, norm g, b (fp32); biases may be
// null. x [rows][H] in and out; qkv [rows][3 H], attn [rows][H], up [rows][F] and parts [5][rows][H] fp32 are scratch.
extern "C" int mxk_enc_layers(const void* const* w, int n_layers, uint16_t* x, int rows, int B, int Smax, const int* cu,
                              const int* klen, int H, int heads, int F, float scale, float eps, uint16_t* qkv, uint16_t* attn,
                              float* parts, uint16_t* up, hipStream_t st) {
    if (rows <= 0 || n_layers <= 0) return 0;
    if (!enc_width_ok(H) || H % 32 || F % 32 || heads <= 0 || H % heads) return (int)hipErrorInvalidValue;
    static_assert(enc_parts(32) == 1 && enc_parts(1 << 20) == 4, "parts");
    const int np = enc_parts(F);
    const bool one = B == 1 && H / heads == 64 && rows <= ENC_ATTN_ROWS && H <= ENC_FUSED_H;
    // (layers alone, captured, 2 x 8 rows, us, norms apart / inside: 512 x 2048, 4 layers, 90 / 84, 640 x 2560 103 / 107)
    const bool norms = rows <= (one || H <= 512 ? ENC_NORM_ROWS : 8) && H <= ENC_FUSED_H;
    uint16_t* xm = norms ? (uint16_t*)(parts + (size_t)4 * rows * H) : x;  // the rows between a layer's halves: where none is read and written at once
    for (int l = 0; l < n_layers; ++l, w += 12) {
        auto at = [&](int i) { return (const uint16_t*)w[i]; };
        auto norm = [&](int i) { return (const float*)w[i]; };  // (of the layer before: - 12)
        const int np1 = one ? enc_attn_parts(rows, heads) : enc_parts(H);
        int rc = 0;
        if (norms && l) {
            MX_ACT_DISPATCH((rc = enc_ln_gemm<F16, ENC_ACT>(np, parts, at(-3), xm, norm(-2), norm(-1), eps, x, at(0), at(1), qkv, rows, 3 * H, H, st)));
        } else {
            MX_ACT_DISPATCH((rc = enc_gemm<F16, ENC_ACT>(x, at(0), at(1), qkv, rows, 3 * H, H, st)));
        }
        if (!rc && one) {
            MX_ACT_DISPATCH((rc = enc_attn_gemm<F16>(qkv, klen, scale, heads, at(2), parts, rows, H, st)));
        } else if (!rc) {
            rc = mxk_attn_dense_ragged(qkv, 3 * H, qkv + H, 3 * H, qkv + 2 * H, 3 * H, attn, H, B, Smax, heads, H / heads, cu, klen, scale, nullptr, 0, st);
            if (!rc) MX_ACT_DISPATCH((rc = enc_gemm<F16, ENC_PART>(attn, at(2), nullptr, parts, rows, H, H, st)));
        }
        if (!rc && norms) {
            MX_ACT_DISPATCH((rc = enc_ln_gemm<F16, ENC_GELU>(np1, parts, at(3), x, norm(4), norm(5), eps, xm, at(6), at(7), up, rows, F, H, st)));
        } else if (!rc) {
            rc = enc_parts_ln(np1, parts, at(3), x, x, rows, norm(4), norm(5), H, eps, st);
            if (!rc) MX_ACT_DISPATCH((rc = enc_gemm<F16, ENC_GELU>(x, at(6), at(7), up, rows, F, H, st)));
        }
        if (!rc) MX_ACT_DISPATCH((rc = enc_gemm<F16, ENC_PART>(up, at(8), nullptr, parts, rows, H, F, st)));
        if (!rc && (!norms || l == n_layers - 1)) rc = enc_parts_ln(np, parts, at(9), xm, x, rows, norm(10), norm(11), H, eps, st);
        if (rc) return rc;
    }
    return 0;
}

// The same layers by dense16.hip's tiles. plan: tile of the qkv product; tile and parts of K of the output product; tile of the up product; tile and
// parts of the down product: 1, 2, 3, 4 or 8 parts of fp32 sums, or 0: stored in 16 bits with its bias. H and F multiples of 64; parts
// [most parts][rows][H] where there are any. blocks: as mxk_attn_dense_ragged takes them.
extern "C" int mxk_enc_layers_tiled(const void* const* w, int n_layers, uint16_t* x, int rows, int B, int Smax, const int* cu, const int* klen, int H,
                                    int heads, int F, float scale, float eps, uint16_t* qkv, uint16_t* attn, float* parts, uint16_t* up,
                                    const int* plan, const int* blocks, int n_blocks, hipStream_t st) {
    if (rows <= 0 || n_layers <= 0) return 0;
    if (!enc_width_ok(H) || H % 64 || F <= 0 || F % 64 || heads <= 0 || H % heads) return (int)hipErrorInvalidValue;
    for (int l = 0; l < n_layers; ++l, w += 12) {
        auto at = [&](int i) { return (const uint16_t*)w[i]; };
        auto add_ln = [&](const uint16_t* a, int K, int tile, int np, int i) {  // x = LN(a W^T + bias + x): weights i, bias i + 1, norm i + 2
            const float *g = (const float*)w[i + 2], *b = (const float*)w[i + 3];
            if (np == 0) {  // (the q|k|v rows are read by now)
                const int rc = mx_dense16_enc(D16_ACT, tile, a, K, at(i), rows, H, K, at(i + 1), qkv, H, 1, nullptr, st);
                return rc ? rc : enc_add_ln(qkv, x, rows, g, b, H, eps, st);
            }
            const int rc = mx_dense16_enc(D16_PART, tile, a, K, at(i), rows, H, K, nullptr, nullptr, 0, np, parts, st);
            return rc ? rc : enc_parts_ln(np, parts, at(i + 1), x, x, rows, g, b, H, eps, st);
        };
        int rc = mx_dense16_enc(D16_ACT, plan[0], x, H, at(0), rows, 3 * H, H, at(1), qkv, 3 * H, 1, nullptr, st);
        if (!rc) rc = mxk_attn_dense_ragged(qkv, 3 * H, qkv + H, 3 * H, qkv + 2 * H, 3 * H, attn, H, B, Smax, heads, H / heads, cu, klen, scale, blocks, n_blocks, st);
        if (!rc) rc = add_ln(attn, H, plan[1], plan[2], 2);
        if (!rc) rc = mx_dense16_enc(D16_GELU, plan[3], x, H, at(6), rows, F, H, at(7), up, F, 1, nullptr, st);
        if (!rc) rc = add_ln(up, F, plan[4], plan[5], 8);
        if (rc) return rc;
    }
    return 0;
}
