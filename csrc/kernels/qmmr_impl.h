// qmmr_impl.h — kernel template of qmmr.hip (see there), shared by the per-format translation units.
#pragma once
#include "qmm2_fmt.h"

namespace {

constexpr int QR_PITCH = 528;  // bytes of a staged A row: 256 k of f16 and 16 more, so 16 rows start in 16 bank quads

template <int WM, int GW, int KW>
struct QrGeom {
    static constexpr int NT = 64 * GW * KW;
    static constexpr int BM = 32 * WM;                      // rows
    static constexpr int SLOT = BM * QR_PITCH;              // one super-block of A
    static constexpr int RED = GW * KW * 4096;              // one 32-row block's partial sums
    static constexpr int LDS = 2 * SLOT > RED ? 2 * SLOT : RED;
    static constexpr int AP = BM * 32 / NT;                 // 16-byte pieces of A a thread stages per super-block
};

// (workgroup `bid` of the `nwg` that share the product)
template <int QT, int WM, int GW, int KW, int EPI>
MX_DEV void qmmr_body(const int nwg, const int bid, const uint16_t* __restrict__ A, int lda, const uint8_t* __restrict__ W, int M, int N, int K,
                      int n_mt, int splits, int sbps, void* __restrict__ Cv, int ldc) {
    using G = QrGeom<WM, GW, KW>;
    using F = Q2F<QT>;
    constexpr int BM = G::BM, AP = G::AP, NQ = 4 / KW;
    static_assert(KW == 2 || KW == 4, "KW");
    static_assert(AP >= 1 && AP * G::NT == BM * 32, "A pieces");
    static_assert(G::LDS <= 160 * 1024, "LDS");
    extern __shared__ __attribute__((aligned(16))) char smem[];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int h = lane >> 5, col = lane & 31;
    const int gw = wave % GW, kw = wave / GW;

    // consecutive logical ids run on one XCD (q2_tile_of)
    const int xcd = bid & 7, q8 = nwg >> 3, r8 = nwg & 7;
    const int lid = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + (bid >> 3);
    int mt, rest;
    q2_tile_of(lid, n_mt, nwg / n_mt, mt, rest);
    const int split = rest % splits, ct = rest / splits;
    const int nsb = K >> 8;
    const int sb0 = split * sbps, nv = min(sbps, nsb - sb0);
    if (nv <= 0) return;  // whole workgroup
    const int m_base = mt * BM;
    const int ngrp = N >> 5;
    const int g = ct * GW + gw;  // groups past N decode the last (never stored)

    const char* wg = (const char*)W + ((size_t)min(g, ngrp - 1) * nsb + sb0) * F::UNIT;

    // A staging: piece p of this thread is 16 B number `threadIdx.x + p NT` of the super-block's [BM][512 B]
    const uint16_t* ap[AP];
    uint32_t aw[AP];
#pragma unroll
    for (int p = 0; p < AP; ++p) {
        const int id = threadIdx.x + p * G::NT, row = id >> 5, c = id & 31;
        ap[p] = A + (size_t)min(m_base + row, M - 1) * lda + sb0 * 256 + c * 8;
        aw[p] = (uint32_t)(row * QR_PITCH + c * 16);
    }

    f32x16 acc[WM];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = 0.f;

    auto mainloop = [&](auto q0_c) {
        constexpr int Q0 = decltype(q0_c)::value;  // the wave's quarters of a super-block: Q0 .. Q0 + NQ - 1
        u32x4 ra[2][AP];
        Q2B<QT> b[2][NQ];
        auto load = [&](int t, int u) {  // super-block t's rows and weights into register set u
#pragma unroll
            for (int p = 0; p < AP; ++p) ra[u][p] = *(const u32x4*)(ap[p] + t * 256);
            const char* unit = wg + (size_t)t * F::UNIT;
            if constexpr (QT == MXQ_Q5_K) b[u][0].load_hdr(unit, unit + F::QH, col, h);  // (a header in two places)
            else b[u][0].load_hdr(unit, col, h);
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                if (q > 0) b[u][q] = b[u][0];
                b[u][q].load_q(unit + F::qoff(Q0 + q), col, h);
            }
        };
        auto store = [&](int t, int u) {
            char* d = smem + (t & 1) * G::SLOT;
#pragma unroll
            for (int p = 0; p < AP; ++p) *(u32x4*)(d + aw[p]) = ra[u][p];
        };
        auto barrier = [&] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (u < nv) load(u, u);
        store(0, 0);
        barrier();
        const uint32_t a_rd = (uint32_t)(col * QR_PITCH + Q0 * 128 + 16 * h);
        // super-block t: products from LDS slot t & 1 and register set u, then the loads of t + 2 and the rows of t + 1 into
        // the other slot, which every wave was done with at the last barrier
        for (int t0 = 0; t0 < nv; t0 += 2) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int t = t0 + u;
                if (t < nv) {
                    const char* as = smem + (t & 1) * G::SLOT + a_rd;
                    auto quarter = [&](auto q_c) {
                        constexpr int q = decltype(q_c)::value, JQ = Q0 + q;
                        auto step = [&](auto s_c) {
                            constexpr int S = decltype(s_c)::value;
                            f16x8 af[WM];
#pragma unroll
                            for (int i = 0; i < WM; ++i)
                                af[i] = *(const f16x8*)(as + i * 32 * QR_PITCH + q * 128 + S * 32);
                            const f16x8 bf = b[u][q].template frag<JQ, S>();
#pragma unroll
                            for (int i = 0; i < WM; ++i)
                                acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], bf, acc[i], 0, 0, 0);
                        };
                        step(std::integral_constant<int, 0>{});
                        step(std::integral_constant<int, 1>{});
                        step(std::integral_constant<int, 2>{});
                        step(std::integral_constant<int, 3>{});
                    };
                    quarter(std::integral_constant<int, 0>{});
                    if constexpr (NQ > 1) quarter(std::integral_constant<int, 1>{});
                    if (t + 2 < nv) load(t + 2, u);
                    if (t + 1 < nv) store(t + 1, u ^ 1);
                    barrier();
                }
            }
        }
    };
    if constexpr (KW == 2) {
        if (kw == 0) mainloop(std::integral_constant<int, 0>{});
        else mainloop(std::integral_constant<int, 2>{});
    } else {
        if (kw == 0) mainloop(std::integral_constant<int, 0>{});
        else if (kw == 1) mainloop(std::integral_constant<int, 1>{});
        else if (kw == 2) mainloop(std::integral_constant<int, 2>{});
        else mainloop(std::integral_constant<int, 3>{});
    }

    // ---- sum over the KW waves of a group, a 32-row block at a time; wave kw keeps accumulator registers kw NR .. ----
    // 32x32 C/D layout: col = lane & 31, row = 8 (r >> 2) + 4 (lane >> 5) + (r & 3)
    constexpr int NR = 16 / KW;
#pragma unroll
    for (int i = 0; i < WM; ++i) {
        if (m_base + i * 32 >= M) break;  // (uniform)
        float v[NR];
        float* red = (float*)smem;
#pragma unroll
        for (int r = 0; r < 16; ++r) red[((kw * GW + gw) * 16 + r) * 64 + lane] = acc[i][r];
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            v[r] = 0.f;
#pragma unroll
            for (int k = 0; k < KW; ++k) v[r] += red[((k * GW + gw) * 16 + kw * NR + r) * 64 + lane];
        }
        if (i + 1 < WM) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const int nt = g * 32, n = nt + col;
        if (nt >= N) continue;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int rr = kw * NR + r;
            const int m = m_base + i * 32 + 8 * (rr >> 2) + 4 * h + (rr & 3);
            if constexpr (EPI == E16_SWIGLU || EPI == E16_GEGLU) {
                // W rows interleaved in 16-row groups: columns 0..15 gate, 16..31 up of the same features
                const float up = __shfl_xor(v[r], 16);
                if (col < 16 && m < M)
                    ((uint16_t*)Cv)[(size_t)m * ldc + (nt >> 1) + col] = f32_to_act<true>(glu_gate_f<EPI>(v[r]) * up);
            } else if (m < M) {
                float* cf = (float*)Cv + (size_t)m * ldc + n;
                if constexpr (EPI == E16_F32) *cf = v[r];
                else if constexpr (EPI == E16_ACT) ((uint16_t*)Cv)[(size_t)m * ldc + n] = f32_to_act<true>(v[r]);
                else if (splits == 1) *cf += v[r];
                else atomicAdd(cf, v[r]);
            }
        }
    }
}

template <int QT, int WM, int GW, int KW, int EPI>
__global__ __launch_bounds__(64 * GW * KW) void qmmr_kernel(const uint16_t* __restrict__ A, int lda, const uint8_t* __restrict__ W, int M, int N,
                                                            int K, int n_mt, int splits, int sbps, void* __restrict__ Cv, int ldc) {
    qmmr_body<QT, WM, GW, KW, EPI>(gridDim.x, blockIdx.x, A, lda, W, M, N, K, n_mt, splits, sbps, Cv, ldc);
}

template <int QT, int WM, int GW, int KW, int EPI>
static int launch_qmmr(const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc,
                       hipStream_t st) {
    using G = QrGeom<WM, GW, KW>;
    const int nsb = K >> 8;
    splits = max(1, min(splits, nsb));
    const int sbps = (nsb + splits - 1) / splits;
    splits = (nsb + sbps - 1) / sbps;  // no empty splits
    const int n_ct = (N + 32 * GW - 1) / (32 * GW), n_mt = (M + G::BM - 1) / G::BM;
    const long nwg = (long)n_ct * splits * n_mt;
    if (nwg <= 0 || nwg > 0x7fffffff) return (int)hipErrorInvalidValue;
    static bool attr_set = false;
    if (!attr_set) {
        (void)hipFuncSetAttribute((const void*)qmmr_kernel<QT, WM, GW, KW, EPI>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS);
        attr_set = true;
    }
    qmmr_kernel<QT, WM, GW, KW, EPI><<<dim3((unsigned)nwg), G::NT, G::LDS, st>>>(A, lda, W, M, N, K, n_mt, splits,
                                                                                       sbps, C, ldc);
    MXK_CHECK_LAUNCH();
}

// (wm, gw, kw) compiled: 32-row tiles of 1, 2 or 4 column groups by 2 or 4 waves over a super-block, 64-row ones
template <int QT, int EPI>
static int dispatch_qmmr(int wm, int gw, int kw, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K,
                         int splits, void* C, int ldc, hipStream_t st) {
#define QR_CASE(WM_, GW_, KW_)                     \
    if (wm == WM_ && gw == GW_ && kw == KW_)       \
        return launch_qmmr<QT, WM_, GW_, KW_, EPI>(A, lda, W, M, N, K, splits, C, ldc, st);
    QR_CASE(1, 4, 4) QR_CASE(1, 2, 4) QR_CASE(1, 1, 4) QR_CASE(1, 4, 2) QR_CASE(1, 2, 2) QR_CASE(2, 2, 4) QR_CASE(2, 4, 2)
#undef QR_CASE
    return (int)hipErrorInvalidValue;
}

// all epilogues of one block format (each format's instances live in their own translation unit, qmmr_q*.hip)
template <int QT>
static int qmmr_run(int epi, int wm, int gw, int kw, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st) {
    switch (epi) {
        case E16_F32: return dispatch_qmmr<QT, E16_F32>(wm, gw, kw, A, lda, W, M, N, K, splits, C, ldc, st);
        case E16_ACT: return dispatch_qmmr<QT, E16_ACT>(wm, gw, kw, A, lda, W, M, N, K, splits, C, ldc, st);
        case E16_ADD_F32: return dispatch_qmmr<QT, E16_ADD_F32>(wm, gw, kw, A, lda, W, M, N, K, splits, C, ldc, st);
        case E16_SWIGLU: return dispatch_qmmr<QT, E16_SWIGLU>(wm, gw, kw, A, lda, W, M, N, K, splits, C, ldc, st);
        case E16_GEGLU: return dispatch_qmmr<QT, E16_GEGLU>(wm, gw, kw, A, lda, W, M, N, K, splits, C, ldc, st);
    }
    return (int)hipErrorInvalidValue;
}

}  // namespace

int qmmr_run_q4k(int epi, int wm, int gw, int kw, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st);
int qmmr_run_q5k(int epi, int wm, int gw, int kw, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st);
int qmmr_run_q6k(int epi, int wm, int gw, int kw, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st);
int qmmr_run_q3k(int epi, int wm, int gw, int kw, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st);
int qmmr_run_q2k(int epi, int wm, int gw, int kw, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st);
int qmmr_run_q80(int epi, int wm, int gw, int kw, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st);
int qmmr_run_mx4(int epi, int wm, int gw, int kw, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st);
int qmmr_run_mx5(int epi, int wm, int gw, int kw, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st);
