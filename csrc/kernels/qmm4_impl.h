// qmm4_impl.h — kernel template of qmm4.hip (see there), shared by the per-format translation units.
#pragma once
#include "qmm2_impl.h"

namespace {

// NI: 16-row blocks; the tile is 16 NI rows x 256 columns (8 groups)
template <int QT, int NI>
struct Q4Geom {
    using F = Q2F<QT>;
    static constexpr int NS = 4, NG = 8;               // ring slots (k-tiles of 64), column groups = waves
    static constexpr int BM = 16 * NI;
    static constexpr int A_BYTES = BM * 128;
    static constexpr int STAGE = A_BYTES + NG * F::QB;
    static constexpr int HSZ = NG * F::HB;              // a super-block's headers, two slots
    static constexpr int LDS = NS * STAGE + 2 * HSZ;
    static constexpr int WA = (2 * NI + 7) / 8;          // A LDS-DMA instructions of a wave a stage (spare ones re-load the last block)
};

// splits > 1 (fp32 out alone): sbps super-blocks of K a workgroup, the sums of part p to Cv [p][M][ldc]
template <int QT, int NI, int EPI>
__global__ __launch_bounds__(512) void qmm4_kernel(const uint16_t* __restrict__ A, int lda, const uint8_t* __restrict__ W,
                                                   int M, int N, int K, int n_mt, int splits, int sbps, void* __restrict__ Cv, int ldc) {
    using G = Q4Geom<QT, NI>;
    using F = Q2F<QT>;
    using B = Q2B<QT, 32>;
    constexpr int NS = G::NS, NG = G::NG, BM = G::BM, WA = G::WA, STAGE = G::STAGE, A_BYTES = G::A_BYTES;
    // A fragments read ahead, in registers i % R of the row blocks counted over a super-block's eight steps: eight row blocks of two
    // waves are 512 cycles, and a whole step's fragments leave 13 and 14 row blocks' accumulators too little room
    constexpr int R = 8;
    static_assert(NI >= R, "a step's first fragments are read in the step before");
    static_assert(G::LDS <= 160 * 1024, "LDS");
    static_assert((NS - 2) * (WA + F::QI + F::HI) <= 63, "vmcnt range");
    extern __shared__ __attribute__((aligned(16))) char smem[];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int c = lane & 15, g = lane >> 4;  // column (row) and k share of a 16x16x32 fragment

    // XCD-aware bijective remap: consecutive logical ids (q2_tile_of) run on one XCD and share its L2
    const int nwg = gridDim.x, bid = blockIdx.x;
    const int xcd = bid & 7, q8 = nwg >> 3, r8 = nwg & 7;
    int lid = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + (bid >> 3);
    int mt, ct, tiles = nwg, nsb = K >> 8, sb0 = 0;
    const size_t col_bytes = (size_t)nsb * F::UNIT;  // of a column group
    if constexpr (EPI == E16_F32) {
        // the tiles of a part of K follow one another: they read the same k of A, and its L2 holds that
        tiles = nwg / splits;
        const int p = lid / tiles;
        lid -= p * tiles;
        sb0 = p * sbps;
        nsb = min(sbps, nsb - sb0);
        Cv = (float*)Cv + (size_t)p * M * ldc;
    }
    q2_tile_of(lid, n_mt, tiles / n_mt, mt, ct);
    const int m_base = mt * BM, ngrp = N >> 5;
    // (groups past N re-read the last, never stored)
    const uint8_t* wg = W + (size_t)min(ct * NG + wave, ngrp - 1) * col_bytes + (size_t)sb0 * F::UNIT;
    A += (size_t)sb0 * 256;

    // A LDS-DMA sources and image as qmm2's: 8-row block j, lane p writes image slot (16-k step p >> 4, row (p >> 1) & 7, half
    // (p & 1) ^ (j & 1)) from 16 B of that row
    uint32_t aoff[WA];
#pragma unroll
    for (int i = 0; i < WA; ++i) {
        const int j = min(wave * WA + i, BM / 8 - 1);
        const int s = lane >> 4, r = (lane >> 1) & 7, hh = (lane & 1) ^ (j & 1);
        aoff[i] = 2 * (uint32_t)(min(m_base + 8 * j + r, M - 1) * lda + 16 * s + 8 * hh);
    }
    // fragment reads: row block i of 16 at + 2048 i, k-step T of 32 at + 512 T; the lane's k are Q2B's of MK 32
    const uint32_t a_rd = (uint32_t)((c >> 3) * 1024 + (g & 1) * 256 + (c & 7) * 32 + (((g >> 1) ^ (c >> 3)) << 4));
    const uint32_t b_rd = (uint32_t)(A_BYTES + wave * F::QB), h_rd = (uint32_t)(NS * STAGE + wave * F::HB);

    const uint32_t ring = mx_lds_addr(smem), hring = ring + NS * STAGE;
    struct Stage {
        const uint16_t* a;
        const uint8_t* u;
        uint32_t lds, hd;
    };
    // stage ki (ki & 3 == its ring slot); past the end the last k-tile's rows and super-block's weights again, never consumed
    auto stage = [&](int ki, int slot) {
        const int vi = ki >> 2;
        Stage st;
        st.a = A + (size_t)(uint32_t)min(ki, nsb * 4 - 1) * 64;
        st.u = wg + (size_t)(uint32_t)min(vi, nsb - 1) * F::UNIT;
        st.lds = ring + slot * STAGE;
        st.hd = hring + (vi & 1) * G::HSZ;
        return st;
    };
    constexpr int ND = WA + 1;  // pieces of a stage's issue: an A instruction each, then the weights'
    auto issue = [&](const Stage& st, auto d_c, auto jq_c) {
        constexpr int D = decltype(d_c)::value, JQ = decltype(jq_c)::value;
        if constexpr (D < WA) mx_lds_dma16(st.a, aoff[D], st.lds + min(wave * WA + D, BM / 8 - 1) * 1024);
        else q2_stage_weights<QT, JQ>(st.u, st.lds + A_BYTES + wave * F::QB, st.hd + wave * F::HB, lane);
    };

    // the products are computed transposed (weights first), so that a lane ends with four columns of one row and stores them at once
    f32x4 acc[NI][2];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

    q2_static_for<0, NS - 1>([&](auto k_c) {
        constexpr int k = decltype(k_c)::value;
        const Stage st = stage(k, k);
        q2_static_for<0, ND>([&](auto d_c) { issue(st, d_c, k_c); });
    });
    q2_wait_barrier<q2_cnt_run<WA, F::QI, F::HI, true, 1, NS - 2>()>();

    B bw[2];
    f16x8 af[R], bf[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        bw[j].load_hdr(smem + h_rd, c + 16 * j, g);
        bw[j].load_q(smem + b_rd, c + 16 * j, g);
        bf[j] = bw[j].template frag<0, 0>();
    }
#pragma unroll
    for (int i = 0; i < R; ++i) af[i] = *(const f16x8*)(smem + a_rd + i * 2048);

    // one k-tile (ring slot JQ), two k-steps, pipelined as qmm2's: a step's products consume fragments read and dequantised before,
    // while the next step's are read and dequantised and a stage is issued, piece by piece in the source's order
    auto tile = [&](int sb, auto jq_c) {
        constexpr int JQ = decltype(jq_c)::value, NJ = (JQ + 1) & 3, IJ = (JQ + 3) & 3;
        // stage kt + 1 landed (kt + 2 may still be in flight); every wave is past tile kt - 1
        q2_wait_barrier<q2_cnt_run<WA, F::QI, F::HI, true, (JQ + 2) & 3, NS - 3>()>();
        const Stage st = stage(sb * 4 + JQ + 3, IJ);
        B bn[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            bn[j] = bw[j];
            if constexpr (NJ == 0) bn[j].load_hdr(smem + h_rd + ((sb + 1) & 1) * G::HSZ, c + 16 * j, g);
            bn[j].load_q(smem + NJ * STAGE + b_rd, c + 16 * j, g);
        }
        q2_static_for<0, 2>([&](auto t_c) {
            constexpr int T = decltype(t_c)::value, TN = T ^ 1, JN = T ? NJ : JQ;  // TN, JN: the fragments made here
            const char* const ac = smem + JQ * STAGE + a_rd + T * 512;
            const char* const an = smem + JN * STAGE + a_rd + TN * 512;
            u32x4 bfn[2];
            auto piece = [&](auto u_c) {
                constexpr int j = decltype(u_c)::value / 3, u = decltype(u_c)::value % 3;
                B& w = T ? bn[j] : bw[j];
                if constexpr (u == 0) {
                    w.template prep<JN, TN>();
                } else {
                    const u32x2 x = w.template half<JN, TN, u - 1>();
                    bfn[j][2 * (u - 1)] = x[0];
                    bfn[j][2 * (u - 1) + 1] = x[1];
                }
            };
            constexpr int A0 = (2 * JQ + T) * NI, NP = 6, D0 = T ? (ND + 1) / 2 : 0, D1 = T ? ND : (ND + 1) / 2;
            __builtin_amdgcn_sched_barrier(0);
            q2_static_for<0, NI>([&](auto i_c) {
                constexpr int i = decltype(i_c)::value;
                acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[0], af[(A0 + i) % R], acc[i][0], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                q2_static_for<i * NP / NI, (i + 1) * NP / NI>(piece);
                q2_static_for<D0 + (D1 - D0) * i / NI, D0 + (D1 - D0) * (i + 1) / NI>(
                    [&](auto d_c) { issue(st, d_c, std::integral_constant<int, IJ>{}); });
                __builtin_amdgcn_sched_barrier(0);
                acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[1], af[(A0 + i) % R], acc[i][1], 0, 0, 0);
                af[(A0 + i) % R] = *(const f16x8*)(i + R < NI ? ac + (i + R) * 2048 : an + (i + R - NI) * 2048);
                __builtin_amdgcn_sched_barrier(0);
            });
#pragma unroll
            for (int j = 0; j < 2; ++j) bf[j] = __builtin_bit_cast(f16x8, bfn[j]);
        });
#pragma unroll
        for (int j = 0; j < 2; ++j) bw[j] = bn[j];
    };
    for (int sb = 0; sb < nsb; ++sb) q2_static_for<0, 4>([&](auto jq_c) { tile(sb, jq_c); });
    // the dummy stages land before the LDS is released
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    // ---- epilogue: block (i, j) is rows m_base + 16 i .., columns n0 + 16 j ..; a lane has row c, columns 4 g .. 4 g + 3 ----
    const int n0 = (ct * NG + wave) * 32;
    if (n0 >= N) return;
    // four columns at once where C allows: 16 bytes of fp32, 8 of f16
    constexpr int ES = EPI == E16_F32 ? 4 : 2;
    const bool vec = !(((uintptr_t)Cv & (4 * ES - 1)) | (ldc & 3));
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        if (m_base + i * 16 >= M) break;
        const int m = m_base + i * 16 + c;
        if (m >= M) continue;
        if constexpr (EPI == E16_F32) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                float* const p = (float*)Cv + (size_t)m * ldc + n0 + j * 16 + 4 * g;
                if (vec) {
                    *(f32x4*)p = acc[i][j];
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) p[r] = acc[i][j][r];
                }
            }
        } else {
            // gated: W rows interleaved in 16-row groups, a lane holds gate (j 0) and up (j 1) of the same four features
            constexpr bool GLU = EPI == E16_SWIGLU || EPI == E16_GEGLU;
#pragma unroll
            for (int j = 0; j < (GLU ? 1 : 2); ++j) {
                uint16_t o[4], *const p = (uint16_t*)Cv + (size_t)m * ldc + (GLU ? n0 >> 1 : n0 + j * 16) + 4 * g;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if constexpr (GLU) o[r] = f32_to_act<true>(glu_gate_f<EPI>(acc[i][0][r]) * acc[i][1][r]);
                    else o[r] = f32_to_act<true>(acc[i][j][r]);
                }
                if (vec) {
                    *(uint2*)p = make_uint2(o[0] | (uint32_t)o[1] << 16, o[2] | (uint32_t)o[3] << 16);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) p[r] = o[r];
                }
            }
        }
    }
}

// super-blocks of K in each of `splits` parts (the last one may have fewer; none is empty)
static int qmm4_part_blocks(int K, int splits) { return ((K >> 8) + splits - 1) / splits; }

template <int QT, int NI, int EPI>
static int launch_qmm4(const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st) {
    using G = Q4Geom<QT, NI>;
    const int n_ct = (N + 255) / 256, n_mt = (M + G::BM - 1) / G::BM, sbps = qmm4_part_blocks(K, splits);
    splits = ((K >> 8) + sbps - 1) / sbps;
    const long nwg = (long)n_ct * n_mt * splits;
    if (nwg <= 0 || nwg > 0x7fffffff) return (int)hipErrorInvalidValue;
    static bool attr_set = false;
    if (!attr_set) {
        (void)hipFuncSetAttribute((const void*)qmm4_kernel<QT, NI, EPI>, hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS);
        attr_set = true;
    }
    qmm4_kernel<QT, NI, EPI><<<dim3((unsigned)nwg), 512, G::LDS, st>>>(A, lda, W, M, N, K, n_mt, splits, sbps, C, ldc);
    MXK_CHECK_LAUNCH();
}

template <int QT>
constexpr int qmm4_max_ni() {  // largest tile whose ring fits the LDS
    return Q4Geom<QT, 14>::LDS <= 160 * 1024 ? 14 : Q4Geom<QT, 13>::LDS <= 160 * 1024 ? 13 : Q4Geom<QT, 12>::LDS <= 160 * 1024 ? 12 : 11;
}

// `nb`: 16-row blocks a tile may have, 8 .. 14. The fewest row tiles that hold M rows, as even as blocks allow: 416 rows run as 2 x 208,
// 333 as 2 x 176. (The formats of few checkpoints have tiles of an even number of blocks alone, to halve what is compiled.)
template <int QT, int EPI>
static int dispatch_qmm4(int nb, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st) {
    constexpr int MAX = qmm4_max_ni<QT>();
    constexpr bool ODD = QT == MXQ_Q4_K || QT == MXQ_Q5_K || QT == MXQ_Q6_K || QT == MXQ_Q8_0;
    static_assert(Q4Geom<QT, MAX>::LDS <= 160 * 1024, "LDS");
    nb = max(8, min(nb, ODD ? MAX : MAX & ~1));
    const int blocks = (M + 15) / 16, tiles = (blocks + nb - 1) / nb, ni = (blocks + tiles - 1) / tiles;
#define Q4_CASE(NI_)                                                                                  \
    if constexpr (NI_ <= MAX && (ODD || NI_ % 2 == 0))                                                \
        if (ni <= NI_) return launch_qmm4<QT, NI_, EPI>(A, lda, W, M, N, K, splits, C, ldc, st);
    Q4_CASE(8) Q4_CASE(9) Q4_CASE(10) Q4_CASE(11) Q4_CASE(12) Q4_CASE(13) Q4_CASE(14)
#undef Q4_CASE
    return (int)hipErrorInvalidValue;
}

// the epilogues of one block format (each format's instances live in their own translation unit, qmm4_q*.hip)
template <int QT>
static int qmm4_run(int epi, int nb, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st) {
    switch (epi) {
        case E16_F32: return dispatch_qmm4<QT, E16_F32>(nb, A, lda, W, M, N, K, splits, C, ldc, st);
        case E16_ACT: return dispatch_qmm4<QT, E16_ACT>(nb, A, lda, W, M, N, K, splits, C, ldc, st);
        case E16_SWIGLU: return dispatch_qmm4<QT, E16_SWIGLU>(nb, A, lda, W, M, N, K, splits, C, ldc, st);
        case E16_GEGLU: return dispatch_qmm4<QT, E16_GEGLU>(nb, A, lda, W, M, N, K, splits, C, ldc, st);
    }
    return (int)hipErrorInvalidValue;
}

}  // namespace

int qmm4_run_q4k(int epi, int nb, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st);
int qmm4_run_q5k(int epi, int nb, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st);
int qmm4_run_q6k(int epi, int nb, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st);
int qmm4_run_q3k(int epi, int nb, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st);
int qmm4_run_q2k(int epi, int nb, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st);
int qmm4_run_q80(int epi, int nb, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st);
int qmm4_run_mx4(int epi, int nb, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st);
int qmm4_run_mx5(int epi, int nb, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st);
