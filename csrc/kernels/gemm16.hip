// gemm16.hip — prompts of thousands of rows by quantised weights: the weights are expanded to f16 once (t32_expand) and multiplied by
// a plain f16 GEMM.
//
//   C[M, N] (+)= A[M, K] · B[N, K]^T,   A, B f16, fp32 sums; epilogues as qmm2.hip
//
// qmm2's tiles decode the weights of their columns for themselves: beyond some 2000 rows that is done 10 to 40 times over, beside
// products that want every issue slot (gate|up 28672 x 4096 at 8191 rows: 1750 to 1850 us, 1.04 to 1.1 PFLOP/s). Expanding them
// first moves 2.6 bytes a weight (80 us there) and leaves a GEMM whose inner loop is products, fragment reads and loads:
//   * 256 x 256 tiles, four waves of 128 x 128, one on a SIMD: the sums take all 256 accumulation registers. 16 x 16 x 32 products:
//     32 x 32 x 16 ones of the same tile reach 1.06 PFLOP/s where these reach 1.26 (they write each sum twice as often);
//   * 64-wide k-tiles by LDS-DMA into five 32 KB slots, A and B apart, so that a tile's successor but one is on its way while the
//     next waits in LDS. Deeper rings of 32-wide halves, loads through registers or staggered k order changed nothing;
//   * every product is followed by at most one load or fragment read, and the four waves' loads fall between different products.
//     The address unit takes 16 cycles a load: issued together, all waves queue behind it with their products (1.26 PFLOP/s;
//     spread over the tile 1.34, at different places in each wave 1.40);
//   * the operands are swapped (C^T), so a lane ends with four columns of a row: 16-byte stores, and the residual read a block of
//     16 rows ahead (read just before each store the epilogue of 4096 columns took 110 us of 310, now 15).
// Measured at 8191 rows, us, expansion apart: gate|up 28672 x 4096 with SwiGLU 1370 (1.40 PFLOP/s; the library's product without it
// 1304), 4096 x 14336 with the residual 688, 4096 x 4096 215, 5120 x 4096 275.
#include "gemm16_impl.h"

namespace {

template <int EPI>
__global__ __launch_bounds__(256, 1) void gemm16_kernel(const uint16_t* __restrict__ A, int lda, const uint16_t* __restrict__ B, int ldb,
                                                        int M, int N, int K, int n_mt, void* __restrict__ Cv, int ldc) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int wm = wave >> 1, wn = wave & 1;

    // consecutive logical ids run on one XCD, row tiles in bands (q2_tile_of)
    const int nwg = gridDim.x, lid = g16_lid(blockIdx.x, nwg);
    int mt, nt;
    q2_tile_of(lid, n_mt, nwg / n_mt, mt, nt);
    const int m_base = mt * 256, n_base = nt * 256;
    f32x4 acc[8][8];
    g16_tile<true, 8, 8>(
        smem, (const char*)(A + (size_t)m_base * lda), (const char*)(B + (size_t)n_base * ldb), K / G16_K,
        [&](int r) { return (uint32_t)min(r, M - 1 - m_base) * (uint32_t)(2 * lda); },
        [&](int r) {
            // 16-bit outputs: neighbouring 16-column tiles (gated: pairs of a gate's and an up's) share 32 columns, so that a lane ends
            // with eight in a row; B's rows lie interleaved in 16-row groups, a gate's and the up's of the same features
            if constexpr (EPI == E16_ACT) r = (r & ~31) + ((r & 12) << 1) + ((r >> 2) & 4) + (r & 3);
            if constexpr (EPI == E16_SWIGLU || EPI == E16_GEGLU) {
                const int f = ((r & 12) << 1) + ((r >> 3) & 4) + (r & 3);
                r = (r & ~63) + ((f & 16) << 1) + (r & 16) + (f & 15);
            }
            return (uint32_t)min(r, N - 1 - n_base) * (uint32_t)(2 * ldb);
        },
        acc);

    // ---- epilogue: lane holds columns nb + 4 g .. + 3 of row mb + col; the residual's rows a block ahead of their stores ----
    int el = lane;
    asm volatile("" : "+v"(el));  // (no address of it computed ahead of the loop, whose registers are all taken)
    const int eg = el >> 4, m0 = m_base + wm * 128 + (el & 15), n0 = n_base + wn * 128 + 4 * eg;
    auto put = [&](uint16_t* p, const uint32_t (&w)[4]) {
        if (ldc & 7) {  // (rows 8 bytes apart from 16)
            *(u32x2*)p = (u32x2){w[0], w[1]};
            *(u32x2*)(p + 4) = (u32x2){w[2], w[3]};
        } else {
            *(u32x4*)p = (u32x4){w[0], w[1], w[2], w[3]};
        }
    };
    if constexpr (EPI == E16_SWIGLU || EPI == E16_GEGLU) {
        const int f0 = (n_base >> 1) + wn * 64 + 8 * eg;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (m0 + 16 * i < M)
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    if (f0 + 32 * q >= N >> 1) break;
                    uint32_t v[8], w[4];  // (each rounded once, product and conversion together, as in qmm2; a packed conversion rounds the product first)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const int j = 4 * q + (e >> 2) * 2;
                        v[e] = f32_to_act<true>(glu_gate_f<EPI>(acc[i][j][e & 3]) * acc[i][j + 1][e & 3]);
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) w[e] = v[2 * e] | v[2 * e + 1] << 16;
                    put((uint16_t*)Cv + (size_t)(m0 + 16 * i) * ldc + f0 + 32 * q, w);
                }
    } else if constexpr (EPI == E16_ACT) {
        const int n1 = n_base + wn * 128 + 8 * eg;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (m0 + 16 * i < M)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (n1 + 32 * q >= N) break;
                    uint32_t w[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) w[e] = pack_act2<true>(acc[i][2 * q + (e >> 1)][2 * (e & 1)], acc[i][2 * q + (e >> 1)][2 * (e & 1) + 1]);
                    put((uint16_t*)Cv + (size_t)(m0 + 16 * i) * ldc + n1 + 32 * q, w);
                }
    } else {
        f32x4 old[2][8];
        auto load = [&](int i) {
#pragma unroll
            for (int j = 0; j < 8; ++j)  // (past M / N: the last ones)
                old[i & 1][j] = *(const f32x4*)((const float*)Cv + (size_t)min(m0 + 16 * i, M - 1) * ldc + min(n0 + 16 * j, N - 4));
        };
        if constexpr (EPI == E16_ADD_F32) load(0);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if constexpr (EPI == E16_ADD_F32) {
                if (i < 7) load(i + 1);
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[i][j] += old[i & 1][j];
            }
            if (m0 + 16 * i < M)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    f32x4 v = acc[i][j];
                    asm volatile("" : "+v"(v));  // (stored from there: from where they are, the loop spills)
                    if (n0 + 16 * j < N) *(f32x4*)((float*)Cv + (size_t)(m0 + 16 * i) * ldc + n0 + 16 * j) = v;
                }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

template <int EPI>
int launch_gemm16(const uint16_t* A, int lda, const uint16_t* B, int ldb, int M, int N, int K, void* C, int ldc, hipStream_t st) {
    const int n_mt = (M + 255) / 256;
    const long nwg = (long)n_mt * ((N + 255) / 256);
    if (nwg > 0x7fffffff) return (int)hipErrorInvalidValue;
    static bool attr_set = false;
    if (!attr_set) {
        (void)hipFuncSetAttribute((const void*)gemm16_kernel<EPI>, hipFuncAttributeMaxDynamicSharedMemorySize, G16T<8, 8>::LDS);
        attr_set = true;
    }
    gemm16_kernel<EPI><<<dim3((unsigned)nwg), 256, G16T<8, 8>::LDS, st>>>(A, lda, B, ldb, M, N, K, n_mt, C, ldc);
    MXK_CHECK_LAUNCH();
}

// out[32 g + col][256 sb + ..] = the f16 weights of column group g's super-block sb as the GEMMs decode them (Q2B), a wave each;
// the fragment of k-step s of tile jq is 16 bytes a lane at k 64 jq + 16 s + 8 h. Bound by its stores (2 of 2.6 bytes a weight).
template <int QT>
__global__ __launch_bounds__(256) void t32_expand_kernel(const uint8_t* __restrict__ W, int units, int nsb, uint16_t* __restrict__ out) {
    using F = Q2F<QT>;
    const int unit = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, h = lane >> 5, col = lane & 31;
    if (unit >= units) return;
    const int g = unit / nsb, sb = unit - g * nsb;
    const char* u = (const char*)W + (size_t)unit * F::UNIT;
    uint16_t* o = out + ((size_t)g * 32 + col) * ((size_t)nsb * 256) + sb * 256 + 8 * h;
    Q2B<QT> b[4];
    if constexpr (QT == MXQ_Q5_K) b[0].load_hdr(u, u + F::QH, col, h);  // (a header in two places)
    else b[0].load_hdr(u, col, h);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (q > 0) b[q] = b[0];
        b[q].load_q(u + F::qoff(q), col, h);
    }
    auto tile = [&](auto q_c) {
        constexpr int Q = decltype(q_c)::value;
        *(f16x8*)(o + 64 * Q) = b[Q].template frag<Q, 0>();
        *(f16x8*)(o + 64 * Q + 16) = b[Q].template frag<Q, 1>();
        *(f16x8*)(o + 64 * Q + 32) = b[Q].template frag<Q, 2>();
        *(f16x8*)(o + 64 * Q + 48) = b[Q].template frag<Q, 3>();
    };
    tile(std::integral_constant<int, 0>{});
    tile(std::integral_constant<int, 1>{});
    tile(std::integral_constant<int, 2>{});
    tile(std::integral_constant<int, 3>{});
}

}  // namespace

// t32 weights [N, K] (N % 32 == 0, K % 256 == 0) -> f16 [N, K]
extern "C" int mxk_t32_expand(int qtype, const uint8_t* W, int N, int K, uint16_t* out, hipStream_t st) {
    if (N <= 0 || K <= 0) return 0;
    if (N % 32 || K % 256 || ((uintptr_t)W & 15) || ((uintptr_t)out & 15)) return (int)hipErrorInvalidValue;
    const long units = (long)(N / 32) * (K / 256);
    if (units > 0x7ffffffc) return (int)hipErrorInvalidValue;
#define T32X(QT_) \
    case QT_: t32_expand_kernel<QT_><<<(unsigned)((units + 3) / 4), 256, 0, st>>>(W, (int)units, K / 256, out); break;
    switch (qtype) {
        T32X(MXQ_Q4_K) T32X(MXQ_Q5_K) T32X(MXQ_Q6_K) T32X(MXQ_Q3_K) T32X(MXQ_Q2_K) T32X(MXQ_Q8_0) T32X(MXQ_MX4F) T32X(MXQ_MX5F)
        default: return (int)hipErrorInvalidValue;
    }
#undef T32X
    MXK_CHECK_LAUNCH();
}

// A f16 [M, K], B f16 [N, K], rows 16-byte aligned, K % 64 == 0, N % 32 == 0; C rows of 16-byte (16-bit outputs: 8-byte) aligned
// pieces. epi as mxk_qmm2 (no split).
extern "C" int mxk_gemm16(int epi, const uint16_t* A, int lda, const uint16_t* B, int ldb, int M, int N, int K, void* C, int ldc,
                          hipStream_t st) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || K % G16_K || N % 32 || (lda & 7) || (ldb & 7) || ((uintptr_t)A & 15) || ((uintptr_t)B & 15) || lda < K || ldb < K ||
        lda > (1 << 22) || ldb > (1 << 22) || ((uintptr_t)C & 15) || (ldc & 3))  // (256 rows of 2^23 bytes: the 32-bit lane offsets)
        return (int)hipErrorInvalidValue;
    switch (epi) {
        case E16_F32: return launch_gemm16<E16_F32>(A, lda, B, ldb, M, N, K, C, ldc, st);
        case E16_ACT: return launch_gemm16<E16_ACT>(A, lda, B, ldb, M, N, K, C, ldc, st);
        case E16_ADD_F32: return launch_gemm16<E16_ADD_F32>(A, lda, B, ldb, M, N, K, C, ldc, st);
        case E16_SWIGLU: return launch_gemm16<E16_SWIGLU>(A, lda, B, ldb, M, N, K, C, ldc, st);
        case E16_GEGLU: return launch_gemm16<E16_GEGLU>(A, lda, B, ldb, M, N, K, C, ldc, st);
    }
    return (int)hipErrorInvalidValue;
}
