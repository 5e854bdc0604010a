// dense16_impl.h — products of a 16-bit matrix's rows with 16-bit weights: the kernel of dense16.hip (what it is for and its times stand
// there) over g16_tile's tiles. Tiles whose K is split over workgroups leave their sums in `part`; dense16_sum_kernel adds them in order.
#pragma once
#include "dense16.h"
#include "gemm16_impl.h"

namespace {

struct D16Args {
    const uint16_t *A, *B;
    int lda, ldb, M, N, nk;  // N: columns of C; nk 64-wide k-tiles
    int n_mt, n_nt;          // tiles of C
    int full, parts;         // tiles from `full` on are summed in `parts` parts of K
    float* part;             // [tile - full][part][TM][TN], or with part_rows [part][M][N]
    const float* bias;       // of C's columns, or null
    float* C;
    int ldc;
    // gated columns (D16_GLU): G[m, f] = silu(A · B[gate0 + f] + gate_b[f]) (A · B[up0 + f] + up_b[f]) in 16 bits, beside C
    int g_nt, F, gate0, up0;
    const float *gate_b, *up_b;
    uint16_t* G;
    int ldg;
    // 16-bit outputs (D16_ACT, D16_GELU: gelu of the sum, erf form) instead of C, with a 16-bit bias or null
    uint16_t* Y;
    const uint16_t* bias16;
    int part_rows;
};

template <int EPI, bool F16, int MI, int NJ>
__global__ __launch_bounds__(256, 1) void dense16_kernel(D16Args a) {
    using T = G16T<MI, NJ>;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int bid = blockIdx.x;
    int tile = g16_lid(bid, gridDim.x), p = 0, np = 1;
    if constexpr (EPI == D16_PART) {
        np = a.parts;
        p = tile % np;
        tile = a.full + tile / np;
    }
    const int gt = EPI == D16_GLU || EPI == D16_PART ? a.n_mt * a.g_nt : 0;
    const bool glu = EPI == D16_GLU && tile < gt;
    int mt, nt;
    q2_tile_of(glu ? tile : tile - gt, a.n_mt, glu ? a.g_nt : a.n_nt, mt, nt);
    const int m_base = mt * T::TM, n_base = nt * T::TN;
    const int k0 = (int)((long)a.nk * p / np), k1 = (int)((long)a.nk * (p + 1) / np);
    const char* ab = (const char*)(a.A + (size_t)m_base * a.lda) + (size_t)k0 * 128;
    const char* bb = (const char*)(a.B + (glu ? (size_t)0 : (size_t)n_base * a.ldb)) + (size_t)k0 * 128;
    f32x4 acc[MI][NJ];
    // up to 64 rows workgroups start at different k-tiles: in step, all of them read the same few channels of memory (40992 x 4096, 33 rows 74.4
    // -> 67.3 us, 64 rows 78 -> 72.8; more rows lose, since row tiles of the same columns then meet in no cache: 1990 rows 572 -> 600)
    constexpr bool ROT = MI <= 2 && EPI != D16_PART;
    g16_tile<F16, MI, NJ, ROT>(
        smem, ab, bb, k1 - k0, [&](int r) { return (uint32_t)min(r, a.M - 1 - m_base) * (uint32_t)(2 * a.lda); },
        [&](int r) {
            // gated: rows in 16-row groups, an even one gates and the next one the ups of the same features; two such pairs share 32 features
            // so that a lane ends with eight in a row
            if (EPI == D16_GLU && glu) {
                const int f = NJ % 4 ? (r >> 5) * 16 + (r & 15) : (r >> 6) * 32 + ((r & 12) << 1) + ((r >> 3) & 4) + (r & 3);
                return (uint32_t)((r & 16 ? a.up0 : a.gate0) + min(nt * (T::TN / 2) + f, a.F - 1)) * (uint32_t)(2 * a.ldb);
            }
            // 16-bit outputs: neighbouring 16-column tiles share 32 columns so that a lane ends with eight in a row
            if (EPI == D16_ACT || EPI == D16_GELU) r = (r & ~31) + ((r & 12) << 1) + ((r >> 2) & 4) + (r & 3);
            return (uint32_t)min(r, a.N - 1 - n_base) * (uint32_t)(2 * a.ldb);
        },
        acc, ROT ? (int)(bid * 17u % (unsigned)(k1 - k0)) : 0);

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int el = threadIdx.x & 63;
    asm volatile("" : "+v"(el));  // (no address of it computed ahead of the loop, whose registers are all taken)
    const int eg = el >> 4, wm = wave >> 1, wn = wave & 1;
    const int m0 = m_base + wm * (16 * MI) + (el & 15), n0 = n_base + wn * (16 * NJ) + 4 * eg;
    if constexpr (EPI == D16_GLU) {
        if (glu) {
            constexpr int FL = NJ % 4 ? 4 : 8, NQ = NJ * 2 / FL;  // features of a lane's piece, pieces
            static_assert(NJ % 2 == 0, "gates and ups in pairs of tiles");
            const int f0 = nt * (T::TN / 2) + wn * (8 * NJ) + FL * eg;
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const int f = f0 + 4 * FL * q;
                float gb[FL], ub[FL];
#pragma unroll
                for (int e = 0; e < FL; e += 4) {
                    const int fc = min(f + e, a.F - 4);
                    *(f32x4*)(gb + e) = a.gate_b ? *(const f32x4*)(a.gate_b + fc) : (f32x4){0.f, 0.f, 0.f, 0.f};
                    *(f32x4*)(ub + e) = a.up_b ? *(const f32x4*)(a.up_b + fc) : (f32x4){0.f, 0.f, 0.f, 0.f};
                }
#pragma unroll
                for (int i = 0; i < MI; ++i) {
                    uint32_t w[FL / 2];
                    float v[FL];
#pragma unroll
                    for (int e = 0; e < FL; ++e) {
                        const int j = q * (FL / 2) + (e >> 2) * 2;
                        v[e] = silu_gate_f(acc[i][j][e & 3] + gb[e]) * (acc[i][j + 1][e & 3] + ub[e]);
                    }
#pragma unroll
                    for (int e = 0; e < FL; e += 2) w[e / 2] = pack_act2<F16>(v[e], v[e + 1]);
                    uint16_t* g = a.G + (size_t)(m0 + 16 * i) * a.ldg + f;
                    if (m0 + 16 * i < a.M && f < a.F) {
                        if constexpr (FL == 8) *(u32x4*)g = (u32x4){w[0], w[1], w[2], w[3]};
                        else *(u32x2*)g = (u32x2){w[0], w[1]};
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            return;
        }
    }
    if constexpr (EPI == D16_ACT || EPI == D16_GELU) {
        const int n1 = n_base + wn * (16 * NJ) + 8 * eg;  // a lane's eight columns of a pair of 16-column tiles
        u32x4 b[NJ / 2];
#pragma unroll
        for (int q = 0; q < NJ / 2; ++q) b[q] = a.bias16 ? *(const u32x4*)(a.bias16 + min(n1 + 32 * q, a.N - 8)) : (u32x4){0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
            for (int q = 0; q < NJ / 2; ++q) {
                float v[8];
                u32x4 w;
#pragma unroll
                for (int e = 0; e < 4; ++e) unpack_act2<F16>(b[q][e], v[2 * e], v[2 * e + 1]);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    v[e] += acc[i][2 * q + (e >> 2)][e & 3];
                    if constexpr (EPI == D16_GELU) v[e] = gelu_erf_f(v[e]);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) w[e] = pack_act2<F16>(v[2 * e], v[2 * e + 1]);
                if (m0 + 16 * i < a.M && n1 + 32 * q < a.N) *(u32x4*)(a.Y + (size_t)(m0 + 16 * i) * a.ldc + n1 + 32 * q) = w;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        return;
    }
    // fp32 rows, or a part's sums
    float* C = a.C;
    int ldc = a.ldc;
    if constexpr (EPI == D16_PART) {
        C = a.part_rows ? a.part + (size_t)p * a.M * a.N : a.part + ((size_t)(tile - a.full) * np + p) * (T::TM * T::TN) - ((size_t)m_base * T::TN + n_base);
        ldc = a.part_rows ? a.N : T::TN;
    }
    f32x4 b[NJ], old[2][NJ];
    if constexpr (EPI != D16_PART)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            b[j] = a.bias ? *(const f32x4*)(a.bias + min(n0 + 16 * j, a.N - 4)) : (f32x4){0.f, 0.f, 0.f, 0.f};
    auto load = [&](int i) {
#pragma unroll
        for (int j = 0; j < NJ; ++j)  // (past M / N: the last ones)
            old[i & 1][j] = *(const f32x4*)(C + (size_t)min(m0 + 16 * i, a.M - 1) * ldc + min(n0 + 16 * j, a.N - 4));
    };
    if constexpr (EPI == D16_ADD) load(0);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        if constexpr (EPI == D16_ADD)
            if (i < MI - 1) load(i + 1);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            f32x4 v = acc[i][j];
            asm volatile("" : "+v"(v));  // (stored from there: from where they are, the loop spills)
            if constexpr (EPI != D16_PART) v += b[j];
            if constexpr (EPI == D16_ADD) v += old[i & 1][j];
            if (m0 + 16 * i < a.M && n0 + 16 * j < a.N) *(f32x4*)(C + (size_t)(m0 + 16 * i) * ldc + n0 + 16 * j) = v;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

#define D16_TILES(GO) GO(8, 8) GO(7, 8) GO(6, 8) GO(5, 8) GO(8, 6) GO(6, 6) GO(8, 4) GO(5, 4) GO(4, 4) GO(2, 8) GO(2, 4)

template <int EPI, bool F16, int MI, int NJ>
void dense16_launch(const D16Args& a, unsigned n, hipStream_t st) {
    using T = G16T<MI, NJ>;
    static const hipError_t attr = hipFuncSetAttribute((const void*)dense16_kernel<EPI, F16, MI, NJ>, hipFuncAttributeMaxDynamicSharedMemorySize, T::LDS);
    (void)attr;
    dense16_kernel<EPI, F16, MI, NJ><<<dim3(n), 256, T::LDS, st>>>(a);
}

}  // namespace

// n workgroups of the gated kernel (dense16_glu.hip); tile 16 MI + NJ
void mx_dense16_glu(const void* args, int tile, unsigned n, hipStream_t st);
