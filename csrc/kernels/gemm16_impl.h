// gemm16_impl.h — the plain 16-bit GEMM: C[M, N] = A[M, K] · B[N, K]^T, fp32 sums, bf16 or f16 operands, tiles of 32 MI x 32 NJ by
// four waves of 16 MI x 16 NJ, one on a SIMD. What the 256 x 256 tile (MI = NJ = 8) is built from and what each part of it measured
// stands in gemm16.hip; smaller tiles keep its loop, with the loads and fragment reads spread over the fewer products.
#pragma once
#include "qmm2_fmt.h"

namespace {

constexpr int G16_K = 64;  // k of a tile

// LDS: a ring of NS stages, A and B of a k-tile each; where not even three fit (the largest tiles), five slots instead, A of tile t in
// 2 t mod 5 and B in 2 t + 1 mod 5, each as large as the larger of the two. Either way tile t + NS - 1 is asked for while t is multiplied.
template <int MI, int NJ>
struct G16T {
    static constexpr int TM = 32 * MI, TN = 32 * NJ, AB = TM * 128, BB = TN * 128;  // rows of 128 bytes
    static constexpr bool SLOTS = 3 * (AB + BB) > 163840;
    static constexpr int NS = SLOTS ? 3 : 163840 / (AB + BB) > 8 ? 8 : 163840 / (AB + BB);
    static constexpr int SLOT = AB > BB ? AB : BB;
    static constexpr int LDS = SLOTS ? 5 * SLOT : NS * (AB + BB);  // 256 x 256: all 160 KB
    static constexpr int P = MI * NJ, R = MI + NJ;                 // products and fragment reads of a k-step
    // fragment reads up to and including product m's: in the first three quarters where they fit there
    static constexpr int reads(int m) { return 3 * P / 4 >= R ? (m / (3 * P / 4 / R) + 1 < R ? m / (3 * P / 4 / R) + 1 : R) : (m + 1) * R / P; }
};

// logical id of workgroup `bid` of n: consecutive ones run on one XCD
MX_DEV int g16_lid(int bid, int n) {
    const int xcd = bid & 7, q8 = n >> 3, r8 = n & 7;
    return (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + (bid >> 3);
}

// lane l: 16 bytes from the scalar base plus the lane's offset to LDS dst + 16 l
MX_DEV void g16_dma(const void* base, uint32_t off, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(dst) : "memory", "m0");
}

template <bool F16>
MX_DEV f32x4 g16_mfma(u32x4 a, u32x4 b, f32x4 c) {
    if constexpr (F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// acc[i][j] = the sums of rows 16 i .. + 15, columns 16 j .. + 15 of the wave's part of a tile, transposed: lane l holds columns
// 4 (l >> 4) .. + 3 of row l & 15. A and B are the tile's first rows at its first k; row_a(r) / row_b(r) the byte offset of the
// tile's row r of A / B (rows past the matrix repeat its last one).
// The k-tiles are taken from k-tile `rot` on, in a circle (0 <= rot < nk): with ROT workgroups start at different ones.
template <bool F16, int MI, int NJ, bool ROT = false, class RA, class RB>
MX_DEV void g16_tile(char* smem, const char* ab, const char* bb, int nk, RA row_a, RB row_b, f32x4 (&acc)[MI][NJ], int rot = 0) {
    using T = G16T<MI, NJ>;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int g = lane >> 4, col = lane & 15;
    const int wm = wave >> 1, wn = wave & 1;

    // DMA instruction i of a wave brings rows 8 MI wave + 8 i .. + 7 of A (8 NJ wave + 8 i of B): lane l chunk (l & 7) of row l >> 3,
    // taken from the row's chunk (l & 7) ^ ((row >> 1) & 7), so that 16 rows of one chunk lie in 16 bank quads.
    uint32_t ao[MI], bo[NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int row = 8 * (MI * wave + i) + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        ao[i] = row_a(row) + 16 * c;
    }
#pragma unroll
    for (int i = 0; i < NJ; ++i) {
        const int row = 8 * (NJ * wave + i) + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        bo[i] = row_b(row) + 16 * c;
    }
    const uint32_t base = (uint32_t)(uintptr_t)(MX_LDS char*)smem, adst = base + wave * (MI * 1024), bdst = base + wave * (NJ * 1024);
    // instruction i of tile t's A or B to ring offset o; past the end the last tile again, never read
    auto k_at = [&](int t) {
        t = min(t, nk - 1);
        if constexpr (ROT) t = t + rot >= nk ? t + rot - nk : t + rot;
        return (size_t)t * 128;
    };
    auto dma_a = [&](int t, int o, int i) { g16_dma(ab + k_at(t), ao[i], adst + o + i * 1024); };
    auto dma_b = [&](int t, int o, int i) { g16_dma(bb + k_at(t), bo[i], bdst + o + i * 1024); };

#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

    // fragment reads: row's chunk 4 ks + g at (4 ks + g) ^ ((row >> 1) & 7)
    const uint32_t fx = (uint32_t)((g ^ ((col >> 1) & 7)) << 4);
    const uint32_t a_rd = (uint32_t)((wm * 16 * MI + col) * 128), b_rd = (uint32_t)((wn * 16 * NJ + col) * 128);
    u32x4 f[2][MI + NJ];  // of the two k-steps: [MI of A, NJ of B]
    auto rd = [&](int oa, int ob, int ks, int i) {
        const char* p = smem + (i < MI ? oa + a_rd + i * 2048 : ob + b_rd + (i - MI) * 2048) + (fx ^ (ks * 64));
        f[ks][i] = *(const u32x4*)p;
    };
    constexpr int NS = T::NS, STAGE = T::AB + T::BB, RING = T::SLOTS ? 5 * T::SLOT : NS * STAGE;
    // ring offsets of the next tile's A / B from this one's
    auto next = [](int o) { return T::SLOTS ? (o >= 3 * T::SLOT ? o - 3 * T::SLOT : o + 2 * T::SLOT) : (o + STAGE >= RING ? o + STAGE - RING : o + STAGE); };

    int oa = 0, ob = T::SLOTS ? T::SLOT : T::AB, na = oa, nb = ob;
#pragma unroll
    for (int t = 0; t < NS - 1; ++t) {
#pragma unroll
        for (int i = 0; i < MI; ++i) dma_a(t, na, i);
#pragma unroll
        for (int i = 0; i < NJ; ++i) dma_b(t, nb, i);
        na = next(na);
        nb = next(nb);
    }
    int fa = na;  // where the A of tile t + NS - 1 goes
    q2_wait_barrier<(NS - 2) * (MI + NJ)>();
#pragma unroll
    for (int i = 0; i < MI + NJ; ++i) rd(oa, ob, 0, i);

    // WV: the wave, which puts its loads at places of its own among the products
    auto mainloop = [&](auto w_c) {
        constexpr int WV = decltype(w_c)::value, WA = (2 * WV + 1) * NJ / 8, WB = (2 * WV + 1) * MI / 8;
        for (int t = 0; t < nk; ++t) {
            const int na = next(oa), nb = next(ob);
            auto step = [&](auto ks_c, auto beside) {
                constexpr int ks = decltype(ks_c)::value;
#pragma unroll
                for (int m = 0; m < MI * NJ; ++m) {
                    const int i = m / NJ, j = m % NJ;
                    acc[i][j] = g16_mfma<F16>(f[ks][MI + j], f[ks][i], acc[i][j]);  // (C^T: a lane's four sums are columns)
                    beside(m);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            step(std::integral_constant<int, 0>{}, [&](int m) {
#pragma unroll
                for (int r = m ? T::reads(m - 1) : 0; r < T::reads(m); ++r) rd(oa, ob, 1, r);
                if (m % NJ == WA) dma_a(t + NS - 1, fa, m / NJ);
            });
            // A and B of tile t + 1 have landed (later tiles and A of t + NS - 1 may be on their way), and every wave holds what it
            // needs of tile t: B of t + NS - 1 follows into tile t - 1's, or (five slots) into A's slot of tile t
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NS - 3) * (MI + NJ) + MI) : "memory");
            const int fb = T::SLOTS ? oa : fa + T::AB;
            step(std::integral_constant<int, 1>{}, [&](int m) {
#pragma unroll
                for (int r = m ? T::reads(m - 1) : 0; r < T::reads(m); ++r) rd(na, nb, 0, r);
                if (m % MI == WB) dma_b(t + NS - 1, fb, m / MI);
            });
            fa = T::SLOTS ? ob : oa;
            oa = na;
            ob = nb;
        }
    };
    if (wave == 0) mainloop(std::integral_constant<int, 0>{});
    else if (wave == 1) mainloop(std::integral_constant<int, 1>{});
    else if (wave == 2) mainloop(std::integral_constant<int, 2>{});
    else mainloop(std::integral_constant<int, 3>{});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

}  // namespace
