// dense16.hip — bf16 products with weights that are bf16 in memory (ops/dense.py): C[M, N] (+)= A[M, K] · B[N, K]^T (+ bias), fp32 out, and
// with a gated unit's columns beside them in bf16 (the hybrid decoder's input projection: its gates and ups are 70 % of the columns, and
// in fp32 they were written, read again and written a third time).
//
// gemm16.hip's loop in eleven tiles from 256 x 256 to 64 x 128 (gemm16_impl.h), K split over workgroups where tiles alone leave compute
// units idle: all tiles of a product of few columns, or those behind the last full round. What bounds it: at 1000 rows and more the
// products (1.2 - 1.4 PFLOP/s of 1.55 that a large product of the library reaches), to some 100 rows the weights' bytes (4.7 - 5.2 TB/s),
// between them a k-tile's loads that are as long as its products. Smaller tiles hold more k-tiles on their way (64 x 128: six of 24 KB;
// with two as in the largest 4096 x 20480 took 45 us at 64 rows, now 39). ops/dense.py dense16_plan picks by a fitted estimate.
// us, weights in no cache, library / here: 4096 x 20480 added to the residual at 33 / 128 / 512 / 1990 rows 125 / 38, 112 / 46, 151 / 87, 438 / 240;
// 32000 x 4096 at 33 rows 61 / 54; 12320 + 2 x 14336 x 4096 gated, beside the product and the gating kernel, 33 / 322 / 1990 rows 78 / 67, 214 / 143,
// 649 / 554.
#include "dense16_impl.h"

namespace {

// the tiles summed in parts: C (+)= bias + their parts in order; grid (TM * TN / 1024, tiles)
template <bool ADD>
__global__ __launch_bounds__(256) void dense16_sum_kernel(D16Args a, int TM, int TN) {
    const int gt = a.n_mt * a.g_nt, t = blockIdx.y;
    int mt, nt;
    q2_tile_of(a.full + t - gt, a.n_mt, a.n_nt, mt, nt);
    const int e = (blockIdx.x * 256 + threadIdx.x) * 4, m = mt * TM + e / TN, n = nt * TN + e % TN;
    if (m >= a.M || n >= a.N) return;
    const float* p = a.part + (size_t)t * a.parts * (TM * TN) + e;
    float* c = a.C + (size_t)m * a.ldc + n;
    f32x4 v = *(const f32x4*)p, o = ADD ? *(const f32x4*)c : (f32x4){0.f, 0.f, 0.f, 0.f};
    const f32x4 b = a.bias ? *(const f32x4*)(a.bias + n) : (f32x4){0.f, 0.f, 0.f, 0.f};
    for (int i = 1; i < a.parts; i += 4) {  // four loads at a time
        f32x4 w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = *(const f32x4*)(p + (size_t)min(i + j, a.parts - 1) * (TM * TN));
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (i + j < a.parts) v += w[j];
    }
    v += b;
    if (ADD) v += o;
    *(f32x4*)c = v;
}

void part_go(const D16Args& a, int tile, unsigned n, hipStream_t st) {
#define GO(M_, N_) \
    if (tile == 16 * M_ + N_) dense16_launch<D16_PART, false, M_, N_>(a, n, st);
    D16_TILES(GO)
#undef GO
}

template <int EPI>
void plain_go(const D16Args& a, int tile, unsigned n, hipStream_t st) {
#define GO(M_, N_) \
    if (tile == 16 * M_ + N_) dense16_launch<EPI, false, M_, N_>(a, n, st);
    D16_TILES(GO)
#undef GO
}

}  // namespace

// A [M, K], B [N, K] bf16, rows 16-byte aligned, K % 64 == 0. epi 0: C = , 1: C += , 4: C = the first N rows of B, and G the gated unit of its
// rows gate0 .. + F - 1 and up0 .. + F - 1. tile: 16 MI + NJ of one of D16_TILES. Tiles from `full` on (gated ones come first) are summed in
// `parts` parts of K through `part`: 4 * TM * TN bytes for each tile and part.
extern "C" int mxk_dense16(int epi, int tile, const uint16_t* A, int lda, const uint16_t* B, int ldb, int M, int N, int K, const float* bias, float* C,
                           int ldc, int full, int parts, float* part, int F, int gate0, int up0, const float* gate_b, const float* up_b,
                           uint16_t* G, int ldg, hipStream_t st) {
    if (M <= 0 || N <= 0) return 0;
    if ((epi != D16_F32 && epi != D16_ADD && epi != D16_GLU) || K <= 0 || K % G16_K || N % 4 || (lda & 7) || (ldb & 7) || lda < K || ldb < K ||
        lda > (1 << 22) || ldb > (1 << 22) || (ldc & 3) || ldc < N || (((uintptr_t)A | (uintptr_t)B | (uintptr_t)C | (uintptr_t)bias | (uintptr_t)part) & 15))
        return (int)hipErrorInvalidValue;  // (256 rows of 2^23 bytes: the 32-bit lane offsets)
    if (epi == D16_GLU && (F <= 0 || F % 8 || gate0 < N || up0 < gate0 + F || ((long)up0 + F) * ldb * 2 > 0xffffffffl || !G || (ldg & 7) || ldg < F ||
                           ((uintptr_t)G & 15) || (((uintptr_t)gate_b | (uintptr_t)up_b) & 15) || bias))
        return (int)hipErrorInvalidValue;
    int TM = 0, TN = 0;
#define GO(M_, N_) \
    if (tile == 16 * M_ + N_) TM = 32 * M_, TN = 32 * N_;
    D16_TILES(GO)
#undef GO
    if (!TM) return (int)hipErrorInvalidValue;
    D16Args a{A, B, lda, ldb, M, N, K / G16_K, (M + TM - 1) / TM, (N + TN - 1) / TN, full, parts, part, bias, C, ldc, 0, F, gate0, up0, gate_b, up_b, G, ldg};
    if (epi == D16_GLU) a.g_nt = (int)((2l * F + TN - 1) / TN);
    const long tiles = (long)a.n_mt * (a.n_nt + a.g_nt);
    if (tiles > 0xffffff) return (int)hipErrorInvalidValue;  // (of 256 threads: a grid holds less than 2^32)
    if (parts <= 1) a.full = (int)tiles;
    const long rest = tiles - a.full;
    if (a.full < 0 || rest < 0 || (parts > 1 && (rest > (long)a.n_mt * a.n_nt || parts > a.nk || rest * parts > 0xffffff || !part || rest > 65535)))
        return (int)hipErrorInvalidValue;
    if (a.full) {
        if (epi == D16_GLU) mx_dense16_glu(&a, tile, (unsigned)a.full, st);
        else if (epi == D16_ADD) plain_go<D16_ADD>(a, tile, (unsigned)a.full, st);
        else plain_go<D16_F32>(a, tile, (unsigned)a.full, st);
    }
    if (rest) {
        part_go(a, tile, (unsigned)(rest * parts), st);
        const dim3 grid(TM * TN / 1024, (unsigned)rest);
        if (epi == D16_ADD) dense16_sum_kernel<true><<<grid, 256, 0, st>>>(a, TM, TN);
        else dense16_sum_kernel<false><<<grid, 256, 0, st>>>(a, TM, TN);
    }
    return (int)hipGetLastError();
}
