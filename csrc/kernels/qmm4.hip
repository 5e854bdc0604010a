// qmm4.hip — quantised-weight GEMM for some 130 to 1000 rows by wide matrices (gate|up of a prompt chunk or a mixed step).
//
//   C[M, N] = A[M, K] · W[N, K]^T,   A f16, W in the t32 tiled layout (qmm2_fmt.h)
//
// A workgroup of 8 waves holds up to 224 rows x 256 columns, the whole k loop: each wave all of the rows by one 32-column group,
// which it dequantises for itself and nobody else does. What bounds such a tile on this card is power: at 416 rows by 28672 x 4096
// qmm2's form of it (32x32x16 products) kept the matrix units busy 73 % of the time, and the clock fell to 1.4-1.6 GHz.
//   * The products are 16x16x32 instructions. On random f16 operands they run at 1864 TFLOP/s and 1905 MHz where 32x32x16
//     ones run at 1450 and 1461: the accumulators are read and written half as often a flop.
//   * A lane holds gate and up of the same features, four of them side by side in a row: the gated epilogue has no shuffles and
//     stores 8 bytes (qmm2's, 2 bytes from half the lanes behind two shuffles each, took 10 % of the GEMM).
//   * Rows are cut evenly into tiles of whole 16-row blocks, so few rows of products are for nothing.
//   * Two waves a SIMD, each issuing one vector instruction in eight cycles at best: the loop is ordered by hand (qmm2_impl.h).
// gate|up 28672 x 4096, Q4_K, weights in no cache, qmm2's best tile / this: 256 rows 69 / 62 us, 333 rows 94 / 76, 416 rows 106 / 89, 700 rows
// 178 / 158, 2048 rows 462 / 405 (1.19 PFLOP/s). Narrow matrices (4096-6144 columns, up to 1000 rows) leave compute units idle with 256-column
// tiles and stay with qmm2.
#include "qmm4_impl.h"

// A f16 [M, K] (lda % 8 == 0, 16-B aligned), W t32 Q4_K / Q5_K / Q6_K / Q3_K / Q2_K / Q8_0 / MX4F / MX5F [N, K] (N % 32 == 0, K % 256 == 0).
// epi: 0 fp32 store, 1 f16 store, 3 / 4 SwiGLU / GeGLU over 16-row interleaved gate|up -> f16 [M, N/2].
// nb: 16-row blocks a row tile may have, 8 .. 14 (fewer where the format's ring does not fit the LDS).
extern "C" int mxk_qmm4(int qtype, int epi, int nb, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, void* C, int ldc,
                        hipStream_t st) {
    if (M <= 0) return 0;
    if (K <= 0 || K % 256 || (lda & 7) || ((uintptr_t)A & 15) || ((uintptr_t)W & 15) || (N & 31)) return (int)hipErrorInvalidValue;
    switch (qtype) {
        case MXQ_Q4_K: return qmm4_run_q4k(epi, nb, A, lda, W, M, N, K, C, ldc, st);
        case MXQ_Q5_K: return qmm4_run_q5k(epi, nb, A, lda, W, M, N, K, C, ldc, st);
        case MXQ_Q6_K: return qmm4_run_q6k(epi, nb, A, lda, W, M, N, K, C, ldc, st);
        case MXQ_Q3_K: return qmm4_run_q3k(epi, nb, A, lda, W, M, N, K, C, ldc, st);
        case MXQ_Q2_K: return qmm4_run_q2k(epi, nb, A, lda, W, M, N, K, C, ldc, st);
        case MXQ_Q8_0: return qmm4_run_q80(epi, nb, A, lda, W, M, N, K, C, ldc, st);
        case MXQ_MX4F: return qmm4_run_mx4(epi, nb, A, lda, W, M, N, K, C, ldc, st);
        case MXQ_MX5F: return qmm4_run_mx5(epi, nb, A, lda, W, M, N, K, C, ldc, st);
    }
    return (int)hipErrorInvalidValue;
}
