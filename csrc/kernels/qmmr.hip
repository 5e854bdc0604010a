// qmmr.hip — quantised-weight GEMM of few rows (decode batches of 5 to about 64 sequences).
//
//   C[M, N] (+)= A[M, K] · W[N, K]^T,   A f16, W in the t32 tiled layout (ops/quant.py tile32)
//
// At these sizes a pass reads its weights once and decodes each of them once, however few the rows are. qmm2's tiles send
// the packed bytes through LDS and step through K behind one barrier per 64 columns of it with two waves on a SIMD, which
// neither fills the vector unit nor the memory (gate|up of 32 rows: 55 % issue, 2.3 TB/s). Here
//   * a wave loads the packed bytes of its 32-column group straight into registers (a t32 unit is laid out so that a lane's
//     bytes are contiguous in a row of lanes), two super-blocks ahead: no LDS traffic for weights;
//   * the KW waves of a group take the quarters of each 256-k super-block, so a barrier comes once per 256 k, and up to four
//     waves share a SIMD; their sums meet in LDS at the end, each wave then finishing 16 / KW of the 16 rows a lane holds;
//   * only A, 32 or 64 rows of the super-block, is staged in LDS, through registers, rows 528 bytes apart.
// What bounds it now is the decoding: without any load gate|up 28672 x 4096 takes 18 of its 21 us, without decoding 18, with
// loads alone 17. Larger tiles of columns a wave, more super-blocks a stage, deeper prefetch or decoding with the scaled
// e4m3 conversion (a half-rate instruction) changed nothing or cost 1 to 3 us.
// Measured against the best qmm2 / qmm3 tile, weights in no cache, us: gate|up 28672 x 4096 Q4_K 9 rows 29.2 -> 21.2, 32 rows
// 28.2 -> 21.0, 64 rows 28.9 -> 28.4; 4096 x 4096 9 / 32 / 64 rows 6.7 -> 6.2, 9.0 -> 6.8, 11.3 -> 9.1; 4096 x 14336 Q4_K
// 14.2 -> 12.3, 16.6 -> 14.3, 20.2 -> 19.8, Q6_K 16.0 -> 15.3, 18.3 -> 17.0, 21.8 -> 22.8; 6144 x 4096 8.5 -> 7.5, 10.5 ->
// 8.2, 12.8 -> 11.4. From 128 rows on the row tiles decode the weights again and qmm2 / qmm3 are the faster ones but for
// narrow outputs (4096 x 4096 14.8 -> 12.7); the load-time tuner decides.
#include "qmmr_impl.h"

// A f16 [M, K] (lda % 8 == 0, 16-B aligned), W t32 (N % 32 == 0, K % 256 == 0). epi as mxk_qmm2 (split-K only with epi 2).
// (wm, gw, kw): tiles of 32 wm rows x 32 gw columns, kw waves over each super-block (qmmr_impl.h dispatch_qmmr).
extern "C" int mxk_qmmr(int qtype, int epi, int wm, int gw, int kw, const uint16_t* A, int lda, const uint8_t* W, int M,
                        int N, int K, int splits, void* C, int ldc, hipStream_t st) {
    if (M <= 0) return 0;
    if (K % 256 || (lda & 7) || ((uintptr_t)A & 15) || ((uintptr_t)W & 15) || (N & 31)) return (int)hipErrorInvalidValue;
    if (epi != E16_ADD_F32 && splits != 1) return (int)hipErrorInvalidValue;
    switch (qtype) {
        case MXQ_Q4_K: return qmmr_run_q4k(epi, wm, gw, kw, A, lda, W, M, N, K, splits, C, ldc, st);
        case MXQ_Q5_K: return qmmr_run_q5k(epi, wm, gw, kw, A, lda, W, M, N, K, splits, C, ldc, st);
        case MXQ_Q6_K: return qmmr_run_q6k(epi, wm, gw, kw, A, lda, W, M, N, K, splits, C, ldc, st);
        case MXQ_Q3_K: return qmmr_run_q3k(epi, wm, gw, kw, A, lda, W, M, N, K, splits, C, ldc, st);
        case MXQ_Q2_K: return qmmr_run_q2k(epi, wm, gw, kw, A, lda, W, M, N, K, splits, C, ldc, st);
        case MXQ_Q8_0: return qmmr_run_q80(epi, wm, gw, kw, A, lda, W, M, N, K, splits, C, ldc, st);
        case MXQ_MX4F: return qmmr_run_mx4(epi, wm, gw, kw, A, lda, W, M, N, K, splits, C, ldc, st);
        case MXQ_MX5F: return qmmr_run_mx5(epi, wm, gw, kw, A, lda, W, M, N, K, splits, C, ldc, st);
    }
    return (int)hipErrorInvalidValue;
}
