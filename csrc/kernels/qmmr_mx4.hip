// qmmr_mx4.hip — qmmr.hip kernel instances for MX4F weights (one translation unit per block format, so
// the instances compile in parallel).
#include "qmmr_impl.h"

int qmmr_run_mx4(int epi, int wm, int gw, int kw, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st) {
    return qmmr_run<MXQ_MX4F>(epi, wm, gw, kw, A, lda, W, M, N, K, splits, C, ldc, st);
}
