// qmm4_mx4.hip — qmm4.hip kernel instances for MX4F weights.
#include "qmm4_impl.h"

int qmm4_run_mx4(int epi, int nb, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st) {
    return qmm4_run<MXQ_MX4F>(epi, nb, A, lda, W, M, N, K, splits, C, ldc, st);
}
