// qmm4_q80.hip — qmm4.hip kernel instances for Q8_0 weights.
#include "qmm4_impl.h"

int qmm4_run_q80(int epi, int nb, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st) {
    return qmm4_run<MXQ_Q8_0>(epi, nb, A, lda, W, M, N, K, splits, C, ldc, st);
}
