// qmm4_q3k.hip — qmm4.hip kernel instances for Q3_K weights.
#include "qmm4_impl.h"

int qmm4_run_q3k(int epi, int nb, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st) {
    return qmm4_run<MXQ_Q3_K>(epi, nb, A, lda, W, M, N, K, splits, C, ldc, st);
}
