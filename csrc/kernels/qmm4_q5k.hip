// qmm4_q5k.hip — qmm4.hip kernel instances for Q5_K weights.
#include "qmm4_impl.h"

int qmm4_run_q5k(int epi, int nb, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st) {
    return qmm4_run<MXQ_Q5_K>(epi, nb, A, lda, W, M, N, K, splits, C, ldc, st);
}
