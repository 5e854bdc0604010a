// qmmp_q4k_q6k.hip — qmmp.hip kernel instances for Q4_K and Q6_K weights.
#include "qmmp_impl.h"

int qmmp_run_q4k_q6k(int epi, int kind, int p0, int p1, int p2, const void* args, hipStream_t st) {
    return qmmp_run<MXQ_Q4_K, MXQ_Q6_K>(epi, kind, p0, p1, p2, *(const QpArgs*)args, st);
}
