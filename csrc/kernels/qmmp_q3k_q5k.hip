// qmmp_q3k_q5k.hip — qmmp.hip kernel instances for Q3_K and Q5_K weights.
#include "qmmp_impl.h"

int qmmp_run_q3k_q5k(int epi, int kind, int p0, int p1, int p2, const void* args, hipStream_t st) {
    return qmmp_run<MXQ_Q3_K, MXQ_Q5_K>(epi, kind, p0, p1, p2, *(const QpArgs*)args, st);
}
