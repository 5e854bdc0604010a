// qmmp.hip — two quantised-weight GEMMs of the same rows in one launch: q|k and v of the K_M mixes, whose formats differ.
//
//   C[M, Na + Nb] (+)= A[M, K] · [Wa; Wb][Na + Nb, K]^T,   A f16, fp32 out
//
// v of a grouped-query model is 1024 of 6144 columns: a launch of its own runs on 16 to 64 of 256 compute units, through the whole of K or, split,
// through atomics, and takes 8 us at 32 rows and 12-20 at 128-416, a third to two thirds of q|k's time. Here its workgroups run beside q|k's,
// with the tiles of qmm2.hip and qmmr.hip. Two such layers of four, a pass before / after: 32 sequences 479 -> 464 us, 9 long ones 541 -> 529, 128 sequences
// 706 -> 684, a 333-token prompt 968 -> 920; a 416-token step, whose v ran beside the end of q|k already, even.
#include "qmmp_impl.h"

// qa, qb: Q4_K + Q6_K, Q5_K + Q6_K, Q3_K + Q5_K. epi 0 or 2 as mxk_qmm2 (splits 1 for 0). kind 2: qmm2 tiles (p0, p1, p2) = (wm, ks, wn),
// (4, 2, 1), (3, 2, 1) or (2, 2, 1); kind 0: qmmr tiles (wm, gw, kw), (1, 1, 4), (1, 2, 4), (1, 4, 4) or (2, 2, 4). C 4-byte aligned.
extern "C" int mxk_qmm_pair(int qa, int qb, int epi, int kind, int p0, int p1, int p2, const uint16_t* A, int lda, const uint8_t* Wa, int Na,
                            const uint8_t* Wb, int Nb, int M, int K, int splits, float* C, int ldc, hipStream_t st) {
    if (M <= 0) return 0;
    if (K <= 0 || K % 256 || (lda & 7) || (((uintptr_t)A | (uintptr_t)Wa | (uintptr_t)Wb) & 15) || Na <= 0 || Nb <= 0 || ((Na | Nb) & 31))
        return (int)hipErrorInvalidValue;
    if (epi != E16_ADD_F32 && splits != 1) return (int)hipErrorInvalidValue;
    const QpArgs a{A, lda, Wa, Wb, Na, Nb, M, K, 0, splits, 0, 0, C, ldc};
    if (qa == MXQ_Q4_K && qb == MXQ_Q6_K) return qmmp_run_q4k_q6k(epi, kind, p0, p1, p2, &a, st);
    if (qa == MXQ_Q5_K && qb == MXQ_Q6_K) return qmmp_run_q5k_q6k(epi, kind, p0, p1, p2, &a, st);
    if (qa == MXQ_Q3_K && qb == MXQ_Q5_K) return qmmp_run_q3k_q5k(epi, kind, p0, p1, p2, &a, st);
    return (int)hipErrorInvalidValue;
}
