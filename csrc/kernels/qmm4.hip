// qmm4.hip — quantised-weight GEMM for some 130 to 1000 rows by wide matrices (gate|up of a prompt chunk or a mixed step).
//
//   C[M, N] = A[M, K] · W[N, K]^T,   A f16, W in the t32 tiled layout (qmm2_fmt.h); by long K also C += A · W^T (down)
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
// tiles and stay with qmm2, but by long K: down (4096 x 14336) runs 32 to 96 tiles in as many parts of K as make one round, and a second kernel
// adds their fp32 sums up. (qmm2's 128 x 128 tiles meet in atomics; those are 4 us a part and a million sums here, eight parts' sums written and read 20.)
// 416 rows: product 50 us, of them 10 the sums' stores, the second kernel 9; the parts of an XCD share one part of A's k in its L2. us, weights in no
// cache, qmm2's best / this: Q4_K 333 rows 56.6 / 52.1, 416 64.7 / 59.0, 700 111 / 85; Q6_K 333 60.6 / 55.2, 416 70.7 / 68.0, 700 110 / 92.
#include "qmm4_impl.h"

namespace {

// C[m, n] += parts 0 .. n_parts - 1 of [M][N], in order; V columns a thread (4 where C's rows allow)
template <int V>
__global__ __launch_bounds__(256) void qmm4_sum_kernel(const float* __restrict__ part, int n_parts, int M, int N, float* __restrict__ C, int ldc) {
    typedef float fv __attribute__((ext_vector_type(V)));
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * V, mn = (size_t)M * N;
    if (i >= mn) return;
    const size_t m = i / (unsigned)N, n = i - m * N;
    fv* const c = (fv*)(C + m * ldc + n);
    fv sum = *(const fv*)(part + i), old = *c;
    for (int p = 1; p < n_parts; p += 7) {  // seven loads at a time
        fv w[7];
#pragma unroll
        for (int j = 0; j < 7; ++j) w[j] = *(const fv*)(part + (size_t)min(p + j, n_parts - 1) * mn + i);
#pragma unroll
        for (int j = 0; j < 7; ++j)
            if (p + j < n_parts) sum += w[j];
    }
    *c = old + sum;
}

int run(int qtype, int epi, int nb, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, int splits, void* C, int ldc, hipStream_t st) {
    if (K <= 0 || K % 256 || (lda & 7) || ((uintptr_t)A & 15) || ((uintptr_t)W & 15) || (N & 31)) return (int)hipErrorInvalidValue;
    switch (qtype) {
        case MXQ_Q4_K: return qmm4_run_q4k(epi, nb, A, lda, W, M, N, K, splits, C, ldc, st);
        case MXQ_Q5_K: return qmm4_run_q5k(epi, nb, A, lda, W, M, N, K, splits, C, ldc, st);
        case MXQ_Q6_K: return qmm4_run_q6k(epi, nb, A, lda, W, M, N, K, splits, C, ldc, st);
        case MXQ_Q3_K: return qmm4_run_q3k(epi, nb, A, lda, W, M, N, K, splits, C, ldc, st);
        case MXQ_Q2_K: return qmm4_run_q2k(epi, nb, A, lda, W, M, N, K, splits, C, ldc, st);
        case MXQ_Q8_0: return qmm4_run_q80(epi, nb, A, lda, W, M, N, K, splits, C, ldc, st);
        case MXQ_MX4F: return qmm4_run_mx4(epi, nb, A, lda, W, M, N, K, splits, C, ldc, st);
        case MXQ_MX5F: return qmm4_run_mx5(epi, nb, A, lda, W, M, N, K, splits, C, ldc, st);
    }
    return (int)hipErrorInvalidValue;
}

}  // namespace

// A f16 [M, K] (lda % 8 == 0, 16-B aligned), W t32 Q4_K / Q5_K / Q6_K / Q3_K / Q2_K / Q8_0 / MX4F / MX5F [N, K] (N % 32 == 0, K % 256 == 0).
// epi: 0 fp32 store, 1 f16 store, 3 / 4 SwiGLU / GeGLU over 16-row interleaved gate|up -> f16 [M, N/2].
// nb: 16-row blocks a row tile may have, 8 .. 14 (fewer where the format's ring does not fit the LDS).
extern "C" int mxk_qmm4(int qtype, int epi, int nb, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, void* C, int ldc,
                        hipStream_t st) {
    if (M <= 0) return 0;
    return run(qtype, epi, nb, A, lda, W, M, N, K, 1, C, ldc, st);
}

// C (fp32) += A W^T, K in `splits` parts whose sums go through part, 4 * splits * M * N bytes (16-B aligned).
extern "C" int mxk_qmm4_parts(int qtype, int nb, int splits, const uint16_t* A, int lda, const uint8_t* W, int M, int N, int K, float* part, float* C,
                              int ldc, hipStream_t st) {
    if (M <= 0) return 0;
    if (splits < 2 || K <= 0 || splits > K >> 8 || N <= 0 || ldc < N || ((uintptr_t)part & 15) || ((uintptr_t)C & 3)) return (int)hipErrorInvalidValue;
    const int err = run(qtype, E16_F32, nb, A, lda, W, M, N, K, splits, part, N, st);
    if (err) return err;
    const int sbps = qmm4_part_blocks(K, splits), n_parts = ((K >> 8) + sbps - 1) / sbps;
    const bool vec = !(((uintptr_t)C & 15) | (ldc & 3));
    const size_t wgs = ((size_t)M * N / (vec ? 4 : 1) + 255) / 256;
    if (wgs > 0xffffff) return (int)hipErrorInvalidValue;
    if (vec) qmm4_sum_kernel<4><<<dim3((unsigned)wgs), 256, 0, st>>>(part, n_parts, M, N, C, ldc);
    else qmm4_sum_kernel<1><<<dim3((unsigned)wgs), 256, 0, st>>>(part, n_parts, M, N, C, ldc);
    MXK_CHECK_LAUNCH();
}
