// dense16_enc.hip — dense16.hip's kernel with 16-bit outputs, bias and GELU in the epilogue, for the text encoders' layers (encoder.hip).
//
// With K = 768 a 256 x 256 tile is 12 k-tiles (15 us) and its epilogue as long as half of them, so the stores decide: lanes with four
// columns each (32-byte pieces of 16 rows a store) left 6428 x 2304 x 768 at 34.2 us and 6428 x 768 x 3072 at 34.7; eight columns a lane, by
// the order in which weight rows are staged, and a row's pieces one after another 27.0 and 30.6 (the library's 24.7 and 34.9). With GELU
// 6428 x 3072 x 768 takes 45.6 us, 10 of them GELU's arithmetic (82 with erff), beside the library's product (35) and a pass of 20.
#include "dense16_impl.h"

namespace {

template <int EPI, bool F16>
void enc_go(const D16Args& a, int tile, unsigned n, hipStream_t st) {
#define GO(M_, N_) \
    if (tile == 16 * M_ + N_) dense16_launch<EPI, F16, M_, N_>(a, n, st);
    D16_TILES(GO)
#undef GO
}

}  // namespace

int mx_dense16_enc(int epi, int tile, const uint16_t* A, int lda, const uint16_t* B, int M, int N, int K, const uint16_t* bias, uint16_t* Y, int ldy,
                   int parts, float* part, hipStream_t st) {
    int TM = 0, TN = 0;
#define GO(M_, N_) \
    if (tile == 16 * M_ + N_) TM = 32 * M_, TN = 32 * N_;
    D16_TILES(GO)
#undef GO
    if (!TM || M <= 0 || N <= 0 || K <= 0 || K % G16_K || N % 8 || lda < K || (lda & 7) || lda > (1 << 22) || K > (1 << 22) || parts < 1 || parts > K / G16_K)
        return (int)hipErrorInvalidValue;
    D16Args a{};
    a.A = A;
    a.B = B;
    a.lda = lda;
    a.ldb = K;
    a.M = M;
    a.N = N;
    a.nk = K / G16_K;
    a.n_mt = (M + TM - 1) / TM;
    a.n_nt = (N + TN - 1) / TN;
    a.parts = parts;
    a.part = part;
    a.part_rows = 1;
    a.ldc = ldy;
    a.Y = Y;
    a.bias16 = bias;
    const long n = (long)a.n_mt * a.n_nt * (epi == D16_PART ? parts : 1);
    if (n > 0xffffff || (epi == D16_PART ? !part : !Y || ldy < N || (ldy & 7))) return (int)hipErrorInvalidValue;
    if (epi == D16_ACT) MX_ACT_DISPATCH((enc_go<D16_ACT, F16>(a, tile, (unsigned)n, st)));
    else if (epi == D16_GELU) MX_ACT_DISPATCH((enc_go<D16_GELU, F16>(a, tile, (unsigned)n, st)));
    else if (epi == D16_PART) MX_ACT_DISPATCH((enc_go<D16_PART, F16>(a, tile, (unsigned)n, st)));
    else return (int)hipErrorInvalidValue;
    return (int)hipGetLastError();
}
