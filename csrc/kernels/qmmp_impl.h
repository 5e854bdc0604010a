// qmmp_impl.h — kernel templates of qmmp.hip (see there), shared by the translation units of the format pairs.
#pragma once
#include "qmm2_impl.h"
#include "qmmr_impl.h"

namespace {

struct QpArgs {
    const uint16_t* A;
    int lda;
    const uint8_t *Wa, *Wb;
    int Na, Nb, M, K, n_mt, splits, sbps, nb;  // nb: workgroups of b, a multiple of 8 (the spare ones end at once)
    void* C;
    int ldc;
};

// b's workgroups come first: its few columns are the longer ones. Both parts keep their order of tiles over the XCDs, since nb is a
// multiple of eight
template <int QA, int QB, int WM, int KS, int EPI>
__global__ __launch_bounds__(256 * KS) void qmmp2_kernel(QpArgs a) {
    const int bid = blockIdx.x, own = (a.Nb + 127) / 128 * a.n_mt * a.splits;
    void* const cb = (char*)a.C + (size_t)a.Na * 4;
    if (bid >= a.nb)
        qmm2_body<QA, WM, KS, 1, EPI>(gridDim.x - a.nb, bid - a.nb, a.A, a.lda, a.Wa, a.M, a.Na, a.K, a.n_mt, a.splits, a.sbps, a.C, a.ldc, Q2Group{}, Q2Fuse{});
    else if (bid < own)
        qmm2_body<QB, WM, KS, 1, EPI>(own, bid, a.A, a.lda, a.Wb, a.M, a.Nb, a.K, a.n_mt, a.splits, a.sbps, cb, a.ldc, Q2Group{}, Q2Fuse{});
}

template <int QA, int QB, int WM, int GW, int KW, int EPI>
__global__ __launch_bounds__(64 * GW * KW) void qmmpr_kernel(QpArgs a) {
    const int bid = blockIdx.x, own = (a.Nb + 32 * GW - 1) / (32 * GW) * a.n_mt * a.splits;
    void* const cb = (char*)a.C + (size_t)a.Na * 4;
    if (bid >= a.nb)
        qmmr_body<QA, WM, GW, KW, EPI>(gridDim.x - a.nb, bid - a.nb, a.A, a.lda, a.Wa, a.M, a.Na, a.K, a.n_mt, a.splits, a.sbps, a.C, a.ldc);
    else if (bid < own)
        qmmr_body<QB, WM, GW, KW, EPI>(own, bid, a.A, a.lda, a.Wb, a.M, a.Nb, a.K, a.n_mt, a.splits, a.sbps, cb, a.ldc);
}

// threads, columns of a tile, LDS bytes of both formats
template <class KERN>
static int launch_qmmp(KERN kern, int threads, int bn, int bm, int lds, bool& once, QpArgs a, hipStream_t st) {
    const int nsb = a.K >> 8;
    a.splits = max(1, min(a.splits, nsb));
    a.sbps = (nsb + a.splits - 1) / a.splits;
    a.splits = (nsb + a.sbps - 1) / a.sbps;  // no empty splits
    a.n_mt = (a.M + bm - 1) / bm;
    const long na = (long)((a.Na + bn - 1) / bn) * a.n_mt * a.splits, nb = ((long)((a.Nb + bn - 1) / bn) * a.n_mt * a.splits + 7) / 8 * 8;
    if (na + nb > 0xffffff) return (int)hipErrorInvalidValue;
    a.nb = (int)nb;
    if (!once) {
        (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        once = true;
    }
    kern<<<dim3((unsigned)(na + nb)), threads, lds, st>>>(a);
    MXK_CHECK_LAUNCH();
}

template <int QA, int QB, int EPI>
static int dispatch_qmmp(int kind, int p0, int p1, int p2, const QpArgs& a, hipStream_t st) {
#define QP2(WM_, KS_)                                                                                                                \
    if (kind == 2 && p0 == WM_ && p1 == KS_ && p2 == 1) {                                                                            \
        static bool once = false;                                                                                                     \
        constexpr int LA = Q2Geom<QA, WM_, KS_, 1>::LDS, LB = Q2Geom<QB, WM_, KS_, 1>::LDS;                                           \
        return launch_qmmp(qmmp2_kernel<QA, QB, WM_, KS_, EPI>, 256 * KS_, 128, 32 * WM_, LA > LB ? LA : LB, once, a, st);            \
    }
#define QPR(WM_, GW_, KW_)                                                                                                           \
    if (kind == 0 && p0 == WM_ && p1 == GW_ && p2 == KW_) {                                                                          \
        static bool once = false;                                                                                                     \
        return launch_qmmp(qmmpr_kernel<QA, QB, WM_, GW_, KW_, EPI>, 64 * GW_ * KW_, 32 * GW_, 32 * WM_, QrGeom<WM_, GW_, KW_>::LDS, once, a, st); \
    }
    QP2(4, 2) QP2(3, 2) QP2(2, 2) QPR(1, 1, 4) QPR(1, 2, 4) QPR(1, 4, 4) QPR(2, 2, 4)
#undef QP2
#undef QPR
    return (int)hipErrorInvalidValue;
}

template <int QA, int QB>
static int qmmp_run(int epi, int kind, int p0, int p1, int p2, const QpArgs& a, hipStream_t st) {
    if (epi == E16_F32) return dispatch_qmmp<QA, QB, E16_F32>(kind, p0, p1, p2, a, st);
    if (epi == E16_ADD_F32) return dispatch_qmmp<QA, QB, E16_ADD_F32>(kind, p0, p1, p2, a, st);
    return (int)hipErrorInvalidValue;
}

}  // namespace

int qmmp_run_q4k_q6k(int epi, int kind, int p0, int p1, int p2, const void* args, hipStream_t st);
int qmmp_run_q5k_q6k(int epi, int kind, int p0, int p1, int p2, const void* args, hipStream_t st);
int qmmp_run_q3k_q5k(int epi, int kind, int p0, int p1, int p2, const void* args, hipStream_t st);
