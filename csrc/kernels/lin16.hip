// lin16.hip — products of a few 16-bit rows with a 16-bit weight matrix, fp32 out: y[M, N] (+)= x[M, K] W[N, K]^T, M <= 64
// (ops/dense.py). The weights are read once, so the matrix's bytes bound it. A workgroup has 64 columns (64 rows of W, four
// fragments a k-step, so that the rows of x are fetched for four products each) and one of gridDim.y parts of K; its 8 waves
// take every 8th 32-wide k-step, the next one asked for while one is multiplied, and their sums meet in LDS. Parts go to
// `part` and are added in order by a second launch: no atomics, the same bits every time.
// Against the library, weights in no cache (bf16): 4096 x 20480, 33 rows 122 -> 50 us (3.4 TB/s), 8 rows 55 -> 41; 4096 x 17408
// 124 -> 45; 2048 x 20480 65 -> 28; 28672 x 4096, 4 rows 66 -> 53; ops/dense.py few_rows_parts says where it is chosen.
#include "mx_common.h"

namespace {

constexpr int GW = 8, NC = 4;

template <int MT, bool F16, bool ACC>
__global__ __launch_bounds__(64 * GW, MT <= 2 ? 4 : 2) void lin16_kernel(const uint16_t* __restrict__ x, int ldx,
                                                                         const uint16_t* __restrict__ W, float* __restrict__ y,
                                                                         int ldy, float* __restrict__ part, int M, int N, int K) {
    constexpr int RW = MT > 2 ? 4 : GW;  // waves whose sums are in LDS together (64 KB at most)
    __shared__ __attribute__((aligned(16))) float red[RW * MT * NC * 256];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * (16 * NC), KS = K / 32;
    const int s0 = (int)((long)KS * blockIdx.y / gridDim.y) + wave, s1 = (int)((long)KS * (blockIdx.y + 1) / gridDim.y);
    const uint16_t *wp[NC], *xp[MT];  // (rows past the end read the last one and are not stored)
#pragma unroll
    for (int c = 0; c < NC; ++c) wp[c] = W + (size_t)min(n0 + 16 * c + col, N - 1) * K + 8 * g;
#pragma unroll
    for (int t = 0; t < MT; ++t) xp[t] = x + (size_t)min(16 * t + col, M - 1) * ldx + 8 * g;
    f32x4 acc[MT][NC];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[t][c] = (f32x4){0.f, 0.f, 0.f, 0.f};
    auto load = [&](int s, u32x4 (&w)[NC], u32x4 (&xs)[MT]) {
#pragma unroll
        for (int c = 0; c < NC; ++c) w[c] = *(const u32x4*)(wp[c] + (size_t)32 * s);
#pragma unroll
        for (int t = 0; t < MT; ++t) xs[t] = *(const u32x4*)(xp[t] + (size_t)32 * s);
    };
    auto work = [&](const u32x4 (&w)[NC], const u32x4 (&xs)[MT]) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                if constexpr (F16)
                    acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, xs[t]),
                                                                       __builtin_bit_cast(f16x8, w[c]), acc[t][c], 0, 0, 0);
                else
                    acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, xs[t]),
                                                                        __builtin_bit_cast(bf16x8, w[c]), acc[t][c], 0, 0, 0);
            }
    };
    constexpr int PF = 3;  // k-steps in flight
    u32x4 wf[PF][NC], xf[PF][MT];
#pragma unroll
    for (int u = 0; u < PF; ++u)
        if (s0 + GW * u < s1) load(s0 + GW * u, wf[u], xf[u]);
    for (int s = s0; s < s1; s += GW * PF)
#pragma unroll
        for (int u = 0; u < PF; ++u)
            if (s + GW * u < s1) {
                work(wf[u], xf[u]);
                if (s + GW * (u + PF) < s1) load(s + GW * (u + PF), wf[u], xf[u]);
            }
    auto slot = [&](int w, int t, int c) { return (float4*)(red + (((w * MT + t) * NC + c) * 64 + lane) * 4); };
    if constexpr (RW < GW) {  // waves 4 .. 7 first, added by waves 0 .. 3
        if (wave >= RW)
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int c = 0; c < NC; ++c)
                    *slot(wave - RW, t, c) = make_float4(acc[t][c][0], acc[t][c][1], acc[t][c][2], acc[t][c][3]);
        __syncthreads();
        if (wave < RW)
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    const float4 v = *slot(wave, t, c);
                    acc[t][c] += (f32x4){v.x, v.y, v.z, v.w};
                }
    }
    if (wave < RW)
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int c = 0; c < NC; ++c)
                *slot(wave, t, c) = make_float4(acc[t][c][0], acc[t][c][1], acc[t][c][2], acc[t][c][3]);
    __syncthreads();
    for (int idx = threadIdx.x; idx < MT * NC * 256; idx += 64 * GW) {
        const int n = idx % (16 * NC), m = idx / (16 * NC);
        if (m >= M || n0 + n >= N) continue;
        const int e = ((m >> 4) * NC + (n >> 4)) * 256 + (((m & 15) >> 2) * 16 + (n & 15)) * 4 + (m & 3);
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < RW; ++w) v += red[w * MT * NC * 256 + e];
        if (gridDim.y > 1) {
            part[((size_t)blockIdx.y * M + m) * N + n0 + n] = v;
        } else {
            float* yp = y + (size_t)m * ldy + n0 + n;
            *yp = ACC ? *yp + v : v;
        }
    }
}

template <bool ACC>
__global__ __launch_bounds__(256) void lin16_sum_kernel(const float* __restrict__ part, int parts, float* __restrict__ y, int ldy,
                                                        int M, int N) {
    const int n4 = N / 4, i = blockIdx.x * 256 + threadIdx.x;
    if (i >= M * n4) return;
    const int m = i / n4, n = (i - m * n4) * 4;
    float4 v = *(const float4*)(part + (size_t)m * N + n);
    for (int p = 1; p < parts; ++p) {
        const float4 w = *(const float4*)(part + ((size_t)p * M + m) * N + n);
        v.x += w.x;
        v.y += w.y;
        v.z += w.z;
        v.w += w.w;
    }
    float* yp = y + (size_t)m * ldy + n;
    yp[0] = ACC ? yp[0] + v.x : v.x;
    yp[1] = ACC ? yp[1] + v.y : v.y;
    yp[2] = ACC ? yp[2] + v.z : v.z;
    yp[3] = ACC ? yp[3] + v.w : v.w;
}

template <int MT, bool F16, bool ACC>
int lin16_go(const uint16_t* x, int ldx, const uint16_t* W, float* y, int ldy, float* part, int parts, int M, int N, int K,
             hipStream_t st) {
    lin16_kernel<MT, F16, ACC><<<dim3((N + 63) / 64, parts), 64 * GW, 0, st>>>(x, ldx, W, y, ldy, part, M, N, K);
    if (parts > 1) lin16_sum_kernel<ACC><<<(M * (N / 4) + 255) / 256, 256, 0, st>>>(part, parts, y, ldy, M, N);
    return (int)hipGetLastError();
}

template <bool F16, bool ACC>
int lin16(const uint16_t* x, int ldx, const uint16_t* W, float* y, int ldy, float* part, int parts, int M, int N, int K,
          hipStream_t st) {
    switch ((M + 15) / 16) {
        case 1: return lin16_go<1, F16, ACC>(x, ldx, W, y, ldy, part, parts, M, N, K, st);
        case 2: return lin16_go<2, F16, ACC>(x, ldx, W, y, ldy, part, parts, M, N, K, st);
        case 3: return lin16_go<3, F16, ACC>(x, ldx, W, y, ldy, part, parts, M, N, K, st);
        default: return lin16_go<4, F16, ACC>(x, ldx, W, y, ldy, part, parts, M, N, K, st);
    }
}

}  // namespace

// x, W 16-bit (f16: half, else bf16), rows of K numbers, ldx a multiple of 8, both 16-byte aligned; y fp32; part: parts * M * N
// fp32 where parts > 1
extern "C" int mxk_lin16(const uint16_t* x, int ldx, const uint16_t* W, float* y, int ldy, float* part, int parts, int M, int N,
                         int K, int f16, int acc, hipStream_t st) {
    if (M <= 0) return 0;
    if (M > 64 || N <= 0 || N % 4 || K <= 0 || K % 32 || ldx % 8 || ldx < K || ldy < N) return (int)hipErrorInvalidValue;
    if (parts < 1 || parts > 64 || (parts > 1 && !part) || ((uintptr_t)x | (uintptr_t)W | (uintptr_t)part) % 16)
        return (int)hipErrorInvalidValue;
#define GO(F_, A_) return lin16<F_, A_>(x, ldx, W, y, ldy, part, parts, M, N, K, st)
    if (f16) {
        if (acc) GO(true, true);
        GO(true, false);
    }
    if (acc) GO(false, true);
    GO(false, false);
#undef GO
}
