// attn_tile.h — the key tile of the attention kernels that hold their scores transposed (attention_flash.hip: prompts over the
// paged cache; attention_dense.hip: dense rows): head dims 64 / 128, 64 keys in LDS as a K and a V image, 32 queries (or query and
// head pairs) a wave as columns of 32x32x16 MFMA tiles. S^T = K Q^T gives a lane keys 8 j + 4 h + i of its column (h: half-wave); the
// probabilities are then the B operand of O^T = V^T P^T as they lie, both operands' k slot (h, e) being key 8 (e / 4) + 4 h + e % 4
// of the 16.
#pragma once
#include <type_traits>

#include "mx_common.h"

namespace {

constexpr int AT_KEYS = 64;  // keys per tile

// K image: row p, 16-byte chunk c at c ^ row bits, read as A fragments (ds_read_b128, 32 rows x 1 chunk a half-wave); V image: row p,
// 32-byte region r (16 dims) at r ^ row bits, read with ds_read_b64_tr_b16 (4 keys of a dim per lane). Both reads are free of
// bank conflicts.
template <int D>
MX_DEV int at_k_off(int p, int c) {
    const int f = D == 128 ? (p & 15) : ((p >> 1) & 7);
    return p * (2 * D) + ((c ^ f) << 4);
}
template <int D>
MX_DEV int at_v_off(int p, int r) {
    const int f = D == 128 ? (p & 7) : ((p >> 1) & 3);
    return p * (2 * D) + ((r ^ f) << 5);
}

MX_DEV float at_half_max(float x) {  // max of the two half-waves' values of a column, in both
    const u32x2 r = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false));
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
MX_DEV float at_half_sum(float x) {
    const u32x2 r = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false));
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <bool F16>
MX_DEV f32x16 at_mfma(u32x4 a, u32x4 b, f32x16 c) {
    if constexpr (F16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// A tile in three steps; sc[u][j] is key 32 u + 8 (j / 4) + 4 h + j % 4 of the lane's column. The fences keep the fragment reads ahead
// of what they wait behind: K's before the first product, V's first before the softmax, its others one k-step ahead of their
// products (left alone, the scheduler puts every read next to its use).
// 1. sc = K Q^T; qf: Q^T as B operand (lane = column, dims 16 ks + 8 h). KB: k-steps whose K fragments are read together;
// mid(ks): other work of the wave, issued while k-step ks's two products run (each holds the matrix unit for 32 cycles)
struct AtNone {
    MX_DEV void operator()(int) const {}
};
template <int D, bool F16, int KB, class Mid = AtNone>
MX_DEV void at_scores(const char* kb, int h, int col, const u32x4 (&qf)[D / 16], f32x16 (&sc)[2], Mid mid = {}) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int j = 0; j < 16; ++j) sc[u][j] = 0.f;
    u32x4 kf[D / 16][2];
    auto read_k = [&](int k0) {
#pragma unroll
        for (int ks = k0; ks < k0 + KB; ++ks)
#pragma unroll
            for (int u = 0; u < 2; ++u) kf[ks][u] = *(const u32x4*)(kb + at_k_off<D>(32 * u + col, 2 * ks + h));
    };
    read_k(0);
#pragma unroll
    for (int k0 = 0; k0 < D / 16; k0 += KB) {
        __builtin_amdgcn_sched_barrier(0);
        if (k0 + KB < D / 16) read_k(k0 + KB);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = k0; ks < k0 + KB; ++ks) {
#pragma unroll
            for (int u = 0; u < 2; ++u) sc[u] = at_mfma<F16>(kf[ks][u], qf[ks], sc[u]);
            if constexpr (!std::is_same<Mid, AtNone>::value) {
                __builtin_amdgcn_sched_barrier(0);
                mid(ks);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
}
// Where in a V image this lane's reads of V^T's fragments begin: row 4 h + (lane % 16) / 4, dims 32 mt on. The rows of a k-step and its
// second half are multiples of 8 further, which leaves the row bits of at_v_off as they are.
template <int D>
MX_DEV void at_v_lane(int lane, int (&vo)[D / 32]) {
    const int i16 = lane & 15, dh = (lane >> 4) & 1;
#pragma unroll
    for (int mt = 0; mt < D / 32; ++mt) vo[mt] = at_v_off<D>(4 * (lane >> 5) + (i16 >> 2), 2 * mt + dh) + 8 * (i16 & 3);
}
// 2. (and between 3.'s products) V^T's fragments of k-step ks
template <int D>
MX_DEV void at_read_v(const char* vb, const int (&vo)[D / 32], int ks, u32x4 (&vf)[4][D / 32]) {
#pragma unroll
    for (int mt = 0; mt < D / 32; ++mt) {
        const char* p = vb + vo[mt] + 16 * ks * (2 * D);
        const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((MX_LDS s16x4*)p));
        const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((MX_LDS s16x4*)(p + 8 * (2 * D))));
        vf[ks][mt] = (u32x4){lo[0], lo[1], hi[0], hi[1]};
    }
}
// 3. o += V^T P^T of scores that, times mul, are in the log2 domain (-inf: not seen); m_run, l_run: the column's maximum and this lane's
// share of its sum; vf[0] has been read
template <int D, bool F16>
MX_DEV void at_softmax_v(const char* vb, const int (&vo)[D / 32], f32x16 (&sc)[2], float mul, u32x4 (&vf)[4][D / 32], f32x16 (&o)[D / 32],
                         float& m_run, float& l_run) {
    // (med3 with infinity is the maximum without the quieting of its inputs that fmaxf asks for)
    float mx[2] = {sc[0][0], sc[1][0]};
#pragma unroll
    for (int j = 1; j < 16; ++j)
#pragma unroll
        for (int u = 0; u < 2; ++u) mx[u] = __builtin_amdgcn_fmed3f(mx[u], sc[u][j], INFINITY);
    const float m_new = fmaxf(m_run, at_half_max(fmaxf(mx[0], mx[1])) * mul);
    if (__any(m_new > m_run)) {
        const float alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);
        l_run *= alpha;
#pragma unroll
        for (int i = 0; i < D / 32; ++i)
#pragma unroll
            for (int j = 0; j < 16; ++j) o[i][j] *= alpha;
        m_run = m_new;
    }
    const float m_use = m_run == -INFINITY ? 0.f : m_run;
    float ls[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const int u = ks >> 1, j0 = 8 * (ks & 1);
        if (ks < 3) at_read_v<D>(vb, vo, ks + 1, vf);
        uint32_t pw[4];
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
            const float p0 = __builtin_amdgcn_exp2f(fmaf(sc[u][j0 + j], mul, -m_use));
            const float p1 = __builtin_amdgcn_exp2f(fmaf(sc[u][j0 + j + 1], mul, -m_use));
            ls[j & 2] += p0;
            ls[(j & 2) + 1] += p1;
            pw[j >> 1] = pack_act2<F16>(p0, p1);
        }
        const u32x4 pf = (u32x4){pw[0], pw[1], pw[2], pw[3]};
#pragma unroll
        for (int mt = 0; mt < D / 32; ++mt) o[mt] = at_mfma<F16>(vf[ks][mt], pf, o[mt]);
        __builtin_amdgcn_sched_barrier(0);
    }
    l_run += (ls[0] + ls[1]) + (ls[2] + ls[3]);
}

}  // namespace
