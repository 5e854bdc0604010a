// qmm2_fmt.h — the t32 quantised-weight formats as seen by the MFMA GEMMs (qmm2.hip, qmm3.hip, qmm4.hip, qmmr.hip): per format
// the unit / header / quant byte geometry of one 32-column group x 256-k super-block (Q2F) and the per-lane register
// decoder that turns their bytes into MFMA B fragments (Q2B).
#pragma once
#include "qdeq16.h"

namespace {

template <int N_>
MX_DEV void q2_wait_barrier() {
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N_) : "memory");
}

// Tile order of a GEMM's workgroups: `lid` counts them so that consecutive ones run on one XCD (32 at a time), n_mt row
// tiles by n_rest column panels (and K splits). Row tiles go in bands of Q2_BAND, panels inside a band: the 32 then hold
// 4 row tiles x 8 panels, and per 64-k tile the XCD's L2 takes in 4 x 16 KB of A and 8 x 4.6 KB of Q4_K instead of 32 row
// tiles' 512 KB. With all of a panel's row tiles first (what up to 4 row tiles still are) an 8191-row GEMM reads the whole
// activation matrix once per panel from beyond the L2: bands took gate|up 28672 x 4096 from 1834 to 1736 us there, 4096 x
// 14336 from 952 to 918, and change nothing at one or two row tiles.
constexpr int Q2_BAND = 4;
MX_DEV void q2_tile_of(int lid, int n_mt, int n_rest, int& mt, int& rest) {
    const int band = lid / (Q2_BAND * n_rest), in = lid - band * (Q2_BAND * n_rest);
    const int rows = min(Q2_BAND, n_mt - band * Q2_BAND);
    mt = band * Q2_BAND + in % rows;
    rest = in / rows;
}

template <int QT>
struct Q2F;
// Q4_K t32 unit (per 32-column group, per super-block): [hdr 32 x 16 B][quarter jq: chunk0, chunk1 (32 x 16 B)]
// QB: quant bytes staged per group per k-tile (source unit offset qoff(JQ)); HB: header bytes per group per
// super-block (staged with the super-block's first k-tile); QI / HI: LDS-DMA instructions for each.
template <>
struct Q2F<MXQ_Q4_K> {
    static constexpr int UNIT = 4608, HB = 512, QB = 1024, QI = 1, HI = 1;
    static constexpr int qoff(int jq) { return 512 + jq * 1024; }
};
// Q5_K t32 unit: [hdr 32 x 16 B][qs as Q4_K: quarter jq = chunk0, chunk1][qh: 2 chunks x 32 x 16 B]; the header
// slot holds hdr + qh (the fifth bit of all four k-tiles, staged once per super-block: qoff(4) = 4608)
template <>
struct Q2F<MXQ_Q5_K> {
    static constexpr int UNIT = 5632, HB = 1536, QB = 1024, QI = 1, HI = 2;
    static constexpr int qoff(int jq) { return 512 + jq * 1024; }
    static constexpr int QH = 4608;  // unit offset of the qh chunks
};
// Q6_K t32 unit: [sc 32 x 16 B][d 32 x 4 B][quarter jq: ql0, ql1, qh (32 x 16 B)]
template <>
struct Q2F<MXQ_Q6_K> {
    static constexpr int UNIT = 6784, HB = 640, QB = 1536, QI = 2, HI = 2;
    static constexpr int qoff(int jq) { return 640 + jq * 1536; }
};
// Q3_K t32 unit: [hdr 32 x 16 B {scales[12], d}][hmask: 2 chunks x 32 x 16 B][qs half n: 2 chunks x 32 x 16 B];
// k-tiles 2n, 2n+1 use qs half n (the 2-bit fields 0-1 / 2-3) -> header slot = hdr + hmask (1.5 KB)
template <>
struct Q2F<MXQ_Q3_K> {
    static constexpr int UNIT = 3584, HB = 1536, QB = 1024, QI = 1, HI = 2;
    static constexpr int qoff(int jq) { return 1536 + (jq >> 1) * 1024; }
};
// Q2_K t32 unit: [sc 32 x 16 B][dd 32 x 4 B {d, dmin}][qs half n: 2 chunks x 32 x 16 B]
template <>
struct Q2F<MXQ_Q2_K> {
    static constexpr int UNIT = 2688, HB = 640, QB = 1024, QI = 1, HI = 2;
    static constexpr int qoff(int jq) { return 640 + (jq >> 1) * 1024; }
};

// MX4F / MX5F t32 unit (Q4_0 / Q4_1 / Q5_0 / Q5_1 carried exactly at 4 / 5 bits): [hdr: 2 halves x 32 x 16 B {f16 s[4],
// m[4]}, k-tiles 0-1 read half 0, 2-3 half 1][k-tile jq: 2 x (32 x 16 B codes) (+ MX5F: 32 x 8 B high bits)]
template <>
struct Q2F<MXQ_MX4F> {
    static constexpr int UNIT = 5120, HB = 1024, QB = 1024, QI = 1, HI = 1;
    static constexpr int qoff(int jq) { return 1024 + jq * 1024; }
};
template <>
struct Q2F<MXQ_MX5F> {
    static constexpr int UNIT = 6144, HB = 1024, QB = 1280, QI = 2, HI = 1;
    static constexpr int qoff(int jq) { return 1024 + jq * 1280; }
};
// Q8_0 t32 unit per 64-k tile: [d: 32 x {f16 d0, f16 d1}][4 k-steps x (32 x 16 B int8 codes)] (2176 B); a "super-block"
// here is 4 such tiles, and each tile's scales travel with its codes (no header)
template <>
struct Q2F<MXQ_Q8_0> {
    static constexpr int UNIT = 4 * 2176, HB = 0, QB = 2176, QI = 3, HI = 0;
    static constexpr int qoff(int jq) { return jq * 2176; }
};

// Register decoder of one column's bytes of a k-tile, for the B fragments of two matrix instructions:
//   MK 16 (32x32x16): four fragments S = 0 .. 3, k 16 S ..; the lane is column c = lane & 31, l = lane >> 5, its k 8 l .. 8 l + 7 of the 16.
//     S is chunk S & 1 and nibble (bit pair, ...) S >> 1 of the t32 bytes, the lane's 8 bytes start at 8 l of the chunk.
//   MK 32 (16x16x32): two fragments S = 0, 1, k 32 S ..; c = lane & 15 (+ 16 for the group's second half), l = lane >> 4, its k
//     16 (l & 1) + 8 (l >> 1) .. + 7 of the 32 (in that order the A image's reads are free of bank conflicts): chunk l & 1, nibble S,
//     8 bytes from 8 (l >> 1).
// load_hdr, load_q: a super-block's header, a k-tile's bytes. prep<JQ, S>: fragment S's scales (each S in ascending order, S even
// first). half<JQ, S, H>: its k 4 H .. 4 H + 3. These are pieces of half a dozen instructions that a kernel can spread between its
// products; frag does all of them.
template <int QT, int MK = 16>
struct Q2B;

// four codes of 0 .. 15, one a byte -> f16 pairs, exact: a byte 0 .. 15 is the e4m3 number code * 2^-9, so one conversion with
// a scale of 2^9 does a pair (a byte permutation into 1024 + code and a subtraction take two, each at the same rate).
MX_DEV void q2_codes4(uint32_t t, f16x2& p0, f16x2& p1) {
    p0 = __builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8((int)t, 512.f, false));
    p1 = __builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8((int)t, 512.f, true));
}
MX_DEV u32x2 q2_pack4(f16x2 a, f16x2 b) { return (u32x2){__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b)}; }
// four codes of 0 .. 15 -> code * s + m in f16
MX_DEV u32x2 q2_affine4(uint32_t t, f16x2 s, f16x2 m) {
    f16x2 p0, p1;
    q2_codes4(t, p0, p1);
    return q2_pack4(p0 * s + m, p1 * s + m);
}
// four codes of a byte -> (code - off) * s in f16, k1 = 1024 + off; or code * s + m
MX_DEV u32x2 q2_magic4(uint32_t t, _Float16 k1, f16x2 s) {
    const f16x2 k = {k1, k1};
    f16x2 p0, p1;
    magic4(t, p0, p1);
    return q2_pack4((p0 - k) * s, (p1 - k) * s);
}
MX_DEV u32x2 q2_magic4(uint32_t t, f16x2 s, f16x2 m) {
    const f16x2 k = {(_Float16)1024.f, (_Float16)1024.f};
    f16x2 p0, p1;
    magic4(t, p0, p1);
    return q2_pack4((p0 - k) * s + m, (p1 - k) * s + m);
}
MX_DEV f16x2 q2_lo(f16x2 v) { return (f16x2){v[0], v[0]}; }
MX_DEV f16x2 q2_hi(f16x2 v) { return (f16x2){v[1], v[1]}; }

// what the formats share: the lane's chunks and where fragment S lies in them
template <int MK>
struct Q2Lane {
    static_assert(MK == 16 || MK == 32, "MK");
    static constexpr int NC = MK == 16 ? 2 : 1;                          // chunks a lane reads
    static constexpr int ch(int S) { return MK == 16 ? S & 1 : 0; }     // its chunk of fragment S
    static constexpr int nib(int S) { return MK == 16 ? S >> 1 : S; }   // nibble / bit pair of fragment S
    static constexpr bool fresh(int S) { return MK == 32 || !(S & 1); }  // first fragment of a 32-k sub-block
    static MX_DEV int half(int l) { return MK == 16 ? l : l >> 1; }
    // the lane's 8 bytes of its chunks, of a pair of 32 x 16 B chunks
    static MX_DEV void load(u32x2 (&v)[NC], const char* p, int c, int l) {
        if constexpr (MK == 16) {
            v[0] = *(const u32x2*)(p + c * 16 + 8 * l);
            v[1] = *(const u32x2*)(p + 512 + c * 16 + 8 * l);
        } else {
            v[0] = *(const u32x2*)(p + (l & 1) * 512 + c * 16 + 8 * (l >> 1));
        }
    }
    // bit of 16-k sub-block S (MK 16) / 2 S + (l & 1) (MK 32) in a word of four bytes
    static MX_DEV int byte16(int S, int l) { return MK == 16 ? 8 * S : 16 * S + 8 * (l & 1); }
};
#define Q2_FRAG                                                                                  \
    template <int JQ, int S>                                                                      \
    MX_DEV f16x8 frag() {                                                                         \
        prep<JQ, S>();                                                                            \
        const u32x2 a = half<JQ, S, 0>(), b = half<JQ, S, 1>();                                   \
        return __builtin_bit_cast(f16x8, (u32x4){a[0], a[1], b[0], b[1]});                        \
    }

template <int MK>
struct Q2B<MXQ_Q4_K, MK> {
    using L = Q2Lane<MK>;
    u32x4 hd;
    u32x2 v[L::NC];
    f16x2 sm;  // the sub-block's (scale, -dmin * min) as exact f16 products
    MX_DEV void load_hdr(const char* hb, int c, int) { hd = *(const u32x4*)(hb + c * 16); }
    MX_DEV void load_q(const char* qb, int c, int l) { L::load(v, qb, c, l); }
    template <int JQ, int S>
    MX_DEV void prep() {
        if constexpr (L::fresh(S)) {
            const uint32_t w0 = hd[0];  // scalar first: clang bit-casts the whole vector for bit_cast(T, v[i])
            const f16x2 dd = __builtin_bit_cast(f16x2, w0);
            const f16x2 dn = {dd[0], -dd[1]};
            int sc, mn;
            q4k_scale_min_w(hd[1], hd[2], hd[3], 2 * JQ + L::nib(S), sc, mn);
            const f16x2 q = {(_Float16)sc, (_Float16)mn};
            sm = dn * q;  // d * sc is exact in f32 (11 x 6 bits): the f16 product rounds exactly like the f32 path
        }
    }
    template <int JQ, int S, int H>
    MX_DEV u32x2 half() const {
        return q2_affine4((v[L::ch(S)][H] >> (4 * L::nib(S))) & 0x0F0F0F0Fu, q2_lo(sm), q2_hi(sm));
    }
    Q2_FRAG
};

// Q5_K: Q4_K's nibbles plus the fifth bit, bit 2 JQ + nibble of the qh byte of the lane's k
template <int MK>
struct Q2B<MXQ_Q5_K, MK> {
    using L = Q2Lane<MK>;
    u32x4 hd;
    u32x2 qh[L::NC], v[L::NC];
    f16x2 sm;
    MX_DEV void load_hdr(const char* hb, int c, int l) { load_hdr(hb, hb + 512, c, l); }
    MX_DEV void load_hdr(const char* hb, const char* qhb, int c, int l) {  // qhb: the fifth-bit chunks
        hd = *(const u32x4*)(hb + c * 16);
        L::load(qh, qhb, c, l);
    }
    MX_DEV void load_q(const char* qb, int c, int l) { L::load(v, qb, c, l); }
    template <int JQ, int S>
    MX_DEV void prep() {
        if constexpr (L::fresh(S)) {
            const uint32_t w0 = hd[0];
            const f16x2 dd = __builtin_bit_cast(f16x2, w0);
            const f16x2 dn = {dd[0], -dd[1]};
            int sc, mn;
            q4k_scale_min_w(hd[1], hd[2], hd[3], 2 * JQ + L::nib(S), sc, mn);
            const f16x2 q = {(_Float16)sc, (_Float16)mn};
            sm = dn * q;  // exact f16 products (11 x 6 bits)
        }
    }
    template <int JQ, int S, int H>
    MX_DEV u32x2 half() const {
        const uint32_t t = ((v[L::ch(S)][H] >> (4 * L::nib(S))) & 0x0F0F0F0Fu) |
                           (((qh[L::ch(S)][H] >> (2 * JQ + L::nib(S))) & 0x01010101u) << 4);
        return q2_magic4(t, q2_lo(sm), q2_hi(sm));
    }
    Q2_FRAG
};

// Q6_K: 16 int8 sub-block scales (one per 16 k); the high bit pairs of both chunks share bytes
template <int MK>
struct Q2B<MXQ_Q6_K, MK> {
    using L = Q2Lane<MK>;
    u32x4 sc;
    uint32_t dw;
    u32x2 v[L::NC], vh;  // (MK 32: vh moved down to the lane's chunk)
    int l8;              // MK 32: the lane's chunk
    f16x2 s2;
    MX_DEV void load_hdr(const char* hb, int c, int l) {
        sc = *(const u32x4*)(hb + c * 16);
        dw = *(const uint32_t*)(hb + 512 + c * 4);
        l8 = l;
    }
    MX_DEV void load_q(const char* qb, int c, int l) {
        L::load(v, qb, c, l);
        vh = *(const u32x2*)(qb + 1024 + c * 16 + 8 * L::half(l));
        if constexpr (MK == 32) vh = vh >> (2 * (l & 1));
    }
    template <int JQ, int S>
    MX_DEV void prep() {
        const _Float16 d = __builtin_bit_cast(f16x2, dw)[0];
        const int b = (int)(int8_t)((sc[JQ] >> L::byte16(S, l8)) & 0xFF);
        const _Float16 s = d * (_Float16)b;  // 11 x 8 bits: exact product, one f16 rounding
        s2 = (f16x2){s, s};
    }
    template <int JQ, int S, int H>
    MX_DEV u32x2 half() const {
        const uint32_t t = ((v[L::ch(S)][H] >> (4 * L::nib(S))) & 0x0F0F0F0Fu) |
                           (((vh[H] >> (MK == 16 ? 2 * S : 4 * S)) & 0x03030303u) << 4);
        return q2_magic4(t, (_Float16)1056.f, s2);  // 1024 magic + 32 code offset
    }
    Q2_FRAG
};

// Q3_K: code c = 2-bit field | hmask bit << 2 in [0, 7], weight = d * (sc - 32) * (c - 4). k-tile JQ: qs half
// JQ >> 1, 2-bit field j = 2 (JQ & 1) + nibble, a sub-block scale per 16 k
template <int MK>
struct Q2B<MXQ_Q3_K, MK> {
    using L = Q2Lane<MK>;
    u32x4 hd;  // scales[12] (3 words) + d
    u32x2 hm[L::NC], v[L::NC];
    int l8;
    f16x2 s2;
    MX_DEV void load_hdr(const char* hb, int c, int l) {
        hd = *(const u32x4*)(hb + c * 16);
        L::load(hm, hb + 512, c, l);
        l8 = l;
    }
    MX_DEV void load_q(const char* qb, int c, int l) { L::load(v, qb, c, l); }
    template <int JQ, int S>
    MX_DEV void prep() {
        // 16 6-bit scales from 12 bytes (ggml kmask unpack): word JQ of the unpacked array = scales 4 JQ .. 4 JQ + 3
        constexpr uint32_t km1 = 0x03030303u, km2 = 0x0F0F0F0Fu;
        uint32_t w;
        if constexpr (JQ == 0) w = (hd[0] & km2) | ((hd[2] & km1) << 4);
        else if constexpr (JQ == 1) w = (hd[1] & km2) | (((hd[2] >> 2) & km1) << 4);
        else if constexpr (JQ == 2) w = ((hd[0] >> 4) & km2) | (((hd[2] >> 4) & km1) << 4);
        else w = ((hd[1] >> 4) & km2) | (((hd[2] >> 6) & km1) << 4);
        const uint32_t w3 = hd[3];  // scalar first (see Q4_K prep)
        const _Float16 d = __builtin_bit_cast(f16x2, w3)[0];
        const int b = (int)((w >> L::byte16(S, l8)) & 0xFF) - 32;
        const _Float16 s = d * (_Float16)b;  // 11 x 6 bits: exact product, one f16 rounding
        s2 = (f16x2){s, s};
    }
    template <int JQ, int S, int H>
    MX_DEV u32x2 half() const {
        constexpr int j = 2 * (JQ & 1) + L::nib(S), hb = 4 * (JQ >> 1) + j;
        const uint32_t t =
            ((v[L::ch(S)][H] >> (2 * j)) & 0x03030303u) | (((hm[L::ch(S)][H] >> hb) & 0x01010101u) << 2);
        return q2_magic4(t, (_Float16)1028.f, s2);  // 1024 magic + 4 code offset
    }
    Q2_FRAG
};

// Q2_K: weight = d * (sc & 15) * q - dmin * (sc >> 4), fields and sub-blocks as Q3_K
template <int MK>
struct Q2B<MXQ_Q2_K, MK> {
    using L = Q2Lane<MK>;
    u32x4 sc;
    uint32_t dw;
    u32x2 v[L::NC];
    int l8;
    f16x2 sm;
    MX_DEV void load_hdr(const char* hb, int c, int l) {
        sc = *(const u32x4*)(hb + c * 16);
        dw = *(const uint32_t*)(hb + 512 + c * 4);
        l8 = l;
    }
    MX_DEV void load_q(const char* qb, int c, int l) { L::load(v, qb, c, l); }
    template <int JQ, int S>
    MX_DEV void prep() {
        const f16x2 dd = __builtin_bit_cast(f16x2, dw);
        const f16x2 dn = {dd[0], -dd[1]};
        const uint32_t b = (sc[JQ] >> L::byte16(S, l8)) & 0xFF;
        const f16x2 q = {(_Float16)(int)(b & 15), (_Float16)(int)(b >> 4)};
        sm = dn * q;  // exact f16 products (11 x 4 bits)
    }
    template <int JQ, int S, int H>
    MX_DEV u32x2 half() const {
        constexpr int sh = 2 * (2 * (JQ & 1) + L::nib(S));
        return q2_affine4((v[L::ch(S)][H] >> sh) & 0x03030303u, q2_lo(sm), q2_hi(sm));
    }
    Q2_FRAG
};

// MX4F / MX5F: weight = s * code + m per 32 (f16 s, m); code = nibble (| bit 4 from the k-tile's high-bit word)
template <bool FIVE, int MK>
struct Q2BMX {
    using L = Q2Lane<MK>;
    u32x4 h0, h1;  // header halves (k-tiles 0-1 / 2-3): {s[4], m[4]} of the half's 4 blocks of 32
    u32x2 v[L::NC];
    u32x2 vh;      // high-bit words moved down to the lane's k
    f16x2 s2, m2;
    MX_DEV void load_hdr(const char* hb, int c, int) {
        h0 = *(const u32x4*)(hb + c * 16);
        h1 = *(const u32x4*)(hb + 512 + c * 16);
    }
    MX_DEV void load_q(const char* qb, int c, int l) {
        L::load(v, qb, c, l);
        if constexpr (FIVE) vh = *(const u32x2*)(qb + 1024 + c * 8) >> (8 * L::half(l) + (MK == 32 ? 16 * (l & 1) : 0));
    }
    template <int JQ, int S>
    MX_DEV void prep() {
        if constexpr (L::fresh(S)) {
            // blocks 2 (JQ & 1), + 1 of the half: word JQ & 1 of the scale pairs, word 2 + (JQ & 1) of the offsets
            const u32x4 hh = (JQ >> 1) ? h1 : h0;
            const uint32_t sw = hh[JQ & 1], mw = hh[2 + (JQ & 1)];
            const f16x2 sv = __builtin_bit_cast(f16x2, sw), mv = __builtin_bit_cast(f16x2, mw);
            s2 = L::nib(S) ? q2_hi(sv) : q2_lo(sv);
            m2 = L::nib(S) ? q2_hi(mv) : q2_lo(mv);
        }
    }
    template <int JQ, int S, int H>
    MX_DEV u32x2 half() const {
        const uint32_t t = (v[L::ch(S)][H] >> (4 * L::nib(S))) & 0x0F0F0F0Fu;
        if constexpr (FIVE) return q2_magic4(t | (mx_spread4(vh[L::nib(S)] >> (16 * L::ch(S) + 4 * H)) << 4), s2, m2);
        return q2_affine4(t, s2, m2);
    }
    Q2_FRAG
};
template <int MK>
struct Q2B<MXQ_MX4F, MK> : Q2BMX<false, MK> {};
template <int MK>
struct Q2B<MXQ_MX5F, MK> : Q2BMX<true, MK> {};

// Q8_0: weight = d * int8 code per 32; a pair of code chunks per nibble of the others
template <int MK>
struct Q2B<MXQ_Q8_0, MK> {
    using L = Q2Lane<MK>;
    u32x2 qv[2][L::NC];
    uint32_t dw;
    f16x2 s2;
    MX_DEV void load_hdr(const char*, int, int) {}
    MX_DEV void load_q(const char* qb, int c, int l) {
        dw = *(const uint32_t*)(qb + c * 4);
        L::load(qv[0], qb + 128, c, l);
        L::load(qv[1], qb + 128 + 1024, c, l);
    }
    template <int JQ, int S>
    MX_DEV void prep() {
        if constexpr (L::fresh(S)) {
            const f16x2 dd = __builtin_bit_cast(f16x2, dw);
            s2 = L::nib(S) ? q2_hi(dd) : q2_lo(dd);
        }
    }
    template <int JQ, int S, int H>
    MX_DEV u32x2 half() const {
        // int8 -> u8 + 128; 1024 magic + 128
        return q2_magic4(qv[L::nib(S)][L::ch(S)][H] ^ 0x80808080u, (_Float16)1152.f, s2);
    }
    Q2_FRAG
};
#undef Q2_FRAG

// LDS-DMA of one 32-column group's weight bytes for k-tile JQ of a super-block (unit `u`): the tile's quant bytes
// (F::QB: whole 1 KB pieces plus one partial piece, F::QI instructions) into `qd` and, with the super-block's first
// tile, its header (F::HB bytes in the format's layout, F::HI instructions) into `hd`.
// `u` is uniform over the wave, qd and hd are LDS addresses.
template <int QT, int JQ>
MX_DEV void q2_stage_weights(const uint8_t* u, uint32_t qd, uint32_t hd, int lane) {
    using F = Q2F<QT>;
    const uint8_t* qs = u + F::qoff(JQ);
    constexpr int NF = F::QB / 1024, REM = F::QB % 1024;
    static_assert(NF + (REM ? 1 : 0) == F::QI && REM % 16 == 0, "quant piece count");
#pragma unroll
    for (int i = 0; i < NF; ++i) mx_lds_dma16(qs + i * 1024, lane * 16, qd + i * 1024);
    if constexpr (REM > 0) {
        if (lane < REM / 16) mx_lds_dma16(qs + NF * 1024, lane * 16, qd + NF * 1024);
    }
    if constexpr (JQ == 0) {
        if constexpr (QT == MXQ_Q3_K) {  // hdr (512 B) + hmask (1 KB): one full and one half instruction
            mx_lds_dma16(u, lane * 16, hd);
            if (lane < 32) mx_lds_dma16(u + 1024, lane * 16, hd + 1024);
        } else if constexpr (QT == MXQ_MX4F || QT == MXQ_MX5F) {  // both header halves (1 KB)
            mx_lds_dma16(u, lane * 16, hd);
        } else if constexpr (F::HB > 0) {
            if (lane < 32) mx_lds_dma16(u, lane * 16, hd);
            if constexpr (QT == MXQ_Q6_K || QT == MXQ_Q2_K) {  // + the 32 x 4 B d (/ dmin) words
                if (lane < 32) mx_lds_dma4(u + 512, lane * 4, hd + 512);
            }
            if constexpr (QT == MXQ_Q5_K)  // + the qh chunks (fifth bits of the whole super-block)
                mx_lds_dma16(u + F::QH, lane * 16, hd + 512);
        }
    }
}

}  // namespace
