// hybrid_scan.hip: the linear recurrence of gated-delta-rule and state-space (duality form) layers (ops/hybrid.py
// state_scan). Per sequence and head, over the step's rows in order:
//     S <- a_t S;   u = c_t (v_t - S^T k_t)  [delta]   or   u = c_t v_t;   S <- S + k_t u^T;   o_t = S^T q_t (+ D v_t)
// S has N numbers for each of the head's P value columns, fp32, stored column-major: state [slots, H, P, N]. The
// columns never mix, so a column belongs to LPC neighbouring lanes (4, or the 16 of one DPP row or the 32 of two) that each keep NPL of its
// numbers (every LPC-th quadruple) in registers for the whole chunk. k_t and q_t are the same for every column of a head: the
// block stages them in LDS together with the tokens' decays, write strengths and values, 8 or 16 tokens at a time in two
// buffers; the next tokens' numbers are requested from memory before the current ones are worked on and wait in registers
// meanwhile, so memory latency and the barrier are paid once per 8 or 16 steps. The state is read from the sequence's slot
// unless the chunk starts at position 0, and written back after the chunk's last row: a decode row is a chunk of one, a
// prompt chunk walks its rows inside one launch.
// What bounds a prompt is the issue of a step's instructions by the few waves its columns make (1111 rows, 16 heads of 128 x
// 128: 128 blocks; a step is 32 vector operations a lane and a chain of two sums): the read S^T k uses the undecayed state
// (its decay is multiplied in after the sum), a step's LDS reads are asked for a step ahead, and output sums over a column's
// lanes are made for 8 or 16 steps together, transposed on the way (3 operations a step instead of a chain of 4 and a store).
// Prompts of 301 / 578 / 1111 rows: delta rule 576 -> 250 us, 64 heads of 64 x 128 without it 554 -> 227 (most of the gain is that a
// round's loads no longer wait for each other); with whole rounds free of tests between their steps and the staged numbers' scales and
// masks worked out once (a step 36 instructions for some 65, the delta rule's 58 for 90) 262 -> 217 and 247 -> 201, one of 2900 rows
// 644 -> 512 and 533 -> 390. Steps read two or more ahead change nothing: one wave a SIMD issues a vector instruction every 9 cycles.
// Decode rows and short chunks (ONE) stage one token and sum at once: 33 rows 18.0 -> 12.6 and 30.3 -> 22.2 us (6.2 TB/s of states read
// and written).
// CHD (gated linear attention): the decay is one number per head and state row, a_t[n], staged beside k_t and q_t:
// S[n][p] <- a_t[n] S[n][p] + k_t[n] u[p]; with DELTA as well, the delta rule's read follows that per-row decay. A
// missing write strength means 1, one given as pre-activations (coef_sigmoid, row stride ldc) passes a sigmoid when
// staged; q_t is multiplied by q_scale when staged. A decay row stride of 0 (ldd) is one constant per head for every
// token (retention).
// nout: the state has one more column per head (P + 1 of them) whose value is 1 at every token, so it holds
// n <- a_t n + c_t k_t; its product n^T q_t goes to nout [rows, H] (the normaliser of a matrix memory).
#include "../mx_common.h"

#include <type_traits>

namespace {

template <int CTRL>
MX_DEV float dpp_add(float v) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
MX_DEV float dpp_move(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
// sum over the DPP rows 2 r and 2 r + 1 (32 lanes), lane by lane, returned to both
MX_DEV float row_pair_sum(float v) {
    const u32x2 x = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false));
    return __uint_as_float(x[0]) + __uint_as_float(x[1]);
}
// sum over the LPC (4, 16 or 32) neighbouring lanes of a column, returned to each of them
template <int LPC>
MX_DEV float lanes_sum(float v) {
    v = dpp_add<0xB1>(v);  // quad_perm [1, 0, 3, 2]
    v = dpp_add<0x4E>(v);  // quad_perm [2, 3, 0, 1]
    if constexpr (LPC >= 16) {
        v = dpp_add<0x124>(v);  // row_ror 4
        v = dpp_add<0x128>(v);  // row_ror 8
    }
    if constexpr (LPC == 32) v = row_pair_sum(v);
    return v;
}

MX_DEV float chains_sum(const float (&c)[1]) { return c[0]; }
MX_DEV float chains_sum(const float (&c)[2]) { return c[0] + c[1]; }
MX_DEV float chains_sum(const float (&c)[4]) { return (c[0] + c[1]) + (c[2] + c[3]); }

// what a round of tokens is: one token; up to TB with a test between steps; or whole rounds in a body of their own without that test
enum { ROUND_ONE = 0, ROUND_ANY = 1, ROUND_WHOLE = 2 };

// grid (column blocks, H, sequences from s0 on); block = 256 threads (512 of 32 lanes a column) = 256 / LPC (16) columns
template <int NPL, int LPC, bool DELTA, bool CHD, int ROUND>
__global__ __launch_bounds__(LPC == 32 ? 512 : 256) void state_scan_kernel(const float* k, int ldk, const float* q, int ldq,
                                                         const float* v, int ldv, const float* decay, int ldd,
                                                         const float* coef, int ldc, int coef_sigmoid,
                                                         const float* skip, float* state, const int* seq_state,
                                                         const int* positions, int n_dec, const int* pf_cu, float* out,
                                                         int ldo, int H, int G, int N, int P, float q_scale,
                                                         float* nout, int s0, int n_pf, int rows_pf) {
    static_assert(LPC == 4 || LPC == 16 || LPC == 32, "a column's lanes are a quad, a DPP row or two");
    constexpr bool ONE = ROUND == ROUND_ONE;
    constexpr int NT = LPC == 32 ? 512 : 256;
    constexpr int NP = NPL * LPC;  // padded N
    constexpr int COLS = NT / LPC;
    constexpr int TB = ONE ? 1 : NP <= 128 ? 16 : 8;  // tokens staged together
    constexpr int NW = CHD ? 3 : 2;  // vectors of N numbers staged per token: k, q (, channel decays)
    constexpr int KQ_PT = (TB * NW * NP + NT - 1) / NT, V_PT = (TB * COLS + NT - 1) / NT;
    __shared__ __attribute__((aligned(16))) float kq[2][TB][NW][NP];
    __shared__ float vs[2][TB][COLS];
    __shared__ __attribute__((aligned(8))) float ac[2][TB][2];
    const int cl = threadIdx.x / LPC;
    const int col = blockIdx.x * COLS + cl;
    const int part = threadIdx.x % LPC;
    const int h = blockIdx.y, s = s0 + blockIdx.z;
    int row0, n;
    if (s < n_dec) {
        row0 = s;
        n = 1;
    } else {
        const int i = s - n_dec;
        row0 = n_dec + pf_cu[i];
        n = pf_cu[i + 1] - pf_cu[i];
    }
    if (n <= 0) return;
    // the longest chunks end the launch, so chunks above the mean issue before the others' waves of a SIMD: 301 / 578 / 1111 rows, 16 heads of 128 x 128
    // with the delta rule 202 -> 177 us, 64 of 128 x 64 without 184 -> 169
    if constexpr (!ONE) {
        if ((long)n * n_pf > rows_pf) __builtin_amdgcn_s_setprio(2);
    }
    const int slot = seq_state[s];
    const bool fresh = positions[row0] == 0 || slot < 0;
    const int PT = P + (nout ? 1 : 0);  // state columns of a head
    const bool live = col < PT;
    const int g = h / (H / G);
    // addresses are clamped so that every load below is unconditional (all in flight together); what a lane must not
    // use is replaced by zero afterwards
    const int colc = min(col, PT - 1);
    float* sp = state + (((long)(slot < 0 ? 0 : slot) * H + h) * PT + colc) * N;
    const bool whole = N == NP && (N & 3) == 0;  // no padding: a lane's numbers are NPL / 4 aligned quadruples
    auto at = [&](int j) { return (j >> 2) * (4 * LPC) + part * 4 + (j & 3); };  // which number of the column S[j] is
    float S[NPL];
    if (whole) {
        const f32x4* s4 = (const f32x4*)sp + part;
#pragma unroll
        for (int j = 0; j < NPL / 4; ++j) {
            const f32x4 x = s4[j * LPC];  // (as a vector: as four numbers the compiler joins them with the other branch's single loads)
            S[4 * j] = x[0];
            S[4 * j + 1] = x[1];
            S[4 * j + 2] = x[2];
            S[4 * j + 3] = x[3];
        }
    } else {
#pragma unroll
        for (int j = 0; j < NPL; ++j) S[j] = sp[min(at(j), N - 1)];
    }
    const bool keep = !fresh && live;
#pragma unroll
    for (int j = 0; j < NPL; ++j) S[j] = (keep && at(j) < N) ? S[j] : 0.f;
    const float* kp = k + (long)g * N;
    const float* qp = q + (long)g * N;
    const float sk = skip ? skip[h] : 0.f;
    const int last = row0 + n - 1;
    // TB tokens' k, q, value, decay and write strength wait in registers while the TB tokens before them are worked
    // on, then move to LDS: memory latency is paid once per TB steps, and a barrier too
    float st_kq[KQ_PT], st_v[V_PT], st_ac = 0.f;
    // a round's loads are unconditional (one load from a selected, clamped address; scaled, masked and squashed when they
    // move to LDS) so that all are in flight together; whole groups of NT loads beyond the round's tokens are skipped by a
    // block-uniform test: a decode row asks for one token's numbers, not TB copies of them
    auto fetch = [&](int c) {
        const int r0 = row0 + c * TB;
        const int ntc = min(TB, n - c * TB);
#pragma unroll
        for (int i = 0; i < KQ_PT; ++i) {
            const int idx = ONE ? min((int)threadIdx.x + i * NT, TB * NW * NP - 1) : threadIdx.x + i * NT;
            if (i * NT < ntc * NW * NP) {
                const int tt = idx / (NW * NP), w = (idx / NP) % NW;
                const long row = min(r0 + tt, last);
                const float* src = CHD && w == 2 ? decay + (long)h * N : w ? qp : kp;
                const long ld = CHD && w == 2 ? (long)H * N : w ? ldq : ldk;
                st_kq[i] = src[row * ld + min(idx % NP, N - 1)];
            }
        }
#pragma unroll
        for (int i = 0; i < V_PT; ++i) {
            if (i * NT < ntc * COLS) {
                const int idx = min(threadIdx.x + i * NT, TB * COLS - 1);
                const int tt = idx / COLS, cc = idx % COLS;
                const long row = min(r0 + tt, last);
                st_v[i] = v[row * ldv + (long)h * P + min((int)blockIdx.x * COLS + cc, P - 1)];
            }
        }
        if (threadIdx.x < 2 * TB) {
            const long row = min(r0 + (int)threadIdx.x / 2, last);
            const bool cf = threadIdx.x & 1;
            // (what has no source reads the decay and is replaced)
            const float* src = cf && coef ? coef + row * ldc + h : decay + (CHD ? row * ((long)H * N) + (long)h * N : row * ldd + h);
            st_ac = *src;
        }
    };
    // which vector and number of it, and which column, a thread stages: the same in every group where groups are whole tokens. (With channel decays
    // they are not, and an entry for each of up to 24 groups took so many registers that one block ran on a compute unit for two: 30 chunks of 250
    // rows, 32 heads of 128 x 128 1081 -> 1704 us. There they are worked out where they are needed.)
    constexpr bool SAME = !ONE && NT % (NW * NP) == 0;
    constexpr int VC = NT % COLS ? V_PT : 1;
    const float st_mul = (threadIdx.x / NP) % NW == 1 ? q_scale : 1.f;
    const bool st_on = threadIdx.x % NP < N;
    int st_col[VC];
#pragma unroll
    for (int i = 0; i < VC; ++i) st_col[i] = blockIdx.x * COLS + (threadIdx.x + i * NT) % COLS;
    auto publish = [&](int b) {
#pragma unroll
        for (int i = 0; i < KQ_PT; ++i) {
            const int idx = threadIdx.x + i * NT;
            if (ONE && idx >= TB * NW * NP) continue;
            if constexpr (SAME) (&kq[b][0][0][0])[idx] = st_on ? st_kq[i] * st_mul : 0.f;
            else (&kq[b][0][0][0])[idx] = idx % NP < N ? ((idx / NP) % NW == 1 ? st_kq[i] * q_scale : st_kq[i]) : 0.f;
        }
#pragma unroll
        for (int i = 0; i < V_PT; ++i)
            if (threadIdx.x + i * NT < TB * COLS) (&vs[b][0][0])[threadIdx.x + i * NT] = ONE || st_col[i % VC] < P ? st_v[i] : st_col[i % VC] < PT ? 1.f : 0.f;
        if (threadIdx.x < 2 * TB) {
            float x = st_ac;
            if (threadIdx.x & 1) x = !coef ? 1.f : coef_sigmoid ? 1.f / (1.f + expf(-x)) : x;
            else if (CHD) x = 1.f;
            (&ac[b][0][0])[threadIdx.x] = x;
        }
    };
#pragma unroll
    for (int i = 0; i < KQ_PT; ++i) st_kq[i] = 0.f;  // (tokens past the end are staged as zeros and not worked on)
#pragma unroll
    for (int i = 0; i < V_PT; ++i) st_v[i] = 0.f;
    const int nchunks = (n + TB - 1) / TB;
    fetch(0);
    publish(0);
    __syncthreads();
    for (int c = 0; c < nchunks; ++c) {
        const int b = c & 1;
        if (c + 1 < nchunks) fetch(c + 1);
        const int nt = min(TB, n - c * TB);
        // a step leaves the lane's share of its output (and of the skip term's value) here: they are summed over the
        // column's lanes TB at a time
        float os[TB];
        // a step's numbers are read from LDS while the step before it is worked on
        struct Tok {
            float k[NPL], q[NPL], d[CHD ? NPL : 1], a, cf, v;
        } tok[2];
        auto read = [&](int tt, Tok& x) {
            const float2 y = *(const float2*)ac[b][tt];
            x.a = y.x;
            x.cf = y.y;
            x.v = vs[b][tt][cl];
#pragma unroll
            for (int j = 0; j < NPL; j += 4) {
                *(float4*)(x.k + j) = *(const float4*)&kq[b][tt][0][j * LPC + part * 4];
                *(float4*)(x.q + j) = *(const float4*)&kq[b][tt][1][j * LPC + part * 4];
                if constexpr (CHD) *(float4*)(x.d + j) = *(const float4*)&kq[b][tt][NW - 1][j * LPC + part * 4];
            }
        };
        // a lane's products are summed in chains of four (quads of lanes: in four chains, 2 % slower)
        constexpr int NC = LPC == 4 ? 4 : NPL / 4;
        auto chain = [](int j) { return LPC == 4 ? j & 3 : j >> 2; };
        auto head = [](int j) { return LPC == 4 ? j & 3 : j & ~3; };  // the first of j's chain
        // whole rounds without a test between steps: those cost nine register moves a step beside the branch
        auto steps = [&](auto whole_c) {
            constexpr bool ALL = decltype(whole_c)::value;
            read(0, tok[0]);
#pragma unroll
            for (int tt = 0; tt < TB; ++tt) {
                os[tt] = 0.f;
                if (tt + 1 < TB && (ALL || tt + 1 < nt)) read(tt + 1, tok[(tt + 1) & 1]);
                __builtin_amdgcn_sched_barrier(0);
                if (!ALL && tt >= nt) continue;
                const Tok& x = tok[tt & 1];
                const float a = x.a, cf = x.cf, vv = !ONE || col < P ? x.v : live ? 1.f : 0.f;
                const float *kb = x.k, *qb = x.q, *ab = x.d;
                float u;
                if constexpr (DELTA) {
                    if constexpr (CHD) {
#pragma unroll
                        for (int j = 0; j < NPL; ++j) S[j] *= ab[j];
                    }
                    float d[NC];
#pragma unroll
                    for (int j = 0; j < NPL; ++j) d[chain(j)] = j != head(j) ? fmaf(S[j], kb[j], d[chain(j)]) : S[j] * kb[j];
                    const float dk = lanes_sum<LPC>(chains_sum(d));
                    u = cf * (CHD ? vv - dk : vv - a * dk);  // (one decay for all rows: taken out of the sum)
                } else {
                    u = cf * vv;
                }
                float o[NC];
#pragma unroll
                for (int j = 0; j < NPL; ++j) {
                    if constexpr (!(DELTA && CHD)) S[j] *= CHD ? ab[CHD ? j : 0] : a;
                    S[j] += kb[j] * u;
                    o[chain(j)] = j != head(j) ? fmaf(S[j], qb[j], o[chain(j)]) : S[j] * qb[j];
                }
                os[tt] = chains_sum(o);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        if constexpr (ONE) steps(std::true_type{});
        else if (ROUND == ROUND_WHOLE && nt == TB) steps(std::true_type{});
        else steps(std::false_type{});
        auto put = [&](int tt, float o) {
            if (tt >= nt || !live) return;
            const long row = row0 + c * TB + tt;
            if (col < P) out[row * ldo + (long)h * P + col] = o + sk * vs[b][tt][cl];
            else nout[row * H + h] = o;
        };
        // sums over the lanes of a column, transposed on the way: lane `part` ends with steps part, part + LPC, ...
        float o4[ONE ? 1 : TB / 4];
#pragma unroll
        for (int j = 0; j < TB / 4; ++j) {
            const float a0 = part & 1 ? os[4 * j + 1] : os[4 * j], b0 = part & 1 ? os[4 * j] : os[4 * j + 1];
            const float a1 = part & 1 ? os[4 * j + 3] : os[4 * j + 2], b1 = part & 1 ? os[4 * j + 2] : os[4 * j + 3];
            const float e0 = a0 + dpp_move<0xB1>(b0), e1 = a1 + dpp_move<0xB1>(b1);  // quad_perm [1, 0, 3, 2]
            const float f0 = part & 2 ? e1 : e0, f1 = part & 2 ? e0 : e1;
            o4[j] = f0 + dpp_move<0x4E>(f1);                                          // quad_perm [2, 3, 0, 1]
            if constexpr (LPC >= 16) {
                o4[j] = dpp_add<0x124>(o4[j]);  // row_ror 4
                o4[j] = dpp_add<0x128>(o4[j]);  // row_ror 8
            }
        }
        if constexpr (ONE) {
            const float o = lanes_sum<LPC>(os[0]);
            if (part == 0) put(0, o);
        } else if constexpr (LPC >= 16) {
            float o = o4[0];
#pragma unroll
            for (int j = 1; j < TB / 4; ++j) o = (part >> 2 & 3) == j ? o4[j] : o;
            if constexpr (LPC == 32) o = row_pair_sum(o);
            if (part < 16) put(part, o);
        } else {
#pragma unroll
            for (int j = 0; j < TB / 4; ++j) put(4 * j + part, o4[j]);
        }
        // the other buffer was last read while chunk c - 1 was worked on, before the barrier that ended that round
        if (c + 1 < nchunks) publish(b ^ 1);
        __syncthreads();
    }
    if (slot >= 0 && live) {
        if (whole) {
            float4* s4 = (float4*)sp + part;
#pragma unroll
            for (int j = 0; j < NPL / 4; ++j) s4[j * LPC] = make_float4(S[4 * j], S[4 * j + 1], S[4 * j + 2], S[4 * j + 3]);
        } else {
#pragma unroll
            for (int j = 0; j < NPL; ++j)
                if (at(j) < N) sp[at(j)] = S[j];
        }
    }
}

// Scales of an exponentially gated matrix memory (ops/hybrid.py mlstm_gates). Per sequence and head, over the step's rows:
//     i = cap tanh((zi + bi) / cap),  f = log sigmoid(cap tanh((zf + bf) / cap)),  m_t = max(f_t + m_(t-1), i_t)
//     decay_t = exp(f_t + m_(t-1) - m_t),  coef_t = exp(i_t - m_t),  floor_t = exp(-m_t)
// The running maximum is a scan of the maps m -> max(m + A, B), which compose to maps of the same form: a block takes
// blockDim.x tokens at a time (a wave-wide prefix, the waves' totals through LDS), and every token reads its
// predecessor's m as that one computed it, so stored states and scales always refer to the same number. m starts at 0
// and is carried in peak[slot][h]. grid (H, sequences)
__global__ __launch_bounds__(1024) void mlstm_gates_kernel(const float* zi, const float* zf, int ldz, const float* bi,
                                                          const float* bf, float cap, float* peak, const int* seq_state,
                                                          const int* positions, int n_dec, const int* pf_cu,
                                                          float* decay, float* coef, float* floor_, int H) {
    __shared__ float ms[1025];  // m of the token before the round's first, then of its tokens
    __shared__ float ta[16], tb[16];  // a wave's 64 maps composed
    const int h = blockIdx.x, s = blockIdx.y, nt = blockDim.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int row0, n;
    if (s < n_dec) {
        row0 = s;
        n = 1;
    } else {
        const int k = s - n_dec;
        row0 = n_dec + pf_cu[k];
        n = pf_cu[k + 1] - pf_cu[k];
    }
    if (n <= 0) return;
    const int slot = seq_state[s];
    const bool fresh = positions[row0] == 0 || slot < 0;
    float m0 = fresh ? 0.f : peak[(long)slot * H + h];
    const float b0 = bi ? bi[h] : 0.f, b1 = bf ? bf[h] : 0.f;
    for (int base = 0; base < n; base += nt) {
        const bool ok = base + tid < n;
        const long row = row0 + min(base + tid, n - 1);
        const float x = -cap * tanhf((zf[row * ldz + h] + b1) / cap);
        const float gi = cap * tanhf((zi[row * ldz + h] + b0) / cap);
        const float gf = -(x > 30.f ? x : log1pf(expf(x)));
        float A = ok ? gf : 0.f, B = ok ? gi : -INFINITY;  // past the end: the identity
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const float Ap = __shfl_up(A, o, 64), Bp = __shfl_up(B, o, 64);
            if (lane >= o) {
                B = fmaxf(Bp + A, B);
                A += Ap;
            }
        }
        if (lane == 63) {
            ta[wave] = A;
            tb[wave] = B;
        }
        if (tid == 0) ms[0] = m0;
        __syncthreads();
        float m = m0;
        for (int w = 0; w < wave; ++w) m = fmaxf(m + ta[w], tb[w]);
        m = fmaxf(m + A, B);
        ms[tid + 1] = m;
        __syncthreads();
        if (ok) {
            const long o = row * H + h;
            decay[o] = expf(gf + ms[tid] - m);
            coef[o] = expf(gi - m);
            floor_[o] = expf(-m);
        }
        m0 = ms[min(nt, n - base)];
        __syncthreads();  // (the next round writes ms and the totals)
    }
    if (slot >= 0 && tid == 0) peak[(long)slot * H + h] = m0;
}

}  // namespace

#define MXH_CHECK(cond) \
    if (!(cond)) return (int)hipErrorInvalidValue

extern "C" int mxh_state_scan(const float* k, int ldk, const float* q, int ldq, const float* v, int ldv,
                              const float* decay, int decay_rows, const float* coef, int ldc, int coef_sigmoid,
                              const float* skip, float* state, const int* seq_state, const int* positions, int n_dec,
                              const int* pf_cu, int n_pf, float* out, int ldo, int H, int G, int N, int P, int delta,
                              int channel, float q_scale, float* nout, int T, hipStream_t st) {
    const int n_seqs = n_dec + n_pf;
    if (n_seqs <= 0) return 0;
    MXH_CHECK(k && q && v && decay && state && seq_state && positions && out && (n_pf == 0 || pf_cu));
    MXH_CHECK((decay_rows || !channel) && (!coef || ldc >= H));  // decay_rows 0: one constant per head, [H]
    const int ldd = decay_rows ? H : 0;
    MXH_CHECK(H > 0 && G > 0 && H % G == 0 && N > 0 && N <= 256 && P > 0 && H <= 65535 && n_seqs <= 65535);
    MXH_CHECK(ldk >= G * N && ldq >= G * N && ldv >= H * P && ldo >= H * P);
    const int cols = N <= 32 ? 64 : 16;  // of a block
    const dim3 grid((P + (nout ? 1 : 0) + cols - 1) / cols, H, n_seqs);
    // Short prompt chunks step token by token as decode rows do (ONE): staging 8 or 16 tokens and reading them ahead costs registers,
    // which are what keeps states in flight. us, staged / one by one: 8 heads of 128 x 256 with channel decays, 64 chunks of 3
    // tokens 89 / 30, 16 of 4 26.5 / 11.4, 33 decode rows + 3 tokens 46 / 15; 16 heads of 128 x 128, one chunk of 4 tokens 4.8 / 5.0,
    // of 8 5.4 / 7.0, with channel decays 8.4 / 7.5.
    // Decode rows that fill the chip by themselves run as a launch of their own beside longer chunks: 127 rows + 64 tokens, 16 heads of
    // 128 x 128 66 -> 58 us, with channel decays 165 -> 66; few stay in the chunks' launch (8 rows + 289 tokens 70).
    const int few = N > 64 ? (!channel ? 4 : n_pf < 8 ? 12 : 16) : channel ? 4 : 3;
    const bool one = T - n_dec <= (long)few * n_pf, apart = !one && (long)grid.x * H * n_dec >= 4096;
    const dim3 grid_dec(grid.x, H, n_dec), grid_pf(grid.x, H, apart ? n_pf : n_seqs);
    // Whole rounds take a fifth less time (one chunk of 2900 rows 644 -> 512 us) and more registers, so fewer blocks run on a compute unit: chunks of
    // less than a round gain nothing (20 of 9 rows, 32 heads of 128 x 128 30.1 -> 35.0, 100 decode rows beside 18 rows in three chunks, 24 heads
    // of 32 x 32 11.9 -> 14.0), and with channel decays and N 65 to 128 one block of 16 lanes a column runs where two did, so only grids that leave it
    // alone anyway gain (one chunk of 1111 rows 277 -> 238, three of 301 to 1111 365 -> 428, 30 of 64 338 -> 523).
    const long blocks_pf = (long)grid_pf.x * H * grid_pf.z;
    // Columns over 32 lanes in blocks of 512 threads: twice the waves with fewer instructions each, since a wave alone on its SIMD issues one
    // in nine cycles. It wins until the chunks' blocks bring more than two such waves to a SIMD. us, 16 / 32 lanes: one chunk of 1111 rows, 16 heads of 128 x
    // 128 with the delta rule 190 / 168, without 149 / 110, with channel decays 231 / 192 and 189 / 145; three of 301 to 1111, delta rule 199 / 189 (384
    // blocks), 64 heads of 128 x 64 without 173 / 166, with it 223 / 244 (768 blocks; these before chunks had priorities); four of 200, 16 heads of 128 x 128 (512 blocks) 45.4 / 50.7 and 35.0 /
    // 35.5, with channel decays 64.9 / 77.7 and 55.6 / 60.7. N above 128 always: 16 numbers a lane leave one block a compute unit (8 heads of 256 x 256, one
    // chunk of 1111 328 / 271, 30 of 64 rows with channel decays 443 / 336, eight of 250 without 182 / 186).
    const bool wide = N > 128 || (N > 64 && (long)grid.x * H * n_pf <= (delta || channel ? 384 : 768));
    const bool full = T - n_dec >= 16l * n_pf, whole = full && !(channel && blocks_pf > 256);
#define GO(NPL, LPC)                              \
    do {                                          \
        if (delta && channel) GO2(NPL, LPC, true, true); \
        else if (delta) GO2(NPL, LPC, true, false);   \
        else if (channel) GO2(NPL, LPC, false, true); \
        else GO2(NPL, LPC, false, false);         \
    } while (0)
#define GO2(NPL, LPC, D_, C_)                                                                          \
    do {                                                                                               \
        if (one) {                                                                                     \
            GO3(NPL, LPC, D_, C_, ROUND_ONE, grid, 0);                                                 \
            break;                                                                                     \
        }                                                                                              \
        if (apart) GO3(NPL, LPC, D_, C_, ROUND_ONE, grid_dec, 0);                                      \
        if constexpr (NPL * LPC > 64) {                                                                \
            if (NPL == 16 || wide) {                                                                   \
                if (full) GO3(NPL / 2, 32, D_, C_, ROUND_WHOLE, grid_pf, apart ? n_dec : 0);           \
                else GO3(NPL / 2, 32, D_, C_, ROUND_ANY, grid_pf, apart ? n_dec : 0);                  \
                break;                                                                                 \
            }                                                                                          \
        }                                                                                              \
        if constexpr (NPL < 16) {                                                                      \
            if (NPL * LPC > 64 ? whole : full) GO3(NPL, LPC, D_, C_, ROUND_WHOLE, grid_pf, apart ? n_dec : 0); \
            else GO3(NPL, LPC, D_, C_, ROUND_ANY, grid_pf, apart ? n_dec : 0);                         \
        }                                                                                              \
    } while (0)
#define GO3(NPL, LPC, D_, C_, O_, GRID, S0)                                                                                  \
    state_scan_kernel<NPL, LPC, D_, C_, O_><<<GRID, LPC == 32 ? 512 : 256, 0, st>>>(k, ldk, q, ldq, v, ldv, decay, ldd, coef, ldc, \
                                                                  coef_sigmoid, skip, state, seq_state, positions,    \
                                                                  n_dec, pf_cu, out, ldo, H, G, N, P, q_scale, nout, S0, n_pf, T - n_dec)
    if (N <= 16) GO(4, 4);
    else if (N <= 32) GO(8, 4);
    else if (N <= 64) GO(4, 16);
    else if (N <= 128) GO(8, 16);
    else GO(16, 16);
#undef GO
#undef GO2
#undef GO3
    return (int)hipGetLastError();
}

extern "C" int mxh_mlstm_gates(const float* zi, const float* zf, int ldz, const float* bi, const float* bf, float cap,
                               float* peak, const int* seq_state, const int* positions, int n_dec, const int* pf_cu,
                               int n_pf, float* decay, float* coef, float* floor_, int H, int T, hipStream_t st) {
    const int n_seqs = n_dec + n_pf;
    if (n_seqs <= 0) return 0;
    MXH_CHECK(zi && zf && peak && seq_state && positions && decay && coef && floor_ && (n_pf == 0 || pf_cu));
    MXH_CHECK(H > 0 && ldz >= H && cap > 0.f && n_seqs <= 65535);
    const int nt = n_pf ? min(1024, (max(T - n_dec, 1) + 63) / 64 * 64) : 64;  // a prompt chunk of up to 1024 rows in one round
    mlstm_gates_kernel<<<dim3(H, n_seqs), nt, 0, st>>>(zi, zf, ldz, bi, bf, cap, peak, seq_state, positions, n_dec, pf_cu,
                                                       decay, coef, floor_, H);
    return (int)hipGetLastError();
}
