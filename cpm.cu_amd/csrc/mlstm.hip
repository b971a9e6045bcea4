// The matrix-memory recurrence of the mLSTM kind, per head with key size d and value size dv:
//
//   a_t = cap tanh((i_t + bi) / cap)                     log input gate
//   b_t = logsigmoid(cap tanh((f_t + bf) / cap))         log forget gate
//   m_t = max(b_t + m_(t-1), a_t)                        running maximum, 0 before the first token
//   S_t = exp(b_t + m_(t-1) - m_t) S_(t-1) + exp(a_t - m_t) k_t v_t^T          S: [d, dv], zero at the start
//   n_t = exp(b_t + m_(t-1) - m_t) n_(t-1) + exp(a_t - m_t) k_t
//   y_t = S_t^T q_t / (max(|n_t . q_t|, exp(-m_t)) + 1e-6)
//
// q, k, v and the raw gates i, f are columns of one projection (q is multiplied by `q_scale` as it is read);
// gates, decays, the state and the output are float.  The kernel leaves S_t^T q_t and the denominator side by side;
// the head norm that follows divides.  S, n and m live per cache slot and are carried from step to
// step, so a step of any number of tokens continues where the last one ended.
#include "common.h"
#include "runs.h"
#include "vec4.h"

// A workgroup of 256 threads walks ML_PB = 256 / ML_L columns; a column's d state values lie over ML_L neighbouring
// lanes (8 or 32: key index c = l + ML_L i), which sum their shares inside the vector unit.  Keys beyond 128
// features take 32 lanes a column: four times the workgroups (several a CU, whose walks hide each other's waits)
// and a quarter of the chain of dependent steps a token.

__device__ inline float log_sigmoid_f(float v) { return fminf(v, 0.f) - log1pf(expf(-fabsf(v))); }

// grid (sequences x heads, ceil((dv + 1) / ML_PB)), 256 threads: a sequence's workgroups are dealt to all XCDs, also where
// one sequence of a step is much longer than the others.  The launch takes the sequences of lo <= tokens < hi (runs.h).  proj: [n, ld]; q at column q_off + h * d, k at
// k_off + h * d, v at v_off + h * dv, raw gates at i_off + h and f_off + h.  S: [slots][heads][dv][d],
// nst: [slots][heads][d], mst: [slots][heads].
//
// Every workgroup of a (sequence, head) starts from its slot's maximum, and a launch may have more of them than run at a
// time: none may write it.  The maximum behind the step goes to m_next [sequences][heads], which mlstm_maximum_kernel, a
// launch of its own, moves to the slots.
//
// The normaliser n obeys the recurrence of a column of S whose value is always 1, so it is walked as column dv:
// columns 0 .. dv - 1 give the unnormalised y = S^T q (float [n, heads * dv]) and column dv gives n . q, from which
// den[t, h] = max(|n . q|, exp(-m)) + 1e-6 (float [n, heads]); whoever reads y divides by den (the head norm does).
// Tiles of ML_TT tokens pass through LDS; the running maximum of a tile is walked by one thread first (additions and
// maxima only), then the tile's exponentials are formed side by side, so the walk over the state itself holds
// nothing but multiply-adds.
template <int NR, int ML_L, int ML_TT, typename T>
__global__ __launch_bounds__(256) void mlstm_scan_kernel(const T* __restrict__ proj, long ld, long q_off, long k_off,
                                                         long v_off, long i_off, long f_off,
                                                         const float* __restrict__ i_bias,
                                                         const float* __restrict__ f_bias, float cap, float q_scale,
                                                         float* __restrict__ S_state, float* __restrict__ n_state,
                                                         const float* __restrict__ m_state, float* __restrict__ m_next,
                                                         float* __restrict__ y,
                                                         float* __restrict__ den, const int* __restrict__ cu_q,
                                                         const int* __restrict__ seq_slot, int heads, int d, int dv,
                                                         int write_state, int n_seqs, int lo, int hi) {
    constexpr int ML_PB = 256 / ML_L;               // columns a workgroup
    constexpr int NS = NR * ML_L;                   // key features, padded
    constexpr int QK = ML_TT * NS / 256;            // q (and k) values a thread brings a tile
    constexpr int XV = (ML_TT * ML_PB + 255) / 256;   // v values a thread brings a tile
    __shared__ float qs[ML_TT][NS];
    __shared__ float ks[ML_TT][NS];
    __shared__ float vs[ML_TT][ML_PB];
    __shared__ float keep_s[ML_TT], take_s[ML_TT], em_s[ML_TT];
    __shared__ float m_carry;
    const int b = nth_run(cu_q, n_seqs, blockIdx.x / heads, lo, hi), h = blockIdx.x % heads, p0 = blockIdx.y * ML_PB;
    if (b < 0) return;
    const int start = cu_q[b], q = cu_q[b + 1] - start;
    const int slot = seq_slot[b];
    const int pl = threadIdx.x / ML_L, l = threadIdx.x % ML_L;
    const int p = p0 + pl;
    const bool p_ok = p <= dv, is_n = p == dv;
    float S[NR];
    float* sp = is_n ? n_state + ((long)slot * heads + h) * d
                     : S_state + (((long)slot * heads + h) * dv + (p_ok ? p : 0)) * d;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
        const int c = l + ML_L * i;
        S[i] = (p_ok && c < d) ? sp[c] : 0.f;
    }
    if (threadIdx.x == 0) m_carry = m_state[(long)slot * heads + h];
    const float bi = i_bias[h], bf = f_bias[h], inv_cap = 1.0f / cap;
    float rq[QK], rk[QK], rx[XV], ri = 0.f, rf = 0.f;
    auto fetch = [&](int t0) {
        const int tn = min(ML_TT, q - t0);
#pragma unroll
        for (int e2 = 0; e2 < QK; ++e2) {
            const int e = threadIdx.x + e2 * 256;
            const int tt = e / NS, c = e % NS;
            const bool ok = tt < tn && c < d;
            const T* row = proj + (long)(start + t0 + min(tt, tn - 1)) * ld + (long)h * d + min(c, d - 1);
            rq[e2] = ok ? to_f32(row[q_off]) * q_scale : 0.f;
            rk[e2] = ok ? to_f32(row[k_off]) : 0.f;
        }
#pragma unroll
        for (int e2 = 0; e2 < XV; ++e2) {
            const int e = threadIdx.x + e2 * 256;
            const int tt = e / ML_PB, pp = p0 + e % ML_PB;
            const long at = (long)(start + t0 + min(tt, tn - 1)) * ld + v_off + (long)h * dv + min(pp, dv - 1);
            const float v = to_f32(proj[at]);
            rx[e2] = tt < tn ? (pp < dv ? v : (pp == dv ? 1.0f : 0.f)) : 0.f;
        }
        if ((int)threadIdx.x < tn) {
            const T* row = proj + (long)(start + t0 + threadIdx.x) * ld + h;
            ri = to_f32(row[i_off]);
            rf = to_f32(row[f_off]);
        }
    };
    fetch(0);
    for (int t0 = 0; t0 < q; t0 += ML_TT) {
        const int tn = min(ML_TT, q - t0);
        __syncthreads();
#pragma unroll
        for (int e2 = 0; e2 < QK; ++e2) {
            const int e = threadIdx.x + e2 * 256;
            qs[e / NS][e % NS] = rq[e2];
            ks[e / NS][e % NS] = rk[e2];
        }
#pragma unroll
        for (int e2 = 0; e2 < XV; ++e2) {
            const int e = threadIdx.x + e2 * 256;
            if (e < ML_TT * ML_PB) vs[e / ML_PB][e % ML_PB] = rx[e2];
        }
        if ((int)threadIdx.x < tn) {                 // log gates, parked where their exponentials will stand
            take_s[threadIdx.x] = cap * tanhf((ri + bi) * inv_cap);
            keep_s[threadIdx.x] = log_sigmoid_f(cap * tanhf((rf + bf) * inv_cap));
        }
        __syncthreads();
        if (threadIdx.x == 0) {                      // the running maximum through the tile, in registers
            float av[ML_TT], bv[ML_TT];
#pragma unroll
            for (int tt = 0; tt < ML_TT; ++tt) {
                av[tt] = take_s[tt];
                bv[tt] = keep_s[tt];
            }
            float m = m_carry;
#pragma unroll
            for (int tt = 0; tt < ML_TT; ++tt) {
                const float m_new = tt < tn ? fmaxf(bv[tt] + m, av[tt]) : m;
                bv[tt] = bv[tt] + m - m_new;
                av[tt] = av[tt] - m_new;
                m = m_new;
                keep_s[tt] = bv[tt];
                take_s[tt] = av[tt];
                em_s[tt] = -m_new;
            }
            m_carry = m;
        }
        __syncthreads();
        if ((int)threadIdx.x < tn) {
            keep_s[threadIdx.x] = expf(keep_s[threadIdx.x]);
            take_s[threadIdx.x] = expf(take_s[threadIdx.x]);
            em_s[threadIdx.x] = expf(em_s[threadIdx.x]);
        }
        __syncthreads();
        if (t0 + ML_TT < q) fetch(t0 + ML_TT);
        // a token's keys and queries are asked of LDS while the token before it is worked on
        float kc[NR], qc[NR], keep_c, tv_c, em_c;
        auto ask = [&](int tt, float* kk, float* qq, float& keep, float& tv, float& em) {
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                kk[i] = ks[tt][l + ML_L * i];
                qq[i] = qs[tt][l + ML_L * i];
            }
            keep = keep_s[tt];
            tv = take_s[tt] * vs[tt][pl];
            em = em_s[tt];
        };
        ask(0, kc, qc, keep_c, tv_c, em_c);
        float* yp = y + (long)(start + t0) * heads * dv + (long)h * dv + p;
        float* dp = den + (long)(start + t0) * heads + h;
#pragma unroll 2
        for (int tt = 0; tt < tn; ++tt) {
            float kn[NR], qn[NR], keep_n, tv_n, em_n;
            ask(min(tt + 1, tn - 1), kn, qn, keep_n, tv_n, em_n);
            float part[4] = {0.f, 0.f, 0.f, 0.f};       // four chains of additions side by side
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                S[i] = keep_c * S[i] + tv_c * kc[i];
                part[i & 3] += S[i] * qc[i];
            }
            float num = (part[0] + part[1]) + (part[2] + part[3]);
            // the column's lanes are neighbours: the sum inside the vector unit
            num += CPMCU_DPP(num, 0xB1);
            num += CPMCU_DPP(num, 0x4E);
            num += CPMCU_DPP(num, 0x141);
            if (ML_L >= 16) num += CPMCU_DPP(num, 0x140);
            if (ML_L == 32) {                            // the two rows of 16 lanes that share a column
                cpmcu_u32x2_t sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(num), __float_as_uint(num), false, false);
                num = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
            }
            if (l == 0 && p_ok) {
                if (is_n) *dp = fmaxf(fabsf(num), em_c) + 1e-6f;
                else *yp = num;
            }
            yp += (long)heads * dv;
            dp += heads;
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                kc[i] = kn[i];
                qc[i] = qn[i];
            }
            keep_c = keep_n;
            tv_c = tv_n;
            em_c = em_n;
        }
    }
    __syncthreads();
    if (write_state) {
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int c = l + ML_L * i;
            if (p_ok && c < d) sp[c] = S[i];
        }
        if (blockIdx.y == 0 && threadIdx.x == 0) m_next[(long)b * heads + h] = m_carry;
    }
}

// the slots' maxima behind a step: a launch behind the one whose workgroups all read those before it
__global__ __launch_bounds__(256) void mlstm_maximum_kernel(const float* __restrict__ m_next, float* __restrict__ m_state,
                                                            const int* __restrict__ cu_q, const int* __restrict__ seq_slot,
                                                            int n_seqs, int heads) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= (long)n_seqs * heads) return;
    const int b = (int)(i / heads);
    if (cu_q[b + 1] > cu_q[b]) m_state[(long)seq_slot[b] * heads + i % heads] = m_next[i];
}

// ---------------------------------------------------------------------------
// The same recurrence for prompts, 32 tokens at a time on the matrix cores' float instruction (v_mfma_f32_16x16x4_f32:
// operands as they are, sums in float).  With F_t = the sum of b over the chunk's tokens up to t, w_s = a_s - F_s and
// M_t = max(m before the chunk, w_s for s <= t), all three in double, m_t = F_t + M_t and
//     y_t = exp(m - M_t) S^T q_t + sum_(s <= t) exp(w_s - M_t) (q_t . k_s) v_s
//     S  <- exp(m - M_31) S + sum_s exp(w_s - M_31) k_s v_s^T
// where no exponent is positive; the normaliser is column dv, whose value is always 1, as in the walk.  A workgroup owns
// one (sequence, head, 32 columns); its state stays in the accumulators' registers and passes through LDS as an operand.
// 8 heads of 256 by 512, prompts of 613, 479, 211, 345 and 400 tokens in one pass: 870 -> 311 us.
// A token's infinities reach no earlier token: their weights are zero, but a zero does not silence an infinity in a product,
// so outputs that are not all finite are added up again term by term.
// A lane's 16 bytes serve four instructions: instruction j of a block takes index 4 g + j of the 16 in both operands.
// ---------------------------------------------------------------------------
typedef float mlfloatx4_t __attribute__((ext_vector_type(4)));
#define MCHUNK_T 32       // tokens a chunk
#define MCHUNK_P 32       // columns a workgroup
#define MCHUNK_LT 36      // LDS rows of MCHUNK_T: rows 4 banks apart, so that 8 rows' 16 bytes read all banks

// NB: blocks of 16 key features, a multiple of 8
template <int NB, typename T>
__global__ __launch_bounds__(512) void mlstm_chunk_kernel(const T* __restrict__ proj, long ld, long q_off, long k_off,
                                                          long v_off, long i_off, long f_off,
                                                          const float* __restrict__ i_bias, const float* __restrict__ f_bias,
                                                          float cap, float q_scale, float* __restrict__ S_state,
                                                          float* __restrict__ n_state, const float* __restrict__ m_state,
                                                          float* __restrict__ m_next,
                                                          float* __restrict__ y, float* __restrict__ den,
                                                          const int* __restrict__ cu_q, const int* __restrict__ seq_slot,
                                                          int heads, int d, int dv, int write_state, int n_seqs, int lo,
                                                          int hi) {
    constexpr int LN = 16 * NB + 4, NJ = NB / 8, C4 = 4 * NB, QK = MCHUNK_T * C4 / 512;
    __shared__ __align__(16) float Qs[MCHUNK_T * LN], Ks[MCHUNK_T * LN];
    __shared__ __align__(16) float Ss[MCHUNK_P * LN];                  // the state before the chunk, [p][c]
    __shared__ __align__(16) float Gs[MCHUNK_T * MCHUNK_LT];            // exp(w_s - M_t) q_t . k_s
    __shared__ __align__(16) float vT[MCHUNK_P * MCHUNK_LT];            // [p][t]
    __shared__ __align__(16) float left_s[MCHUNK_T], from_s[MCHUNK_T], floor_s[MCHUNK_T];
    __shared__ double w_s[MCHUNK_T], M_s[MCHUNK_T];
    const int b = nth_run(cu_q, n_seqs, blockIdx.x / heads, lo, hi), h = blockIdx.x % heads, p0 = blockIdx.y * MCHUNK_P;
    if (b < 0) return;
    const int start = cu_q[b], q = cu_q[b + 1] - start, slot = seq_slot[b];
    if (q <= 0) return;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    auto state_row = [&](int p) {
        return p == dv ? n_state + ((long)slot * heads + h) * d : S_state + (((long)slot * heads + h) * dv + min(p, dv - 1)) * d;
    };
    // the state as the accumulators hold it: st[i][j][e] is column p = 16 i + 4 g + e, key feature c = 16 (NJ wave + j) + r
    mlfloatx4_t st[2][NJ];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int p = p0 + 16 * i + 4 * g + e, c = 16 * (NJ * wave + j) + r;
                st[i][j][e] = (p <= dv && c < d) ? state_row(p)[c] : 0.f;
            }
    double m = (double)m_state[(long)slot * heads + h];                // wavefront 0 carries it on (m_next: see the walk)
    const float bi = i_bias[h], bf = f_bias[h], inv_cap = 1.0f / cap;
    const mlfloatx4_t zero4 = {0.f, 0.f, 0.f, 0.f};
    const int vrow = threadIdx.x >> 3, vcol = (threadIdx.x & 7) * 4;   // (256 threads bring values)
    float4 rq[QK], rk[QK], rv = make_float4(0.f, 0.f, 0.f, 0.f);
    float ri = 0.f, rf = 0.f;
    auto fetch = [&](int t0) {
        const int tn = min(MCHUNK_T, q - t0);
        const T* base = proj + (long)(start + t0) * ld;
#pragma unroll
        for (int i = 0; i < QK; ++i) {
            const int e = threadIdx.x + 512 * i, c = (e % C4) * 4;
            const T* row = base + (long)min(e / C4, tn - 1) * ld + (long)h * d + min(c, d - 4);
            rq[i] = load4(row + q_off);
            rk[i] = load4(row + k_off);
            if (c >= d) rq[i] = rk[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
        const int p = p0 + vcol;
        rv = load4(base + (long)min(vrow, tn - 1) * ld + v_off + (long)h * dv + min(p, dv - 4));
        if (p >= dv) rv = make_float4(p == dv ? 1.f : 0.f, 0.f, 0.f, 0.f);
        if (wave == 0) {
            const T* row = base + (long)min(lane, tn - 1) * ld + h;
            ri = to_f32(row[i_off]);
            rf = to_f32(row[f_off]);
        }
    };
    // one 16 x 16 tile of rows[i] . cols[j] over the key features
    auto dot_tile = [&](const float* rows, int i, const float* cols, int j) {
        mlfloatx4_t a = zero4;
#pragma unroll
        for (int kb = 0; kb < NB; ++kb) {
            const mlfloatx4_t x = *(const mlfloatx4_t*)&rows[(16 * i + r) * LN + 16 * kb + 4 * g];
            const mlfloatx4_t z = *(const mlfloatx4_t*)&cols[(16 * j + r) * LN + 16 * kb + 4 * g];
#pragma unroll
            for (int e = 0; e < 4; ++e) a = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], z[e], a, 0, 0, 0);
        }
        return a;
    };
    fetch(0);
    for (int t0 = 0; t0 < q; t0 += MCHUNK_T) {
        const int tn = min(MCHUNK_T, q - t0);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) Ss[(16 * i + 4 * g + e) * LN + 16 * (NJ * wave + j) + r] = st[i][j][e];
        if (tn < MCHUNK_T) {                                           // rows behind the run's end repeat its last token
#pragma unroll
            for (int i = 0; i < QK; ++i)
                if ((int)(threadIdx.x + 512 * i) / C4 >= tn) rk[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (vrow >= tn) rv = make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int i = 0; i < QK; ++i) {
            const int e = threadIdx.x + 512 * i, at = (e / C4) * LN + (e % C4) * 4;
            store4(&Qs[at], rq[i].x * q_scale, rq[i].y * q_scale, rq[i].z * q_scale, rq[i].w * q_scale);
            store4(&Ks[at], rk[i].x, rk[i].y, rk[i].z, rk[i].w);
        }
        if (vrow < MCHUNK_T) {
            vT[vcol * MCHUNK_LT + vrow] = rv.x;
            vT[(vcol + 1) * MCHUNK_LT + vrow] = rv.y;
            vT[(vcol + 2) * MCHUNK_LT + vrow] = rv.z;
            vT[(vcol + 3) * MCHUNK_LT + vrow] = rv.w;
        }
        if (wave == 0) {
            // a token beyond the end neither writes (w = -inf) nor forgets (b = 0); lanes 32 .. 63 are such tokens too
            const bool in = lane < tn;
            double F = in ? (double)log_sigmoid_f(cap * tanhf((rf + bf) * inv_cap)) : 0.0;
#pragma unroll
            for (int k = 1; k < 64; k <<= 1) {
                const double up = __shfl_up(F, k, 64);
                if (lane >= k) F += up;
            }
            const double w = in ? (double)(cap * tanhf((ri + bi) * inv_cap)) - F : -INFINITY;
            double M = fmax(m, w);
#pragma unroll
            for (int k = 1; k < 64; k <<= 1) {
                const double up = __shfl_up(M, k, 64);
                if (lane >= k) M = fmax(M, up);
            }
            const double M_end = __shfl(M, 63, 64);
            if (lane < MCHUNK_T) {
                w_s[lane] = w;
                M_s[lane] = M;
                left_s[lane] = expf((float)(w - M_end));
                from_s[lane] = expf((float)(m - M));
                floor_s[lane] = expf((float)(-(F + M)));
            }
            m = __shfl(F, 63, 64) + M_end;
        }
        __syncthreads();
        if (t0 + MCHUNK_T < q) fetch(t0 + MCHUNK_T);
        // wavefronts 0 to 2: the tiles of G on and below the diagonal; 3 to 6: what the state before the chunk gives tokens
        // 16 tt .. + 15 in columns 16 pt .. + 15
        const int tt = wave < 3 ? (wave + 1) / 2 : ((wave - 3) >> 1) & 1, pt = (wave - 3) & 1;
        const bool owns = wave >= 3 && wave < 7;
        auto write_y = [&](const mlfloatx4_t& v) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 16 * tt + 4 * g + e, p = p0 + 16 * pt + r;
                if (t >= tn) continue;
                if (p < dv) y[(long)(start + t0 + t) * heads * dv + (long)h * dv + p] = v[e];
                else if (p == dv) den[(long)(start + t0 + t) * heads + h] = fmaxf(fabsf(v[e]), floor_s[t]) + 1e-6f;
            }
        };
        mlfloatx4_t yt = zero4;
        if (wave < 3) {
            const int j = wave == 2 ? 1 : 0, s = 16 * j + r;
            const mlfloatx4_t a = dot_tile(Qs, tt, Ks, j);
            const double w = w_s[s];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 16 * tt + 4 * g + e;
                Gs[t * MCHUNK_LT + s] = s <= t ? a[e] * expf((float)(w - M_s[t])) : 0.f;
            }
        } else if (wave < 7) {
            yt = dot_tile(Qs, tt, Ss, pt);
#pragma unroll
            for (int e = 0; e < 4; ++e) yt[e] *= from_s[16 * tt + 4 * g + e];
        }
        const mlfloatx4_t y0 = yt;
        __syncthreads();
        if (owns) {
            // ... and what the chunk's own tokens give them
            for (int kb = 0; kb <= tt; ++kb) {
                const mlfloatx4_t a = *(const mlfloatx4_t*)&Gs[(16 * tt + r) * MCHUNK_LT + 16 * kb + 4 * g];
                const mlfloatx4_t v = *(const mlfloatx4_t*)&vT[(16 * pt + r) * MCHUNK_LT + 16 * kb + 4 * g];
#pragma unroll
                for (int e = 0; e < 4; ++e) yt = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], v[e], yt, 0, 0, 0);
            }
            write_y(yt);
        }
        // the state behind the chunk
        const float keep = from_s[MCHUNK_T - 1];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) st[i][j] *= keep;
#pragma unroll
        for (int kb = 0; kb < MCHUNK_T / 16; ++kb) {
            const mlfloatx4_t w4 = *(const mlfloatx4_t*)&left_s[16 * kb + 4 * g];
            mlfloatx4_t v4[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) v4[i] = *(const mlfloatx4_t*)&vT[(16 * i + r) * MCHUNK_LT + 16 * kb + 4 * g] * w4;
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float kv = Ks[(16 * kb + 4 * g + e) * LN + 16 * (NJ * wave + j) + r];
#pragma unroll
                    for (int i = 0; i < 2; ++i) st[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(v4[i][e], kv, st[i][j], 0, 0, 0);
                }
        }
        if (owns && wave_odd(yt[0], yt[1], yt[2], yt[3])) {
            mlfloatx4_t again = y0;
#pragma unroll 1
            for (int s = 0; s < MCHUNK_T; ++s) {
                const float one = vT[(16 * pt + r) * MCHUNK_LT + s];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int t = 16 * tt + 4 * g + e;
                    if (s <= t) again[e] += Gs[t * MCHUNK_LT + s] * one;
                }
            }
            write_y(again);
        }
        __syncthreads();
    }
    if (write_state) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int p = p0 + 16 * i + 4 * g + e, c = 16 * (NJ * wave + j) + r;
                    if (p <= dv && c < d) state_row(p)[c] = st[i][j][e];
                }
        if (blockIdx.y == 0 && threadIdx.x == 0) m_next[(long)b * heads + h] = (float)m;
    }
}

// The n_chunked sequences that bring at least chunk_from tokens are taken in chunks, the others are walked: two launches
// where there are both.  (0, 0: all are walked, as they are where the chunks' kernel does not take the sizes.)
// m_next: float [n_seqs * heads], scratch.
extern "C" const char* cpmcu_mlstm_scan(const void* proj, long ld, int dtype, long q_off, long k_off, long v_off,
                                        long i_off, long f_off, const float* i_bias, const float* f_bias, float cap,
                                        float q_scale, float* S_state, float* n_state, float* m_state, float* m_next,
                                        float* y, float* den, const int* cu_q, const int* seq_slot, int n_seqs, int heads,
                                        int d, int dv, int write_state, int chunk_from, int n_chunked,
                                        hipStream_t stream) {
    CPMCU_REQUIRE(n_seqs > 0 && heads > 0 && d > 0 && dv > 0, "mlstm_scan: empty shape");
    CPMCU_REQUIRE(d <= 1024, "mlstm_scan: a key size of %d is not supported (at most 1024)", d);
    CPMCU_REQUIRE(cap > 0.f, "mlstm_scan: gate cap %g", cap);
    CPMCU_REQUIRE(q_off >= 0 && k_off >= 0 && v_off >= 0 && i_off >= 0 && f_off >= 0 && q_off + (long)heads * d <= ld &&
                  k_off + (long)heads * d <= ld && v_off + (long)heads * dv <= ld && i_off + heads <= ld && f_off + heads <= ld,
                  "mlstm_scan: columns beyond rows of %ld", ld);
    CPMCU_REQUIRE(!write_state || m_next, "mlstm_scan: scratch for the maxima is missing");
    const auto move_maxima = [&]() {
        if (write_state)
            mlstm_maximum_kernel<<<(unsigned)(((long)n_seqs * heads + 255) / 256), 256, 0, stream>>>(m_next, m_state, cu_q,
                                                                                                    seq_slot, n_seqs, heads);
    };
    CPMCU_REQUIRE(chunk_from >= 0 && n_chunked >= 0 && n_chunked <= n_seqs, "mlstm_scan: %d sequences of %d in chunks", n_chunked, n_seqs);
    CPMCU_REQUIRE((long)n_seqs * heads < (1L << 31), "mlstm_scan: shape exceeds the launch grid");
    if (!(d <= 256 && d % 4 == 0 && dv % 4 == 0 && ld % 4 == 0 && q_off % 4 == 0 && k_off % 4 == 0 && v_off % 4 == 0 &&
          (uintptr_t)proj % 16 == 0 && (dtype == CPMCU_F32 || dtype == CPMCU_BF16)))
        n_chunked = 0;
    if (n_chunked > 0) {
        const dim3 grid(heads * n_chunked, (dv + 1 + MCHUNK_P - 1) / MCHUNK_P);
        const int hi = n_chunked < n_seqs ? 0x7fffffff : 0;
        CPMCU_REQUIRE(grid.y <= 65535, "mlstm_scan: shape exceeds the launch grid");
#define CHUNKS(NBv, Tv)                                                                                             \
    mlstm_chunk_kernel<NBv, Tv><<<grid, 512, 0, stream>>>((const Tv*)proj, ld, q_off, k_off, v_off, i_off, f_off,   \
                                                          i_bias, f_bias, cap, q_scale, S_state, n_state, m_state,  \
                                                          m_next, y, den, cu_q, seq_slot, heads, d, dv, write_state, \
                                                          n_seqs, chunk_from, hi)
        if (dtype == CPMCU_F32) {
            if (d <= 128) CHUNKS(8, float);
            else CHUNKS(16, float);
        } else {
            if (d <= 128) CHUNKS(8, bf16_t);
            else CHUNKS(16, bf16_t);
        }
#undef CHUNKS
        CPMCU_LAUNCH_CHECK("mlstm_chunk");
        if (n_chunked == n_seqs) {
            move_maxima();
            CPMCU_LAUNCH_CHECK("mlstm_maximum");
            return nullptr;
        }
    }
    const int lo = 0, hi = n_chunked > 0 ? chunk_from : 0;
    const int lanes = d > 128 ? 32 : 8, cols = 256 / lanes;
    const int pb = (dv + 1 + cols - 1) / cols;       // the normaliser is walked as column dv
    CPMCU_REQUIRE(pb <= 65535, "mlstm_scan: shape exceeds the launch grid");
    dim3 grid(heads * (n_seqs - n_chunked), pb);
    const int need = (d + lanes - 1) / lanes;
#define LAUNCH(NRv, Lv, TTv, Tv)                                                                                     \
    mlstm_scan_kernel<NRv, Lv, TTv, Tv><<<grid, 256, 0, stream>>>((const Tv*)proj, ld, q_off, k_off, v_off, i_off,   \
                                                                  f_off, i_bias, f_bias, cap, q_scale, S_state,      \
                                                                  n_state, m_state, m_next, y, den, cu_q, seq_slot,  \
                                                                  heads, d, dv, write_state, n_seqs, lo, hi)
#define BY_NR(Tv)                                  \
    do {                                           \
        if (lanes == 32 && need <= 8) LAUNCH(8, 32, 16, Tv);        \
        else if (lanes == 32 && need <= 16) LAUNCH(16, 32, 8, Tv);  \
        else if (lanes == 32) LAUNCH(32, 32, 4, Tv);                \
        else if (need <= 2) LAUNCH(2, 8, 32, Tv);  \
        else if (need <= 4) LAUNCH(4, 8, 32, Tv);  \
        else if (need <= 8) LAUNCH(8, 8, 32, Tv);  \
        else LAUNCH(16, 8, 32, Tv);                \
    } while (0)
    if (dtype == CPMCU_F32) BY_NR(float);
    else if (dtype == CPMCU_BF16) BY_NR(bf16_t);
    else CPMCU_FAIL("mlstm_scan: unknown dtype %d", dtype);
#undef BY_NR
#undef LAUNCH
    CPMCU_LAUNCH_CHECK("mlstm_scan");
    move_maxima();
    CPMCU_LAUNCH_CHECK("mlstm_maximum");
    return nullptr;
}
