// Gated delta rule over a packed batch, with per-slot state: a linear recurrence whose state is a matrix a head
// that forgets by a decay and corrects what it holds under the current key before it writes the new value.
//
// Per head h (its q and k come from head h / (heads / kv_heads)), everything in float:
//     qn = q / sqrt(sum q^2 + 1e-6) * q_scale,  kn = k / sqrt(sum k^2 + 1e-6)
//     beta = sigmoid(b_raw),  g = exp(-exp(A_log[h]) * softplus(a_raw + dt_bias[h]))
//     S <- g S;  u = beta (v - S^T kn);  S <- S + kn u^T;  o = S^T qn            S: [dk, dv], zero at the start
// Since S^T qn after the write is g (S_old^T qn) + (kn . qn) u, both products with the old state are formed in
// one pass over it (a column's two sums meet in one reduction) and the state is read and written once a token.
//
// A workgroup owns one (sequence, head, 32 or 16 columns of dv) and walks the sequence's tokens in order; a
// column's dk state values are spread over 8 or 16 neighbouring lanes (state index i = l + L r), the tokens' q,
// k, v and gates pass through LDS in tiles of 16 or 32 tokens, where the unit norms and k . q are formed once a
// token, and the next tile's values are asked for while the current one is walked.  A token's cost is one
// dependent chain of multiply-adds over a lane's share of the column and a reduction over the column's lanes:
// where the batch has too few (sequence, head, column) triples to fill the chip (a single prompt, a step of one
// sequence), 16 lanes a column halve that chain and double the number of workgroups.
//
// The same walk serves two relatives of the rule (RULE):
//   * RULE_CHANNEL: the decay is a number a head and key channel, g[i] = exp(-exp(A_log[h]) * softplus(a_raw[h, i] +
//     dt_bias[h, i])), acting on the rows of S: S <- diag(g) S, then as above.  With t_i = g_i S_i the two sums are
//     sum t_i kn_i and sum t_i qn_i, the write is S_i = t_i + kn_i u and the read-out sum t_i qn_i + (kn . qn) u.
//   * RULE_DECAY: linear attention with a fixed decay a head and nothing learned in the recurrence:
//     S <- d_h S + k v^T;  o = S^T q = d_h (S_old^T q) + (k . q) v, with q and k taken as they come (no unit
//     norm, no beta, no gates); `A_log` then holds the decays d_h themselves.
#include "common.h"
#include "runs.h"

enum { RULE_DELTA = 0, RULE_CHANNEL = 1, RULE_DECAY = 2 };

__device__ inline float delta_softplus(float v) { return fmaxf(v, 0.f) + log1pf(expf(-fabsf(v))); }

// qkv: float [n, ld] = [q: kv_heads*dk | k: kv_heads*dk | v: heads*dv] (after convolution and activation);
// gates: raw projections [n, ldg], the decay's at column a_off + h, beta's at b_off + h;
// state: float [slots][heads][dv][dk]; y: float [n, heads*dv].
// chan_a (RULE_CHANNEL): float [n, ld_a], the raw decay projection of head h and key channel i at column h*dk + i;
// dt_bias then has heads*dk numbers.
// grid (sequences x heads, blocks of DELTA_PB columns): a sequence's workgroups are dealt to all XCDs, also where one
// sequence of a step is much longer than the others.  The launch takes the sequences of lo <= tokens < hi (runs.h).
template <int NR, int TT, int DELTA_L, typename GT, int RULE>
__global__ __launch_bounds__(256) void delta_scan_kernel(const float* __restrict__ qkv, long ld,
                                                         const GT* __restrict__ gates, long ldg, long a_off, long b_off,
                                                         const float* __restrict__ chan_a, long ld_a,
                                                         const float* __restrict__ dt_bias,
                                                         const float* __restrict__ A_log, float* __restrict__ state,
                                                         float* __restrict__ y, const int* __restrict__ cu_q,
                                                         const int* __restrict__ seq_slot, int heads, int kv_heads,
                                                         int dk, int dv, float q_scale, int write_state, int n_seqs,
                                                         int lo, int hi) {
    constexpr int DELTA_PB = 256 / DELTA_L;         // columns of dv a workgroup
    constexpr int NS = NR * DELTA_L;                // state values a column, padded
    constexpr int QK = TT * NS / 256;               // q (and k) values a thread brings a tile
    constexpr int VV = (TT * DELTA_PB + 255) / 256; // v values a thread brings a tile
    constexpr int TPT = 256 / TT;                   // threads that share a token's norms
    static_assert(TT * NS % 256 == 0 && (TT == 16 || TT == 32), "tile shape");
    __shared__ float qs[TT][NS];
    __shared__ float ks[TT][NS];
    __shared__ float vs[TT][DELTA_PB];
    __shared__ float betas[TT], gs[TT], kqs[TT];
    __shared__ float gcs[RULE == RULE_CHANNEL ? TT : 1][RULE == RULE_CHANNEL ? NS : 1];   // a decay a channel
    const int b = nth_run(cu_q, n_seqs, blockIdx.x / heads, lo, hi), p0 = blockIdx.y * DELTA_PB;
    const int h = grouped_head(blockIdx.x % heads, heads, kv_heads);
    if (b < 0) return;
    const int start = cu_q[b], n_q = cu_q[b + 1] - start;
    const int slot = seq_slot[b];
    const int kvh = h / (heads / kv_heads);
    const long k_col = (long)kv_heads * dk, v_col = 2L * kv_heads * dk;
    const int pl = threadIdx.x / DELTA_L, l = threadIdx.x % DELTA_L;
    const int p = p0 + pl;
    const bool p_ok = p < dv;
    float S[NR];
    float* sp = state + (((long)slot * heads + h) * dv + (p_ok ? p : 0)) * dk;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
        const int n = l + DELTA_L * i;
        S[i] = (p_ok && n < dk) ? sp[n] : 0.f;
    }
    // RULE_DECAY: A_log holds the head's fixed decay itself
    const float A = RULE == RULE_DECAY ? A_log[h] : expf(A_log[h]);
    const float bias = RULE == RULE_DELTA ? dt_bias[h] : 0.f;
    float rq[QK], rk[QK], rv[VV], ra = 0.f, rb = 0.f;
    float rg[RULE == RULE_CHANNEL ? QK : 1];
    auto fetch = [&](int t0) {
        const int tn = min(TT, n_q - t0);
#pragma unroll
        for (int k = 0; k < QK; ++k) {
            const int e = threadIdx.x + k * 256;
            const int tt = e / NS, n = e % NS;
            const bool ok = tt < tn && n < dk;
            const float* row = qkv + (long)(start + t0 + min(tt, tn - 1)) * ld + (long)kvh * dk + min(n, dk - 1);
            rq[k] = ok ? row[0] : 0.f;
            rk[k] = ok ? row[k_col] : 0.f;
            if (RULE == RULE_CHANNEL) {
                const float a = chan_a[(long)(start + t0 + min(tt, tn - 1)) * ld_a + (long)h * dk + min(n, dk - 1)];
                rg[k] = ok ? a + dt_bias[(long)h * dk + min(n, dk - 1)] : 0.f;
            }
        }
#pragma unroll
        for (int k = 0; k < VV; ++k) {
            const int e = threadIdx.x + k * 256;
            const int tt = e / DELTA_PB, pp = e % DELTA_PB;
            rv[k] = (tt < tn && p0 + pp < dv) ? qkv[(long)(start + t0 + tt) * ld + v_col + (long)h * dv + p0 + pp] : 0.f;
        }
        if (RULE != RULE_DECAY && (int)threadIdx.x < tn) {
            const GT* gr = gates + (long)(start + t0 + threadIdx.x) * ldg;
            if (RULE == RULE_DELTA) ra = to_f32(gr[a_off + h]);
            rb = to_f32(gr[b_off + h]);
        }
    };
    fetch(0);
    for (int t0 = 0; t0 < n_q; t0 += TT) {
        const int tn = min(TT, n_q - t0);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < QK; ++k) {
            const int e = threadIdx.x + k * 256;
            qs[e / NS][e % NS] = rq[k];
            ks[e / NS][e % NS] = rk[k];
            // (rows of the tile that this step does not bring are never walked: no exponentials for them)
            if (RULE == RULE_CHANNEL && e / NS < tn) gcs[e / NS][e % NS] = expf(-A * delta_softplus(rg[k]));
        }
#pragma unroll
        for (int k = 0; k < VV; ++k) {
            const int e = threadIdx.x + k * 256;
            if (e < TT * DELTA_PB) vs[e / DELTA_PB][e % DELTA_PB] = rv[k];
        }
        if ((int)threadIdx.x < tn) {
            betas[threadIdx.x] = RULE == RULE_DECAY ? 1.0f : 1.0f / (1.0f + expf(-rb));
            gs[threadIdx.x] = RULE == RULE_DELTA ? expf(-A * delta_softplus(ra + bias)) : A;
        }
        __syncthreads();
        {
            // unit vectors and k . q, once a token: TPT neighbouring threads share a token's NS values
            const int tt = threadIdx.x / TPT, part = threadIdx.x % TPT;
            float sq = 0.f, sk = 0.f, dot = 0.f;
            for (int n = part; n < NS; n += TPT) {
                const float a = qs[tt][n], c = ks[tt][n];
                sq += a * a;
                sk += c * c;
                dot += a * c;
            }
            sq = lanes_sum<TPT>(sq);
            sk = lanes_sum<TPT>(sk);
            dot = lanes_sum<TPT>(dot);
            if (RULE == RULE_DECAY) {
                if (part == 0) kqs[tt] = dot;
            } else {
                const float fq = q_scale / sqrtf(sq + 1e-6f), fk = 1.0f / sqrtf(sk + 1e-6f);
                for (int n = part; n < NS; n += TPT) {
                    qs[tt][n] *= fq;
                    ks[tt][n] *= fk;
                }
                if (part == 0) kqs[tt] = dot * fq * fk;
            }
        }
        __syncthreads();
        if (t0 + TT < n_q) fetch(t0 + TT);
        for (int tt = 0; tt < tn; ++tt) {
            const float g = gs[tt], beta = betas[tt], vv = vs[tt][pl], kq = kqs[tt];
            float kr[NR];
            float r = 0.f, o = 0.f;
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                const int n = l + DELTA_L * i;
                kr[i] = ks[tt][n];
                if (RULE == RULE_CHANNEL) S[i] *= gcs[tt][n];      // the channel's decay first: the sums see g_i S_i
                if (RULE != RULE_DECAY) r += S[i] * kr[i];
                o += S[i] * qs[tt][n];
            }
            // the column's lanes are neighbours: both sums meet inside the vector unit, every lane gets them
            if (RULE != RULE_DECAY) r += CPMCU_DPP(r, 0xB1);
            o += CPMCU_DPP(o, 0xB1);
            if (RULE != RULE_DECAY) r += CPMCU_DPP(r, 0x4E);
            o += CPMCU_DPP(o, 0x4E);
            if (RULE != RULE_DECAY) r += CPMCU_DPP(r, 0x141);
            o += CPMCU_DPP(o, 0x141);
            if (DELTA_L == 16) {
                if (RULE != RULE_DECAY) r += CPMCU_DPP(r, 0x140);
                o += CPMCU_DPP(o, 0x140);
            }
            // the decay that the sums still lack: the head's (RULE_CHANNEL applied its own above)
            const float gg = RULE == RULE_CHANNEL ? 1.0f : g;
            const float u = RULE == RULE_DECAY ? vv : beta * (vv - gg * r);
#pragma unroll
            for (int i = 0; i < NR; ++i) S[i] = gg * S[i] + kr[i] * u;
            if (l == 0 && p_ok) y[(long)(start + t0 + tt) * heads * dv + (long)h * dv + p] = gg * o + kq * u;
        }
    }
    if (write_state && p_ok) {
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int n = l + DELTA_L * i;
            if (n < dk) sp[n] = S[i];
        }
    }
}

// The same walk where every sequence brings one token (any number is walked right): the tile's 16 or 32 rows of LDS, their
// norms and their barriers are a token's.  A workgroup asks for its share of the state first; the decays of the key channels
// pass through LDS, one a thread.  TPT: threads that share the norms' sums; every sum keeps the walk's order, so results are
// the same (with a decay a head the compiler may fuse g S + k u the other way).  32 heads of 128 by 128, us, walk -> here:
// 8 sequences in a serving, a decay a channel 26.7 -> 10.7, fixed decays 14.9 -> 10.4 (their states' 34 MB in and out take 5);
// 24 in a chain of calls 63 -> 29, 31 -> 27, a decay a head 42 -> 28; 64, a decay a channel 153 -> 63.
template <int NR, int TPT, int DELTA_L, typename GT, int RULE>
__global__ __launch_bounds__(256) void delta_step_kernel(const float* __restrict__ qkv, long ld,
                                                         const GT* __restrict__ gates, long ldg, long a_off, long b_off,
                                                         const float* __restrict__ chan_a, long ld_a,
                                                         const float* __restrict__ dt_bias,
                                                         const float* __restrict__ A_log, float* __restrict__ state,
                                                         float* __restrict__ y, const int* __restrict__ cu_q,
                                                         const int* __restrict__ seq_slot, int heads, int kv_heads,
                                                         int dk, int dv, float q_scale, int write_state) {
    constexpr int NS = NR * DELTA_L;                // state values a column, padded
    static_assert(NS <= 256, "a thread a key feature");
    __shared__ float qs[2][NS], ks[2][NS], gcs[2][RULE == RULE_CHANNEL ? NS : 1];
    const int b = blockIdx.x / heads, h = grouped_head(blockIdx.x % heads, heads, kv_heads);
    const int start = cu_q[b], n_q = cu_q[b + 1] - start;
    const int kvh = h / (heads / kv_heads);
    const long k_col = (long)kv_heads * dk, v_col = 2L * kv_heads * dk;
    const int l = threadIdx.x % DELTA_L, p = blockIdx.y * (256 / DELTA_L) + threadIdx.x / DELTA_L;
    const bool p_ok = p < dv;
    float* sp = state + (((long)seq_slot[b] * heads + h) * dv + (p_ok ? p : 0)) * dk;
    float S[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) S[i] = sp[min(l + DELTA_L * i, dk - 1)];
    const float A = RULE == RULE_DECAY ? A_log[h] : expf(A_log[h]);
    const float bias = RULE == RULE_DELTA ? dt_bias[h] : 0.f;
    const int n_own = min((int)threadIdx.x, dk - 1);
    const bool own = (int)threadIdx.x < dk;
    for (int tt = 0; tt < n_q; ++tt) {
        const int buf = tt & 1;
        const float* row = qkv + (long)(start + tt) * ld + (long)kvh * dk + n_own;
        const float rq = row[0], rk = row[k_col];
        const float vv = p_ok ? qkv[(long)(start + tt) * ld + v_col + (long)h * dv + p] : 0.f;
        float beta = 1.0f, g = A;
        if (RULE != RULE_DECAY) {
            const GT* gr = gates + (long)(start + tt) * ldg;
            beta = 1.0f / (1.0f + expf(-to_f32(gr[b_off + h])));
            if (RULE == RULE_DELTA) g = expf(-A * delta_softplus(to_f32(gr[a_off + h]) + bias));
        }
        if (threadIdx.x < NS) {
            qs[buf][threadIdx.x] = own ? rq : 0.f;
            ks[buf][threadIdx.x] = own ? rk : 0.f;
            if (RULE == RULE_CHANNEL) {
                const float a = chan_a[(long)(start + tt) * ld_a + (long)h * dk + n_own] + dt_bias[(long)h * dk + n_own];
                gcs[buf][threadIdx.x] = expf(-A * delta_softplus(own ? a : 0.f));
            }
        }
        __syncthreads();
        float sq = 0.f, sk = 0.f, dot = 0.f;
#pragma unroll
        for (int n = threadIdx.x % TPT; n < NS; n += TPT) {
            const float a = qs[buf][n], c = ks[buf][n];
            sq += a * a;
            sk += c * c;
            dot += a * c;
        }
        sq = lanes_sum<TPT>(sq);
        sk = lanes_sum<TPT>(sk);
        dot = lanes_sum<TPT>(dot);
        float fq = 1.0f, fk = 1.0f, kq = dot;
        if (RULE != RULE_DECAY) {
            fq = q_scale / sqrtf(sq + 1e-6f);
            fk = 1.0f / sqrtf(sk + 1e-6f);
            kq = dot * fq * fk;
        }
        float kr[NR];
        float r = 0.f, o = 0.f;
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int n = l + DELTA_L * i;
            if (tt == 0 && !(p_ok && n < dk)) S[i] = 0.f;
            float qr = qs[buf][n];
            kr[i] = ks[buf][n];
            if (RULE != RULE_DECAY) {
                qr *= fq;
                kr[i] *= fk;
            }
            if (RULE == RULE_CHANNEL) S[i] *= gcs[buf][n];
            if (RULE != RULE_DECAY) r += S[i] * kr[i];
            o += S[i] * qr;
        }
        r = lanes_sum<DELTA_L>(r);
        o = lanes_sum<DELTA_L>(o);
        const float gg = RULE == RULE_CHANNEL ? 1.0f : g;
        const float u = RULE == RULE_DECAY ? vv : beta * (vv - gg * r);
#pragma unroll
        for (int i = 0; i < NR; ++i) S[i] = gg * S[i] + kr[i] * u;
        if (l == 0 && p_ok) y[(long)(start + tt) * heads * dv + (long)h * dv + p] = gg * o + kq * u;
    }
    if (write_state && p_ok && n_q > 0) {
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int n = l + DELTA_L * i;
            if (n < dk) sp[n] = S[i];
        }
    }
}

// ---------------------------------------------------------------------------
// The delta rule with a decay a head (RULE_DELTA) for prompts, 64 tokens at a time on the matrix cores' float instruction
// (v_mfma_f32_16x16x4_f32: operands as they are, sums in float).  With la_t = the sum of ln g over the chunk's tokens up to
// t (in double, so that a difference of two sums is as good as the walk's product of factors; no exponent is positive) and
// S the state before the chunk, the walk's u_t are the solution of a triangular system, and the rest are products:
//     u_t + sum_(s < t) A[t, s] u_s = beta_t (v_t - exp(la_t) S^T k_t),    A[t, s] = beta_t exp(la_t - la_s) k_t . k_s
//     o_t = exp(la_t) S^T q_t + sum_(s <= t) exp(la_t - la_s) (q_t . k_s) u_s
//     S  <- exp(la_63) S + sum_s exp(la_63 - la_s) k_s u_s^T
// (k, q the unit vectors: their factors are multiplied in where a product's results leave the accumulators.)  The system is
// solved 16 rows at a time: the diagonal blocks of I + A are inverted by one wavefront, a lane a column; then a wavefront
// owns 16 columns of u and needs nobody else's.  A workgroup owns one (sequence, head, 16 PT columns of dv), its state stays
// in the accumulators' registers and passes through LDS as an operand.  The walk's cost is one dependent chain a token (0.35
// us), a chunk takes 11 us: 32 heads of 128 by 128, 1,500 tokens 528 -> 262 us (298 with 32 columns a workgroup).
// A token's infinities reach no earlier token: their factors are zero, but a zero does not silence an infinity in a product,
// so u and outputs that are not all finite are worked out again term by term.
// A lane's 16 bytes serve four instructions: instruction j of a block takes index 4 g + j of the 16 in both operands.
// ---------------------------------------------------------------------------
typedef float dfloatx4_t __attribute__((ext_vector_type(4)));
#define DCHUNK_T 64       // tokens a chunk
#define DCHUNK_N 128      // key features, at most
#define DCHUNK_LN 132     // LDS rows of DCHUNK_N: rows 4 banks apart, so that 8 rows' 16 bytes read all banks
#define DCHUNK_LT 68      // LDS rows of DCHUNK_T

template <int NB, int PT, typename GT>
__global__ __launch_bounds__(512) void delta_chunk_kernel(const float* __restrict__ qkv, long ld,
                                                          const GT* __restrict__ gates, long ldg, long a_off, long b_off,
                                                          const float* __restrict__ dt_bias, const float* __restrict__ A_log,
                                                          float* __restrict__ state, float* __restrict__ y,
                                                          const int* __restrict__ cu_q, const int* __restrict__ seq_slot,
                                                          int heads, int kv_heads, int dk, int dv, float q_scale,
                                                          int write_state, int n_seqs, int lo, int hi) {
    constexpr int PB = 16 * PT;                                         // columns of dv a workgroup
    __shared__ __align__(16) float Ks[DCHUNK_T * DCHUNK_LN], Qs[DCHUNK_T * DCHUNK_LN];
    __shared__ __align__(16) float Ss[PB * DCHUNK_LN];            // the state before the chunk, [p][n]
    __shared__ __align__(16) float As[DCHUNK_T * DCHUNK_LT];            // -A
    __shared__ __align__(16) float Gs[DCHUNK_T * DCHUNK_LT];            // exp(la_t - la_s) q_t . k_s
    __shared__ __align__(16) float rT[PB * DCHUNK_LT], uT[PB * DCHUNK_LT];  // v, then the right-hand side; u: [p][t]
    __shared__ __align__(16) float inv_s[4 * 16 * 20];                  // inverses of the diagonal blocks
    __shared__ __align__(16) float fk_s[DCHUNK_T], fq_s[DCHUNK_T], beta_s[DCHUNK_T], left_s[DCHUNK_T], from_s[DCHUNK_T];
    __shared__ double la_s[DCHUNK_T];
    const int b = nth_run(cu_q, n_seqs, blockIdx.x / heads, lo, hi), p0 = blockIdx.y * PB;
    const int h = grouped_head(blockIdx.x % heads, heads, kv_heads);
    if (b < 0) return;
    const int start = cu_q[b], q = cu_q[b + 1] - start;
    if (q <= 0) return;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int kvh = h / (heads / kv_heads);
    const long q_col = (long)kvh * dk, k_col = q_col + (long)kv_heads * dk, v_col = 2L * kv_heads * dk + (long)h * dv;
    float* sp = state + (((long)seq_slot[b] * heads + h) * dv + p0) * dk;
    // the state as the accumulators hold it: st[i][e] is column p = 16 i + 4 g + e, key feature n = 16 wave + r
    const int n_own = 16 * wave + r;
    dfloatx4_t st[PT];
#pragma unroll
    for (int i = 0; i < PT; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int p = 16 * i + 4 * g + e;
            st[i][e] = (p0 + p < dv && n_own < dk) ? sp[(long)p * dk + n_own] : 0.f;
        }
    const float A = decay_rate(A_log[h]), bias = dt_bias[h];
    const dfloatx4_t zero4 = {0.f, 0.f, 0.f, 0.f};
    const int vrow = threadIdx.x / (PB / 4), vcol = threadIdx.x % (PB / 4) * 4;      // (with 16 columns half of the threads)
    dfloatx4_t rq[4], rk[4], rv;
    float ra = 0.f, rb = 0.f;
    auto fetch = [&](int t0) {
        const int tn = min(DCHUNK_T, q - t0);
        const float* base = qkv + (long)(start + t0) * ld;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = threadIdx.x + 512 * i, n = (e & 31) * 4;
            const float* row = base + (long)min(e >> 5, tn - 1) * ld + min(n, dk - 4);
            rq[i] = *(const dfloatx4_t*)(row + q_col);
            rk[i] = *(const dfloatx4_t*)(row + k_col);
            if (n >= dk) rq[i] = rk[i] = zero4;
        }
        const int p = p0 + vcol;
        rv = *(const dfloatx4_t*)(base + (long)min(vrow, tn - 1) * ld + v_col + min(p, dv - 4));
        if (p >= dv) rv = zero4;
        if (wave == 0) {
            const GT* gr = gates + (long)(start + t0 + min(lane, tn - 1)) * ldg + h;
            ra = to_f32(gr[a_off]);
            rb = to_f32(gr[b_off]);
        }
    };
    // one 16 x 16 tile of rows[i] . cols[j] over the key features
    auto dot_tile = [&](const float* rows, int i, const float* cols, int j) {
        dfloatx4_t a = zero4;
#pragma unroll
        for (int kb = 0; kb < NB; ++kb) {
            const dfloatx4_t x = *(const dfloatx4_t*)&rows[(16 * i + r) * DCHUNK_LN + 16 * kb + 4 * g];
            const dfloatx4_t z = *(const dfloatx4_t*)&cols[(16 * j + r) * DCHUNK_LN + 16 * kb + 4 * g];
#pragma unroll
            for (int e = 0; e < 4; ++e) a = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], z[e], a, 0, 0, 0);
        }
        return a;
    };
    // this wavefront's tokens 16 tt .. and columns 16 pt .. (with 16 columns only the first four have any)
    const int tt = PT == 2 ? wave >> 1 : wave & 3, pt = PT == 2 ? wave & 1 : 0;
    const bool owns = PT == 2 || wave < 4;
    fetch(0);
    for (int t0 = 0; t0 < q; t0 += DCHUNK_T) {
        const int tn = min(DCHUNK_T, q - t0);
#pragma unroll
        for (int i = 0; i < PT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) Ss[(16 * i + 4 * g + e) * DCHUNK_LN + n_own] = st[i][e];
        if (tn < DCHUNK_T) {                                           // rows behind the run's end repeat its last token
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if ((int)(threadIdx.x + 512 * i) >> 5 >= tn) rk[i] = zero4;
            if (vrow >= tn) rv = zero4;
        }
        float largest = 0.f, k2[4], q2[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = threadIdx.x + 512 * i, t = e >> 5, at = t * DCHUNK_LN + (e & 31) * 4;
            *(dfloatx4_t*)&Ks[at] = rk[i];
            *(dfloatx4_t*)&Qs[at] = rq[i];
            // a row's 128 features lie in 32 neighbouring lanes
            float sk = row16_sum(rk[i][0] * rk[i][0] + rk[i][1] * rk[i][1] + rk[i][2] * rk[i][2] + rk[i][3] * rk[i][3]);
            float sq = row16_sum(rq[i][0] * rq[i][0] + rq[i][1] * rq[i][1] + rq[i][2] * rq[i][2] + rq[i][3] * rq[i][3]);
            sk += __shfl_xor(sk, 16, 64);
            sq += __shfl_xor(sq, 16, 64);
            if ((lane & 31) == 0) {
                fk_s[t] = 1.0f / sqrtf(sk + 1e-6f);
                fq_s[t] = q_scale / sqrtf(sq + 1e-6f);
            }
            largest = fmaxf(largest, fmaxf(sk, sq));
            k2[i] = sk;
            q2[i] = sq;
        }
        if (__builtin_amdgcn_ballot_w64(largest == INFINITY)) {
            // a row whose square overflows counts as zero (its factor is), before products of it overflow too
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int e = threadIdx.x + 512 * i, at = (e >> 5) * DCHUNK_LN + (e & 31) * 4;
                if (k2[i] == INFINITY) *(dfloatx4_t*)&Ks[at] = rk[i] * 0.f;
                if (q2[i] == INFINITY) *(dfloatx4_t*)&Qs[at] = rq[i] * 0.f;
            }
        }
        if (vrow < DCHUNK_T) {
#pragma unroll
            for (int j = 0; j < 4; ++j) rT[(vcol + j) * DCHUNK_LT + vrow] = rv[j];
        }
        if (wave == 0) {
            // a token beyond the end has beta = 0 and g = 1: it neither writes nor forgets
            double la = lane < tn ? -(double)A * (double)decay_step(delta_softplus(ra + bias), A) : 0.0;
#pragma unroll
            for (int k = 1; k < 64; k <<= 1) {
                const double up = __shfl_up(la, k, 64);
                if (lane >= k) la += up;
            }
            const double all = __shfl(la, 63, 64);
            beta_s[lane] = lane < tn ? 1.0f / (1.0f + expf(-rb)) : 0.f;
            la_s[lane] = la;
            left_s[lane] = expf((float)(all - la));
            from_s[lane] = expf((float)la);
        }
        __syncthreads();
        if (t0 + DCHUNK_T < q) fetch(t0 + DCHUNK_T);
        // -A: the tiles on and below the diagonal, dealt to the wavefronts, first to those without a tile of their own
        for (int k = (wave + 4) & 7; k < 10; k += 8) {
            const int i = k < 1 ? 0 : (k < 3 ? 1 : (k < 6 ? 2 : 3)), j = k - i * (i + 1) / 2, s = 16 * j + r;
            const dfloatx4_t a = dot_tile(Ks, i, Ks, j);
            const double la = la_s[s];
            const float f = fk_s[s];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 16 * i + 4 * g + e;
                As[t * DCHUNK_LT + s] = s < t ? -beta_s[t] * fk_s[t] * f * a[e] * expf((float)(la_s[t] - la)) : 0.f;
            }
        }
        if (owns) {   // the right-hand side, in place of v
            const dfloatx4_t a = dot_tile(Ks, tt, Ss, pt);
            dfloatx4_t* at = (dfloatx4_t*)&rT[(16 * pt + r) * DCHUNK_LT + 16 * tt + 4 * g];
            dfloatx4_t v = *at;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 16 * tt + 4 * g + e;
                v[e] = beta_s[t] * (v[e] - from_s[t] * fk_s[t] * a[e]);
            }
            *at = v;
        }
        __syncthreads();
        if (wave == 7) {
            // lane (block g, column r) of the inverse of I + A: x_t = [t == r] - sum_(s < t) A[t, s] x_s
            float x[16];
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                float v = t == r ? 1.f : 0.f;
#pragma unroll
                for (int s = 0; s < t; ++s) v += As[(16 * g + t) * DCHUNK_LT + 16 * g + s] * x[s];
                x[t] = v;
            }
#pragma unroll
            for (int t = 0; t < 16; ++t) inv_s[(16 * g + t) * 20 + r] = x[t];
        }
        // what the state before the chunk gives this wavefront's tokens
        auto write_y = [&](const dfloatx4_t& v) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 16 * tt + 4 * g + e, p = 16 * pt + r;
                if (owns && t < tn && p0 + p < dv) y[(long)(start + t0 + t) * heads * dv + (long)h * dv + p0 + p] = v[e];
            }
        };
        dfloatx4_t yt = zero4;
        if (owns) yt = dot_tile(Qs, tt, Ss, pt);
#pragma unroll
        for (int e = 0; e < 4; ++e) yt[e] *= from_s[16 * tt + 4 * g + e] * fq_s[16 * tt + 4 * g + e];
        const dfloatx4_t y0 = yt;
        __syncthreads();
        if (wave < PT) {
            // u of columns 16 wave .. + 15, 16 tokens after 16 tokens
            const float* rhs_p = rT + (16 * wave + r) * DCHUNK_LT;
            float* u_p = uT + (16 * wave + r) * DCHUNK_LT;
            dfloatx4_t odd = zero4;
            for (int i = 0; i < 4; ++i) {
                dfloatx4_t rhs = *(const dfloatx4_t*)(rhs_p + 16 * i + 4 * g);
                for (int j = 0; j < i; ++j) {
                    const dfloatx4_t a = *(const dfloatx4_t*)&As[(16 * i + r) * DCHUNK_LT + 16 * j + 4 * g];
                    const dfloatx4_t x = *(const dfloatx4_t*)(u_p + 16 * j + 4 * g);
#pragma unroll
                    for (int e = 0; e < 4; ++e) rhs = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], x[e], rhs, 0, 0, 0);
                }
                // the accumulators (row 4 g + e, column r) lie where the operand (column r, index 4 g + e) is read
                const dfloatx4_t d = *(const dfloatx4_t*)&inv_s[(16 * i + r) * 20 + 4 * g];
                dfloatx4_t x = zero4;
#pragma unroll
                for (int e = 0; e < 4; ++e) x = __builtin_amdgcn_mfma_f32_16x16x4f32(d[e], rhs[e], x, 0, 0, 0);
                *(dfloatx4_t*)(u_p + 16 * i + 4 * g) = x;
                odd += x * 0.f;
                __builtin_amdgcn_wave_barrier();
            }
            if (wave_odd(odd[0], odd[1], odd[2], odd[3])) {
#pragma unroll 1
                for (int t = 0; t < DCHUNK_T; ++t) {
                    float sum = 0.f;
#pragma unroll 1
                    for (int s0 = 0; s0 < t; s0 += 4) {
                        const float term = As[t * DCHUNK_LT + s0 + g] * u_p[s0 + g];
                        sum += s0 + g < t ? term : 0.f;
                    }
                    sum += __shfl_xor(sum, 16, 64);
                    sum += __shfl_xor(sum, 32, 64);
                    if (g == 0) u_p[t] = rhs_p[t] + sum;
                    __builtin_amdgcn_wave_barrier();
                }
            }
        } else {
            for (int k = wave - PT; k < 10; k += 8 - PT) {
                const int i = k < 1 ? 0 : (k < 3 ? 1 : (k < 6 ? 2 : 3)), j = k - i * (i + 1) / 2, s = 16 * j + r;
                const dfloatx4_t a = dot_tile(Qs, i, Ks, j);
                const double la = la_s[s];
                const float f = fk_s[s];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int t = 16 * i + 4 * g + e;
                    Gs[t * DCHUNK_LT + s] = s <= t ? fq_s[t] * f * a[e] * expf((float)(la_s[t] - la)) : 0.f;
                }
            }
        }
        __syncthreads();
        // ... and what the chunk's own tokens give them
        for (int kb = 0; owns && kb <= tt; ++kb) {
            const dfloatx4_t a = *(const dfloatx4_t*)&Gs[(16 * tt + r) * DCHUNK_LT + 16 * kb + 4 * g];
            const dfloatx4_t u = *(const dfloatx4_t*)&uT[(16 * pt + r) * DCHUNK_LT + 16 * kb + 4 * g];
#pragma unroll
            for (int e = 0; e < 4; ++e) yt = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], u[e], yt, 0, 0, 0);
        }
        write_y(yt);
        // the state behind the chunk
        const float keep = from_s[DCHUNK_T - 1];
#pragma unroll
        for (int i = 0; i < PT; ++i) st[i] *= keep;
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
            const dfloatx4_t w4 = *(const dfloatx4_t*)&left_s[16 * kb + 4 * g] * *(const dfloatx4_t*)&fk_s[16 * kb + 4 * g];
            dfloatx4_t u4[PT];
#pragma unroll
            for (int i = 0; i < PT; ++i) u4[i] = *(const dfloatx4_t*)&uT[(16 * i + r) * DCHUNK_LT + 16 * kb + 4 * g] * w4;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float kv = Ks[(16 * kb + 4 * g + e) * DCHUNK_LN + n_own];
#pragma unroll
                for (int i = 0; i < PT; ++i) st[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(u4[i][e], kv, st[i], 0, 0, 0);
            }
        }
        if (wave_odd(yt[0], yt[1], yt[2], yt[3])) {
            dfloatx4_t again = y0;
#pragma unroll 1
            for (int s = 0; s < DCHUNK_T; ++s) {
                const float one = uT[(16 * pt + r) * DCHUNK_LT + s];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int t = 16 * tt + 4 * g + e;
                    if (s <= t) again[e] += Gs[t * DCHUNK_LT + s] * one;
                }
            }
            write_y(again);
        }
        __syncthreads();
    }
    if (write_state) {
#pragma unroll
        for (int i = 0; i < PT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int p = 16 * i + 4 * g + e;
                if (p0 + p < dv && n_own < dk) sp[(long)p * dk + n_own] = st[i][e];
            }
    }
}

// The n_chunked sequences that bring at least chunk_from tokens are taken in chunks, the others are walked: two launches
// where there are both.  (0, 0: all are walked, as they are under the rules and sizes that the chunks' kernel does not take.)
extern "C" const char* cpmcu_delta_scan(const float* qkv, long ld, const void* gates, long ldg, int gate_dtype,
                                        long a_off, long b_off, const float* chan_a, long ld_a, const float* dt_bias,
                                        const float* A_log, float* state, float* y, const int* cu_q,
                                        const int* seq_slot, int n_rows, int n_seqs, int heads, int kv_heads, int dk, int dv,
                                        float q_scale, int write_state, int lanes, int rule, int chunk_from,
                                        int n_chunked, hipStream_t stream) {
    CPMCU_REQUIRE(rule == RULE_DELTA || rule == RULE_CHANNEL || rule == RULE_DECAY, "delta_scan: unknown rule %d", rule);
    CPMCU_REQUIRE(n_seqs > 0 && heads > 0 && kv_heads > 0 && dk > 0 && dv > 0, "delta_scan: empty shape");
    CPMCU_REQUIRE(heads % kv_heads == 0, "delta_scan: %d heads are not a multiple of %d key heads", heads, kv_heads);
    CPMCU_REQUIRE(dk <= 256, "delta_scan: a key size of %d is not supported (at most 256)", dk);
    CPMCU_REQUIRE(ld >= 2L * kv_heads * dk + (long)heads * dv, "delta_scan: rows of %ld too short", ld);
    CPMCU_REQUIRE(rule == RULE_DECAY || (gates && b_off >= 0 && ldg >= b_off + heads), "delta_scan: gate rows too short");
    CPMCU_REQUIRE(rule != RULE_DELTA || (a_off >= 0 && ldg >= a_off + heads), "delta_scan: gate rows too short");
    CPMCU_REQUIRE(rule != RULE_CHANNEL || (chan_a && ld_a >= (long)heads * dk), "delta_scan: channel decay rows too short");
    CPMCU_REQUIRE(A_log && (rule == RULE_DECAY || dt_bias), "delta_scan: decay constants missing");
    CPMCU_REQUIRE(lanes == 0 || lanes == 8 || lanes == 16, "delta_scan: %d lanes a column (0: chosen here, 8 or 16)", lanes);
    CPMCU_REQUIRE(chunk_from >= 0 && n_chunked >= 0 && n_chunked <= n_seqs, "delta_scan: %d sequences of %d in chunks", n_chunked, n_seqs);
    CPMCU_REQUIRE((long)n_seqs * heads < (1L << 31), "delta_scan: shape exceeds the launch grid");
    if (!(rule == RULE_DELTA && lanes == 0 && dk <= DCHUNK_N && dk % 4 == 0 && dv % 4 == 0 && ld % 4 == 0 &&
          (uintptr_t)qkv % 16 == 0 && (gate_dtype == CPMCU_F32 || gate_dtype == CPMCU_BF16)))
        n_chunked = 0;
    if (n_chunked > 0) {
        // 32 columns a workgroup share the products among keys and queries; 16 where 32 would leave CUs without one (a
        // workgroup's LDS leaves a CU one at a time)
        const bool narrow = (long)n_chunked * heads * ((dv + 31) / 32) < 256;
        const dim3 grid(heads * n_chunked, narrow ? (dv + 15) / 16 : (dv + 31) / 32);
        const int hi = n_chunked < n_seqs ? 0x7fffffff : 0;
        CPMCU_REQUIRE(grid.y <= 65535, "delta_scan: shape exceeds the launch grid");
#define CHUNKS(NBv, GTv)                                       \
    do {                                                       \
        if (narrow) CHUNKS_OF(NBv, 1, GTv);                    \
        else CHUNKS_OF(NBv, 2, GTv);                           \
    } while (0)
#define CHUNKS_OF(NBv, PTv, GTv)                                                                                               \
    delta_chunk_kernel<NBv, PTv, GTv><<<grid, 512, 0, stream>>>(qkv, ld, (const GTv*)gates, ldg, a_off, b_off, dt_bias, A_log, \
                                                           state, y, cu_q, seq_slot, heads, kv_heads, dk, dv, q_scale,    \
                                                           write_state, n_seqs, chunk_from, hi)
        if (gate_dtype == CPMCU_F32) {
            if (dk <= 64) CHUNKS(4, float);
            else CHUNKS(8, float);
        } else {
            if (dk <= 64) CHUNKS(4, bf16_t);
            else CHUNKS(8, bf16_t);
        }
#undef CHUNKS
#undef CHUNKS_OF
        CPMCU_LAUNCH_CHECK("delta_chunk");
        if (n_chunked == n_seqs) return nullptr;
    }
    const int n_walked = n_seqs - n_chunked, lo = 0, hi = n_chunked > 0 ? chunk_from : 0;
    // 16 lanes a column where 8 would leave fewer than two workgroups a compute unit and a column is long enough
    if (lanes == 0) lanes = ((long)n_walked * heads * ((dv + 31) / 32) < 512 && dk > 16 && dv > 16) ? 16 : 8;
    const int cols = 256 / lanes;
    const int pb = (dv + cols - 1) / cols;
    CPMCU_REQUIRE(pb <= 65535, "delta_scan: shape exceeds the launch grid");
    dim3 grid(heads * n_walked, pb);
    const int need = (dk + lanes - 1) / lanes;
    const bool one = n_rows == n_seqs && n_chunked == 0;                // as a step of decoding does
#define LAUNCH(NRv, TTv, Lv, GTv, Rv)                                                                                \
    if (one)                                                                                                          \
        delta_step_kernel<NRv, 256 / TTv, Lv, GTv, Rv><<<grid, 256, 0, stream>>>(qkv, ld, (const GTv*)gates, ldg, a_off, b_off, \
                                                                                 chan_a, ld_a, dt_bias, A_log, state, y, cu_q, \
                                                                                 seq_slot, heads, kv_heads, dk, dv, q_scale, write_state); \
    else delta_scan_kernel<NRv, TTv, Lv, GTv, Rv><<<grid, 256, 0, stream>>>(qkv, ld, (const GTv*)gates, ldg, a_off, b_off, \
                                                                       chan_a, ld_a, dt_bias, A_log, state, y, cu_q,  \
                                                                       seq_slot, heads, kv_heads, dk, dv, q_scale,    \
                                                                       write_state, n_seqs, lo, hi)
#define BY_NR(GTv, Rv)                                              \
    do {                                                            \
        if (lanes == 16) {                                          \
            if (need <= 2) { LAUNCH(2, 32, 16, GTv, Rv); }          \
            else if (need <= 4) { LAUNCH(4, 32, 16, GTv, Rv); }     \
            else if (need <= 8) { LAUNCH(8, 32, 16, GTv, Rv); }     \
            else { LAUNCH(16, 16, 16, GTv, Rv); }                   \
        } else {                                                    \
            if (need <= 2) { LAUNCH(2, 32, 8, GTv, Rv); }           \
            else if (need <= 4) { LAUNCH(4, 32, 8, GTv, Rv); }      \
            else if (need <= 8) { LAUNCH(8, 32, 8, GTv, Rv); }      \
            else if (need <= 16) { LAUNCH(16, 32, 8, GTv, Rv); }    \
            else { LAUNCH(32, 16, 8, GTv, Rv); }                    \
        }                                                           \
    } while (0)
    if (rule == RULE_DECAY) BY_NR(float, RULE_DECAY);
    else if (gate_dtype == CPMCU_F32 && rule == RULE_DELTA) BY_NR(float, RULE_DELTA);
    else if (gate_dtype == CPMCU_BF16 && rule == RULE_DELTA) BY_NR(bf16_t, RULE_DELTA);
    else if (gate_dtype == CPMCU_F32) BY_NR(float, RULE_CHANNEL);
    else if (gate_dtype == CPMCU_BF16) BY_NR(bf16_t, RULE_CHANNEL);
    else CPMCU_FAIL("delta_scan: unknown dtype %d", gate_dtype);
#undef BY_NR
#undef LAUNCH
    CPMCU_LAUNCH_CHECK("delta_scan");
    return nullptr;
}

// What linear attention puts between its input projection and the recurrence, in float: from a projection's rows
// (q heads at column q_off, k heads at k_off, heads x dk each; v heads at v_off, heads x dv) to rows [q | k | v] of
// float.  With silu, all three pass z sigmoid(z); the first rot_dims features of q and k heads are rotated by
// position * inv_freq[i] (pairs (i, i + rot_dims/2), or (2i, 2i + 1) when interleaved); k is multiplied by k_scale
// afterwards.  grid (tokens, heads), 64 threads.
template <typename T>
__global__ __launch_bounds__(64) void linear_attention_prepare_kernel(const T* __restrict__ proj, long ld, long q_off,
                                                                      long k_off, long v_off, float* __restrict__ out,
                                                                      int heads, int dk, int dv, int silu, int rot_dims,
                                                                      int interleaved, const float* __restrict__ inv_freq,
                                                                      const int* __restrict__ positions, float k_scale) {
    const long t = blockIdx.x;
    const int h = blockIdx.y, lane = threadIdx.x;
    const T* row = proj + t * ld;
    const long ow = 2L * heads * dk + (long)heads * dv;
    float* o = out + t * ow;
    auto act = [&](float z) { return silu ? z / (1.0f + expf(-z)) : z; };
    const float pos = rot_dims ? (float)positions[t] : 0.f;
    const int half = rot_dims / 2;
#pragma unroll
    for (int which = 0; which < 2; ++which) {
        const T* src = row + (which ? k_off : q_off) + (long)h * dk;
        float* dst = o + (which ? (long)heads * dk : 0) + (long)h * dk;
        const float mul = which ? k_scale : 1.0f;
        for (int i = lane; i < half; i += 64) {
            const float ang = pos * inv_freq[i];
            const float cs = cosf(ang), sn = sinf(ang);
            const int ia = interleaved ? 2 * i : i, ib = interleaved ? 2 * i + 1 : i + half;
            const float u = act(to_f32(src[ia])), v = act(to_f32(src[ib]));
            dst[ia] = (u * cs - v * sn) * mul;
            dst[ib] = (v * cs + u * sn) * mul;
        }
        for (int i = rot_dims + lane; i < dk; i += 64) dst[i] = act(to_f32(src[i])) * mul;
    }
    const T* vsrc = row + v_off + (long)h * dv;
    float* vdst = o + 2L * heads * dk + (long)h * dv;
    for (int i = lane; i < dv; i += 64) vdst[i] = act(to_f32(vsrc[i]));
}

extern "C" const char* cpmcu_linear_attention_prepare(const void* proj, int dtype, long ld, long q_off, long k_off,
                                                      long v_off, float* out, int n, int heads, int dk, int dv, int silu,
                                                      int rot_dims, int interleaved, const float* inv_freq,
                                                      const int* positions, float k_scale, hipStream_t stream) {
    CPMCU_REQUIRE(n > 0 && heads > 0 && dk > 0 && dv > 0, "linear_attention_prepare: empty shape");
    CPMCU_REQUIRE(heads <= 65535, "linear_attention_prepare: %d heads exceed the launch grid", heads);
    CPMCU_REQUIRE(rot_dims >= 0 && rot_dims % 2 == 0 && rot_dims <= dk && (rot_dims == 0 || (inv_freq && positions)),
                  "linear_attention_prepare: %d rotated features of %d", rot_dims, dk);
    CPMCU_REQUIRE(q_off >= 0 && k_off >= 0 && v_off >= 0 && ld >= q_off + (long)heads * dk && ld >= k_off + (long)heads * dk &&
                  ld >= v_off + (long)heads * dv, "linear_attention_prepare: rows of %ld too short", ld);
    dim3 grid(n, heads);
    if (dtype == CPMCU_F32)
        linear_attention_prepare_kernel<float><<<grid, 64, 0, stream>>>((const float*)proj, ld, q_off, k_off, v_off, out, heads,
                                                                        dk, dv, silu, rot_dims, interleaved, inv_freq,
                                                                        positions, k_scale);
    else if (dtype == CPMCU_BF16)
        linear_attention_prepare_kernel<bf16_t><<<grid, 64, 0, stream>>>((const bf16_t*)proj, ld, q_off, k_off, v_off, out,
                                                                         heads, dk, dv, silu, rot_dims, interleaved, inv_freq,
                                                                         positions, k_scale);
    else
        CPMCU_FAIL("linear_attention_prepare: unknown dtype %d", dtype);
    CPMCU_LAUNCH_CHECK("linear_attention_prepare");
    return nullptr;
}
