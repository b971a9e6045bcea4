// A feed-forward of routed experts, for steps of any number of tokens and both element types:
//
//  * moe_logits_kernel, moe_select_kernel: router logits z = Wr h in float (Wr float [E, H]), a wavefront a row,
//    into scratch; then, a wavefront a token: s = softmax(z) over the experts, or sigmoid(z) of each (score_fn);
//    choice scores c = s + correction; the experts form `n_groups` equal groups of neighbours, a group's score is
//    its largest c, or the sum of its two largest (group_fn), and only experts of the `keep_groups` best groups may be
//    chosen (n_groups = 1: any; the others' c count as -inf); the `top` largest c are chosen (ties: the lower index),
//    their weights are s / (sum of the chosen s + 1e-20) * weight_scale, or s * weight_scale without `normalize`.  A bias
//    may be added to the logits first; with MOE_SCORE_LOGIT the choice goes by the logits themselves (+ correction) and
//    the weights are the softmax of the chosen ones among themselves, * weight_scale.  The
//    router may have more rows than there are experts with matrices: the rows behind those are identity experts,
//    whose output is h_t itself; the kernels below skip them and the last one adds their share.  With w_sg (float [H]) it also
//    gives sigmoid(w_sg . h), the gate of an expert that every token uses.
//  * moe_gated_kernel: act[t, k, :] = act(Wg_e h_t) * (Wu_e h_t) for the k-th chosen expert e of token t (the
//    nonlinearities of common.h: SiLU, or the clamped swish with its limit); the experts' gate and up rows are
//    stacked: wgu [E, 2F, H], gate rows first.
//  * moe_up_kernel: the same for experts without a gate, act[t, k, :] = act(Wu_e h_t); wu [E, F, H].
//  * moe_down_kernel: out[t] = sum_k w[t, k] Wd_e act[t, k] (+ sg[t] * shared[t]); wd [E, H, F]; float out.  With a
//    residual (Join) the layer's sum ends here: x[t] += out[t] + another result of the layer (float partial sums or
//    one bf16 / float tensor, and a bias), in place, and x once more in the activations' type for a product that
//    reads it; nothing else is written.
//
// A wavefront owns output rows and its lanes stride over the input features (16-byte loads when the rows are
// aligned), so an expert's weights stream once for every token that chose it: the form for steps of few tokens.
#include "lds_direct.h"
#include "moe_product.h"

#include <type_traits>

#define MOE_MAX_EXPERTS 1024
enum { MOE_SCORE_SOFTMAX = 0, MOE_SCORE_SIGMOID = 1, MOE_SCORE_LOGIT = 2 };
enum { MOE_GROUP_MAX = 0, MOE_GROUP_TOP2_SUM = 1 };

// Where a layer's sum ends: the residual x [n, H], another result `a` to add (parts `stride` apart; may be absent) with
// an optional bias, and a copy of the new x in the activations' type (may be absent)
struct Join {
    float* x;
    const void* a;
    int a_bf16, a_parts;
    long a_stride;
    const float* a_bias;
    void* copy;
};
__device__ inline float join_part(const Join& j, int p, long i) {
    return j.a_bf16 ? to_f32(((const bf16_t*)j.a)[p * j.a_stride + i]) : ((const float*)j.a)[p * j.a_stride + i];
}

template <typename T> struct Vec8;
template <> struct Vec8<bf16_t> { typedef uint4 type; };
template <> struct Vec8<float> { struct type { float4 a, b; }; };

template <typename T>
__device__ inline void load8(const T* p, float* v);
template <>
__device__ inline void load8<bf16_t>(const bf16_t* p, float* v) {
    const uint4 u = *(const uint4*)p;
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = __uint_as_float(w[i] << 16);
        v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
}
template <>
__device__ inline void load8<float>(const float* p, float* v) {
    const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

// the same for an expert's weights, which a step reads once: past the caches, where nothing else of them would be found
__device__ inline void stream8(const bf16_t* p, float* v) {
    typedef uint32_t words_t __attribute__((ext_vector_type(4)));
    const words_t w = __builtin_nontemporal_load((const words_t*)p);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = __uint_as_float(w[i] << 16);
        v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
}
__device__ inline void stream8(const float* p, float* v) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        typedef float floats_t __attribute__((ext_vector_type(4)));
        const floats_t w = __builtin_nontemporal_load((const floats_t*)p + i);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[4 * i + j] = w[j];
    }
}

// the lane's share of dot(a[0:K], b[0:K]); `vec`: both rows are 16-byte aligned (32 for float) and K % 8 == 0
template <typename TA, typename TB>
__device__ inline float lane_dot(const TA* __restrict__ a, const TB* __restrict__ b, int K, int lane, bool vec) {
    float s = 0.f;
    if (vec) {
        for (int c = lane * 8; c < K; c += 64 * 8) {
            float x[8], y[8];
            load8<TA>(a + c, x);
            load8<TB>(b + c, y);
#pragma unroll
            for (int i = 0; i < 8; ++i) s += x[i] * y[i];
        }
    } else {
        for (int c = lane; c < K; c += 64) s += to_f32(a[c]) * to_f32(b[c]);
    }
    return s;
}

__device__ inline float wave_min_f(float v) { return -wave_max(-v); }

// grid (tokens, ceil((E + 1) / 4)), 256 threads: a wavefront a row of the router (row E: the shared expert's gate);
// logits float [n, E + 1]
template <typename T>
__global__ __launch_bounds__(256) void moe_logits_kernel(const T* __restrict__ h, long ldh, const float* __restrict__ wr,
                                                         const float* __restrict__ w_sg, int H, int E,
                                                         float* __restrict__ logits) {
    const long t = blockIdx.x;
    const int lane = threadIdx.x & 63;
    const int e = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (e > E || (e == E && !w_sg)) return;
    const T* hr = h + t * ldh;
    const float* row = e < E ? wr + (long)e * H : w_sg;
    const bool vec = (H % 8 == 0) && (ldh % 8 == 0) && ((uintptr_t)h % 32 == 0) && ((uintptr_t)row % 32 == 0);
    const float s = wave_sum(lane_dot<T, float>(hr, row, H, lane, vec));
    if (lane == 0) logits[t * (E + 1) + e] = s;
}

// grid (tokens), 64 threads: softmax, groups, the top choices and their weights from a row of logits
__global__ __launch_bounds__(64) void moe_select_kernel(const float* __restrict__ logits,
                                                        const float* __restrict__ bias,
                                                        const float* __restrict__ correction, int has_sg, int E,
                                                        int n_groups, int keep_groups, int top, int* __restrict__ idx_out,
                                                        float* __restrict__ w_out, float* __restrict__ sg_out,
                                                        int score_fn, int group_fn, float weight_scale, int normalize) {
    __shared__ float z[MOE_MAX_EXPERTS];      // logits, then softmax scores
    __shared__ float c[MOE_MAX_EXPERTS];      // choice scores; -inf once an expert is chosen or shut out
    __shared__ float gs[MOE_MAX_EXPERTS];     // group scores
    const long t = blockIdx.x;
    const int lane = threadIdx.x;
    const float* zr = logits + t * (E + 1);
    if (has_sg && lane == 0) sg_out[t] = 1.0f / (1.0f + expf(-zr[E]));
    if (score_fn == MOE_SCORE_SIGMOID) {
        for (int e = lane; e < E; e += 64) {
            z[e] = 1.0f / (1.0f + expf(-(zr[e] + (bias ? bias[e] : 0.f))));
            c[e] = z[e] + (correction ? correction[e] : 0.f);
        }
    } else {
        float mx = -INFINITY;
        for (int e = lane; e < E; e += 64) {
            z[e] = zr[e] + (bias ? bias[e] : 0.f);
            mx = fmaxf(mx, z[e]);
        }
        mx = wave_max(mx);
        float sum = 0.f;
        for (int e = lane; e < E; e += 64) {
            const float p = expf(z[e] - mx);
            if (score_fn == MOE_SCORE_LOGIT) c[e] = z[e] + (correction ? correction[e] : 0.f);
            z[e] = p;
            sum += p;
        }
        if (score_fn == MOE_SCORE_SOFTMAX) {
            sum = wave_sum(sum);
            const float inv = 1.0f / sum;
            for (int e = lane; e < E; e += 64) {
                z[e] *= inv;
                c[e] = z[e] + (correction ? correction[e] : 0.f);
            }
        }
    }
    __builtin_amdgcn_wave_barrier();
    if (n_groups > 1) {
        const int per = E / n_groups;
        for (int g = lane; g < n_groups; g += 64) {
            // the largest and the second largest choice score of the group
            float b = -INFINITY, b2 = -INFINITY;
            for (int i = 0; i < per; ++i) {
                const float v = c[g * per + i];
                if (v > b) {
                    b2 = b;
                    b = v;
                } else if (v > b2) {
                    b2 = v;
                }
            }
            gs[g] = (group_fn == MOE_GROUP_TOP2_SUM && per > 1) ? b + b2 : b;
        }
        __builtin_amdgcn_wave_barrier();
        // the best groups, one a turn, are marked with +inf; afterwards every other group's experts are shut out
        for (int r = 0; r < keep_groups; ++r) {
            float b = -INFINITY;
            for (int g = lane; g < n_groups; g += 64)
                if (gs[g] != INFINITY) b = fmaxf(b, gs[g]);
            b = wave_max(b);
            float first = 3.0e38f;
            for (int g = lane; g < n_groups; g += 64)
                if (gs[g] != INFINITY && gs[g] == b) first = fminf(first, (float)g);
            const int win = (int)wave_min_f(first);
            if (lane == 0) gs[win] = INFINITY;
            __builtin_amdgcn_wave_barrier();
        }
        for (int e = lane; e < E; e += 64)
            if (gs[e / per] != INFINITY) c[e] = -INFINITY;
        __builtin_amdgcn_wave_barrier();
    }
    float chosen_sum = 0.f;
    for (int r = 0; r < top; ++r) {
        float b = -INFINITY;
        for (int e = lane; e < E; e += 64) b = fmaxf(b, c[e]);
        b = wave_max(b);
        float first = 3.0e38f;
        for (int e = lane; e < E; e += 64)
            if (c[e] == b) first = fminf(first, (float)e);
        const int win = (int)wave_min_f(first);
        chosen_sum += z[win];
        if (lane == 0) {
            idx_out[t * top + r] = win;
            w_out[t * top + r] = z[win];
            c[win] = -INFINITY;
        }
        __builtin_amdgcn_wave_barrier();
    }
    const float norm = normalize ? weight_scale / (chosen_sum + 1e-20f) : weight_scale;
    for (int r = lane; r < top; r += 64) w_out[t * top + r] *= norm;
}

extern "C" const char* cpmcu_moe_route(const void* h, long ldh, int dtype, const float* wr, const float* bias,
                                       const float* correction,
                                       const float* w_sg, int n, int H, int E, int n_groups, int keep_groups, int top,
                                       float* logits, int* idx_out, float* w_out, float* sg_out, int score_fn,
                                       int group_fn, float weight_scale, int normalize, int logits_ready,
                                       hipStream_t stream) {
    CPMCU_REQUIRE((score_fn == MOE_SCORE_SOFTMAX || score_fn == MOE_SCORE_SIGMOID || score_fn == MOE_SCORE_LOGIT) &&
                  (group_fn == MOE_GROUP_MAX || group_fn == MOE_GROUP_TOP2_SUM),
                  "moe_route: unknown score function %d or group score %d", score_fn, group_fn);
    CPMCU_REQUIRE(n > 0 && H > 0 && E > 0 && logits, "moe_route: empty shape");
    CPMCU_REQUIRE(E <= MOE_MAX_EXPERTS, "moe_route: %d experts (up to %d are taken)", E, MOE_MAX_EXPERTS);
    CPMCU_REQUIRE(n_groups >= 1 && E % n_groups == 0 && keep_groups >= 1 && keep_groups <= n_groups,
                  "moe_route: %d experts in %d groups of which %d may be chosen from", E, n_groups, keep_groups);
    CPMCU_REQUIRE(top >= 1 && top <= keep_groups * (E / n_groups), "moe_route: %d experts a token of %d that may be chosen",
                  top, keep_groups * (E / n_groups));
    CPMCU_REQUIRE(!w_sg || sg_out, "moe_route: a place for the shared gate is missing");
    dim3 grid(n, (E + 1 + 3) / 4);
    if (logits_ready) {
        // the rows of logits come from a product of the caller's
    } else if (dtype == CPMCU_F32)
        moe_logits_kernel<float><<<grid, 256, 0, stream>>>((const float*)h, ldh, wr, w_sg, H, E, logits);
    else if (dtype == CPMCU_BF16)
        moe_logits_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)h, ldh, wr, w_sg, H, E, logits);
    else
        CPMCU_FAIL("moe_route: unknown dtype %d", dtype);
    CPMCU_LAUNCH_CHECK("moe_logits");
    moe_select_kernel<<<n, 64, 0, stream>>>(logits, bias, correction, w_sg ? 1 : 0, E, n_groups, keep_groups, top, idx_out, w_out,
                                            sg_out, score_fn, group_fn, weight_scale, normalize);
    CPMCU_LAUNCH_CHECK("moe_select");
    return nullptr;
}

#define MOE_ROWS 4       // output rows a wavefront (moe_down_kernel names its four)

// grid (ceil(F / 16), tokens * top), 256 threads: wavefront w takes rows [16 x + 4 w, +4) of the expert's F, gate and up
// rows together, for all pairs of its run of 128 that chose the expert, up to 4 at a time against the same weights; the
// workgroups of the expert's other pairs in the run end at once.  The weights bound it: 8 tokens with 6 of 64 experts of
// 1,408 at width 4,096 (48 pairs, 35 experts) 179 -> 151 us, 5.4 TB/s; 15 tokens 283 -> 192, one token 41 -> 31.  A
// pair's sums do not depend on which others share its expert.
// An expert's workgroups are neighbours in the grid and so are dealt to all 8 XCDs alike: with the pairs first, 48 of them
// gave XCD i the experts of pairs i, i + 8, ..., of which only the first of each expert's
// have work: 8 tokens 148 -> 127 us (6.5 TB/s), 16 tokens 252 -> 178, 4 tokens 80 -> 76, 2 tokens and 1 the same.
#define MOE_RUN 128
#define MOE_GRID_Y 32768

template <typename T, int NT>
__device__ inline void gated_rows(const T* __restrict__ h, long ldh, const T* __restrict__ wg, const long (&pair)[4],
                                  T* __restrict__ act, int H, int F, int top, int act_fn, float act_limit, int j0, int lane,
                                  bool vec) {
    const T *wr[8], *hr[NT];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        wr[r] = wg + (long)min(j0 + r, F - 1) * H;
        wr[4 + r] = wg + (long)(F + min(j0 + r, F - 1)) * H;
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) hr[i] = h + pair[i] / top * ldh;
    float s[NT][8];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int r = 0; r < 8; ++r) s[i][r] = 0.f;
    if (vec) {
        for (int c = lane * 8; c < H; c += 64 * 8) {
            float y[8][8];
#pragma unroll
            for (int r = 0; r < 8; ++r) stream8(wr[r] + c, y[r]);
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                float x[8];
                load8<T>(hr[i] + c, x);
#pragma unroll
                for (int r = 0; r < 8; ++r)
#pragma unroll
                    for (int k = 0; k < 8; ++k) s[i][r] += y[r][k] * x[k];
            }
        }
    } else {
        for (int c = lane; c < H; c += 64) {
            float y[8];
#pragma unroll
            for (int r = 0; r < 8; ++r) y[r] = to_f32(wr[r][c]);
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                const float x = to_f32(hr[i][c]);
#pragma unroll
                for (int r = 0; r < 8; ++r) s[i][r] += y[r] * x;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
#pragma unroll
        for (int r = 0; r < 8; ++r) s[i][r] = wave_sum(s[i][r]);
        float g = s[i][0], u = s[i][4];
#pragma unroll
        for (int r = 1; r < 4; ++r)
            if (lane == r) {
                g = s[i][r];
                u = s[i][4 + r];
            }
        gate_prepare(g, u, act_fn, act_limit);
        if (lane < 4 && j0 + lane < F) act[pair[i] * F + j0 + lane] = from_f32<T>(gate_act(g, act_fn) * u);
    }
}

template <typename T>
__global__ __launch_bounds__(256) void moe_gated_kernel(const T* __restrict__ h, long ldh, const T* __restrict__ wgu,
                                                        const int* __restrict__ idx, T* __restrict__ act, int H, int F,
                                                        int top, int E, int n_pairs, int act_fn, float act_limit) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int p0 = blockIdx.z * MOE_GRID_Y + blockIdx.y;
    if (p0 >= n_pairs) return;
    const int run0 = p0 / MOE_RUN * MOE_RUN, own = p0 - run0;
    const int a = run0 + lane < n_pairs ? idx[run0 + lane] : -1, b = run0 + 64 + lane < n_pairs ? idx[run0 + 64 + lane] : -1;
    const int e = own < 64 ? __builtin_amdgcn_readlane(a, own & 63) : __builtin_amdgcn_readlane(b, own & 63);
    if (e >= E) return;                 // an identity expert
    unsigned long long first = __builtin_amdgcn_ballot_w64(a == e), second = __builtin_amdgcn_ballot_w64(b == e);
    if ((first ? __builtin_ctzll(first) : 64 + __builtin_ctzll(second)) != own) return;
    const int j0 = blockIdx.x * 4 * MOE_ROWS + wave * MOE_ROWS;
    if (j0 >= F) return;
    const T* wg = wgu + (long)e * 2 * F * H;
    const bool vec = (H % 8 == 0) && (ldh % 8 == 0) && ((uintptr_t)h % 32 == 0) && ((uintptr_t)wgu % 32 == 0);
    auto next = [&]() {
        unsigned long long& from = first ? first : second;
        const int at = __builtin_ctzll(from) + (first ? 0 : 64);
        from &= from - 1;
        return (long)(run0 + at);
    };
    while (first | second) {
        long pair[4];
        int count = 0;
        pair[0] = pair[1] = pair[2] = pair[3] = next();
        for (count = 1; count < 4 && (first | second); ++count) {
            const long p = next();
            if (count == 1) pair[1] = pair[2] = pair[3] = p;
            else if (count == 2) pair[2] = pair[3] = p;
            else pair[3] = p;
        }
        if (count == 1) gated_rows<T, 1>(h, ldh, wg, pair, act, H, F, top, act_fn, act_limit, j0, lane, vec);
        else if (count == 2) gated_rows<T, 2>(h, ldh, wg, pair, act, H, F, top, act_fn, act_limit, j0, lane, vec);
        else gated_rows<T, 4>(h, ldh, wg, pair, act, H, F, top, act_fn, act_limit, j0, lane, vec);
    }
}

extern "C" const char* cpmcu_moe_gated(const void* h, long ldh, int dtype, const void* wgu, const int* idx, void* act,
                                       int n, int H, int F, int top, int E, int act_fn, float act_limit,
                                       hipStream_t stream) {
    CPMCU_REQUIRE(n > 0 && H > 0 && F > 0 && top > 0 && E > 0, "moe_gated: empty shape");
    CPMCU_REQUIRE(CPMCU_ACT_KNOWN(act_fn), "moe_gated: unknown nonlinearity %d", act_fn);
    const int fy = (F + 4 * MOE_ROWS - 1) / (4 * MOE_ROWS);
    CPMCU_REQUIRE(fy <= 65535, "moe_gated: %d rows an expert exceed the launch grid", F);
    const long pairs = (long)n * top;
    CPMCU_REQUIRE(pairs < (1L << 31), "moe_gated: %ld pairs", pairs);
    const dim3 grid(fy, (unsigned)(pairs < MOE_GRID_Y ? pairs : MOE_GRID_Y), (unsigned)((pairs + MOE_GRID_Y - 1) / MOE_GRID_Y));
    if (dtype == CPMCU_F32)
        moe_gated_kernel<float><<<grid, 256, 0, stream>>>((const float*)h, ldh, (const float*)wgu, idx, (float*)act, H, F, top, E, (int)pairs, act_fn, act_limit);
    else if (dtype == CPMCU_BF16)
        moe_gated_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)h, ldh, (const bf16_t*)wgu, idx, (bf16_t*)act, H, F, top, E, (int)pairs, act_fn, act_limit);
    else
        CPMCU_FAIL("moe_gated: unknown dtype %d", dtype);
    CPMCU_LAUNCH_CHECK("moe_gated");
    return nullptr;
}

// grid (tokens * top, ceil(F / 16)), 256 threads: a wavefront takes 4 rows of the expert's F and reads them together,
// against one piece of the token's row
template <typename T>
__global__ __launch_bounds__(256) void moe_up_kernel(const T* __restrict__ h, long ldh, const T* __restrict__ wu,
                                                     const int* __restrict__ idx, T* __restrict__ act, int H, int F,
                                                     int top, int E, int act_fn) {
    const long pair = blockIdx.x;
    const long t = pair / top;
    const int e = idx[pair];
    if (e >= E) return;                 // an identity expert
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int j0 = blockIdx.y * 4 * MOE_ROWS + wave * MOE_ROWS;
    if (j0 >= F) return;
    const T* hr = h + t * ldh;
    const T* w = wu + (long)e * F * H;
    const bool vec = (H % 8 == 0) && (ldh % 8 == 0) && ((uintptr_t)h % 32 == 0) && ((uintptr_t)wu % 32 == 0);
    const T *w0 = w + (long)j0 * H, *w1 = w + (long)min(j0 + 1, F - 1) * H, *w2 = w + (long)min(j0 + 2, F - 1) * H,
            *w3 = w + (long)min(j0 + 3, F - 1) * H;
    float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
    if (vec) {
#pragma unroll 2
        for (int c = lane * 8; c < H; c += 64 * 8) {
            float x[8], y0[8], y1[8], y2[8], y3[8];
            load8<T>(w0 + c, y0);
            load8<T>(w1 + c, y1);
            load8<T>(w2 + c, y2);
            load8<T>(w3 + c, y3);
            load8<T>(hr + c, x);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                s0 += x[i] * y0[i];
                s1 += x[i] * y1[i];
                s2 += x[i] * y2[i];
                s3 += x[i] * y3[i];
            }
        }
    } else {
        for (int c = lane; c < H; c += 64) {
            const float x = to_f32(hr[c]);
            s0 += x * to_f32(w0[c]);
            s1 += x * to_f32(w1[c]);
            s2 += x * to_f32(w2[c]);
            s3 += x * to_f32(w3[c]);
        }
    }
    s0 = wave_sum(s0);
    s1 = wave_sum(s1);
    s2 = wave_sum(s2);
    s3 = wave_sum(s3);
    if (lane < 4 && j0 + lane < F)
        act[pair * F + j0 + lane] = from_f32<T>(plain_act(lane == 0 ? s0 : (lane == 1 ? s1 : (lane == 2 ? s2 : s3)), act_fn));
}

extern "C" const char* cpmcu_moe_up(const void* h, long ldh, int dtype, const void* wu, const int* idx, void* act, int n,
                                    int H, int F, int top, int E, int act_fn, hipStream_t stream) {
    CPMCU_REQUIRE(n > 0 && H > 0 && F > 0 && top > 0 && E > 0, "moe_up: empty shape");
    CPMCU_REQUIRE(CPMCU_PLAIN_ACT_KNOWN(act_fn), "moe_up: unknown nonlinearity %d", act_fn);
    const int fy = (F + 4 * MOE_ROWS - 1) / (4 * MOE_ROWS);
    CPMCU_REQUIRE(fy <= 65535, "moe_up: %d rows an expert exceed the launch grid", F);
    dim3 grid((unsigned)((long)n * top), fy);
    if (dtype == CPMCU_F32)
        moe_up_kernel<float><<<grid, 256, 0, stream>>>((const float*)h, ldh, (const float*)wu, idx, (float*)act, H, F, top, E, act_fn);
    else if (dtype == CPMCU_BF16)
        moe_up_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)h, ldh, (const bf16_t*)wu, idx, (bf16_t*)act, H, F, top, E, act_fn);
    else
        CPMCU_FAIL("moe_up: unknown dtype %d", dtype);
    CPMCU_LAUNCH_CHECK("moe_up");
    return nullptr;
}

// grid (tokens, ceil(H / 16)), 256 threads: a wavefront owns 4 columns and reads their 4 weight rows of a chosen expert
// together, against one piece of the pair's act row.  shared: the every-token expert's output [n, H] (or float partial
// sums [parts][n][H]), multiplied by sg[t]; may be absent.  h: the experts' input, what identity experts (e >= E) add.
// What the end adds (shared, residual, the layer's other result) is asked for first: 16 lanes a column bring it, a part a
// lane.
template <typename T, typename ST>
__global__ __launch_bounds__(256) void moe_down_kernel(const T* __restrict__ act, const T* __restrict__ wd,
                                                       const int* __restrict__ idx, const float* __restrict__ w,
                                                       const ST* __restrict__ shared, int shared_parts,
                                                       long shared_stride, const float* __restrict__ sg,
                                                       const T* __restrict__ h, long ldh, int E,
                                                       float* __restrict__ out, int H, int F, int top, Join join) {
    // Workgroups are dealt to the 8 XCDs in turn: an XCD's take all tokens of a block of columns one behind the other, and tokens that
    // share an expert find its rows in that L2 (the experts above: 16 tokens 152 -> 132 us, 12 117 -> 107, 8 83 -> 80).
    long t = blockIdx.x;
    int block = blockIdx.y;
    const int n = gridDim.x, whole = gridDim.y / 8 * 8;
    if (block < whole) {
        const long lin = (long)block * n + t, i = lin / 8;
        t = i % n;
        block = (int)(i / n) * 8 + (int)(lin % 8);
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool vec = (F % 8 == 0) && ((uintptr_t)act % 32 == 0) && ((uintptr_t)wd % 32 == 0);
    const int c0 = block * 4 * MOE_ROWS + wave * MOE_ROWS;
    if (c0 >= H) return;
    const int mine = c0 + (lane >> 4), p0 = lane & 15;               // this lane's column at the end, and its part
    const long at = t * H + min(mine, H - 1);
    float extra = 0.f;
    if (shared) {
        for (int p = p0; p < shared_parts; p += 16) extra += to_f32(shared[(long)p * shared_stride + at]);
        if (sg) extra *= sg[t];
    }
    if (join.x) {
        for (int p = p0; p < join.a_parts; p += 16) extra += join_part(join, p, at);
        if (p0 == 15) extra += join.x[at] + (join.a_bias ? join.a_bias[min(mine, H - 1)] : 0.f);
    }
    const long row0 = (long)min(c0, H - 1) * F, row1 = (long)min(c0 + 1, H - 1) * F, row2 = (long)min(c0 + 2, H - 1) * F,
               row3 = (long)min(c0 + 3, H - 1) * F;
    float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f, same = 0.f;
    for (int k = 0; k < top; ++k) {
        const int e = idx[t * top + k];
        const float wk = w[t * top + k];
        if (e >= E) {
            same += wk;
            continue;
        }
        const T* ap = act + (t * top + k) * F;
        const T* wp = wd + (long)e * H * F;
        float d0 = 0.f, d1 = 0.f, d2 = 0.f, d3 = 0.f;
        if (vec) {
            for (int c = lane * 8; c < F; c += 64 * 8) {
                float x[8], y0[8], y1[8], y2[8], y3[8];
                load8<T>(wp + row0 + c, y0);
                load8<T>(wp + row1 + c, y1);
                load8<T>(wp + row2 + c, y2);
                load8<T>(wp + row3 + c, y3);
                load8<T>(ap + c, x);
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    d0 += x[i] * y0[i];
                    d1 += x[i] * y1[i];
                    d2 += x[i] * y2[i];
                    d3 += x[i] * y3[i];
                }
            }
        } else {
            for (int c = lane; c < F; c += 64) {
                const float x = to_f32(ap[c]);
                d0 += x * to_f32(wp[row0 + c]);
                d1 += x * to_f32(wp[row1 + c]);
                d2 += x * to_f32(wp[row2 + c]);
                d3 += x * to_f32(wp[row3 + c]);
            }
        }
        s0 += wk * d0;
        s1 += wk * d1;
        s2 += wk * d2;
        s3 += wk * d3;
    }
    s0 = wave_sum(s0);
    s1 = wave_sum(s1);
    s2 = wave_sum(s2);
    s3 = wave_sum(s3);
    extra = row16_sum(extra);                       // the 16 lanes of a column are one row of lanes
    const int r = lane >> 4;
    float v = (r == 0 ? s0 : (r == 1 ? s1 : (r == 2 ? s2 : s3))) + extra;
    if (p0 == 0 && mine < H) {
        if (h && same != 0.f) v += same * to_f32(h[t * ldh + mine]);
        if (join.x) {
            join.x[at] = v;
            if (join.copy) ((T*)join.copy)[at] = from_f32<T>(v);
        } else {
            out[at] = v;
        }
    }
}

static const char* join_check(const Join& j, const float* out) {
    CPMCU_REQUIRE(j.x || out, "experts: nowhere to write");
    CPMCU_REQUIRE(!j.x || (j.a_parts >= 0 && j.a_parts <= 32 && (j.a != nullptr) == (j.a_parts > 0)),
                  "experts: %d parts of the layer's other result (up to 32 are taken)", j.a_parts);
    return nullptr;
}

extern "C" const char* cpmcu_moe_down(const void* act, int dtype, const void* wd, const int* idx, const float* w,
                                      const void* shared, int shared_dtype, int shared_parts, long shared_stride,
                                      const float* sg, const void* h, long ldh, int E, float* out, int n, int H, int F,
                                      int top, float* x, const void* a, int a_dtype, int a_parts, long a_stride,
                                      const float* a_bias, void* copy, hipStream_t stream) {
    const Join join{x, a, a_dtype == CPMCU_BF16, a ? a_parts : 0, a_stride, a_bias, copy};
    if (const char* m = join_check(join, out)) return m;
    CPMCU_REQUIRE(n > 0 && H > 0 && F > 0 && top > 0 && E > 0, "moe_down: empty shape");
    const int hy = (H + 4 * MOE_ROWS - 1) / (4 * MOE_ROWS);
    CPMCU_REQUIRE(hy <= 65535, "moe_down: a width of %d exceeds the launch grid", H);
    dim3 grid(n, hy);
#define LAUNCH(Tv, STv)                                                                                            \
    moe_down_kernel<Tv, STv><<<grid, 256, 0, stream>>>((const Tv*)act, (const Tv*)wd, idx, w, (const STv*)shared,   \
                                                       shared_parts, shared_stride, sg, (const Tv*)h, ldh, E, out, H, F, top, join)
    const int sd = shared ? shared_dtype : CPMCU_F32;
    if (dtype == CPMCU_F32 && sd == CPMCU_F32) LAUNCH(float, float);
    else if (dtype == CPMCU_BF16 && sd == CPMCU_F32) LAUNCH(bf16_t, float);
    else if (dtype == CPMCU_BF16 && sd == CPMCU_BF16) LAUNCH(bf16_t, bf16_t);
    else CPMCU_FAIL("moe_down: unsupported dtypes act=%d shared=%d", dtype, sd);
#undef LAUNCH
    CPMCU_LAUNCH_CHECK("moe_down");
    return nullptr;
}

// ===========================================================================
// The same experts for steps of many tokens, bf16 on the matrix cores (v_mfma_f32_16x16x32_bf16): the (token,
// chosen expert) pairs are grouped by expert into tiles of up to MOE_TILE or MOE_WIDE rows, and every tile is a
// product with its expert's weights.
//
//  * moe_group_kernel (one workgroup): counts the pairs of every expert and lists them expert by expert: rows[offs[e] ..
//    offs[e + 1]) are expert e's pairs, tile_expert[tile] = e + 1024 * (the tile's number among its expert's), n_tiles the
//    number of tiles.  Which row of its expert's tiles a pair gets depends on timing; its result does not (a row's sums
//    are its own).
//  * moe_tile_kernel, moe_wide_kernel, moe_product_kernel (moe_product.hip): GATED act[pair] = act(Wg_e h_t) * (Wu_e h_t), PLAIN act[pair] = act(Wu_e h_t), DOWN y[pair] =
//    Wd_e act[pair] (bf16).
//  * moe_combine_kernel: out[t] = sum_k w[t, k] y[t, k] (h_t where the chosen expert is an identity expert) (+ sg[t] * shared[t]) in float, k in order.
// ===========================================================================
typedef __bf16 mbf16x8_t __attribute__((ext_vector_type(8)));
typedef float mfloatx4_t __attribute__((ext_vector_type(4)));
typedef unsigned mu32x4_t __attribute__((ext_vector_type(4)));

#define MOE_TILE 64                            // rows of a tile of moe_tile_kernel at most
#define MOE_WIDE 128                           // of moe_wide_kernel

// tile_rows: rows a tile at most; an expert's pairs are spread evenly over as few tiles as hold them (moe_tile_kernel).
// counters: MOE_PRODUCT_COUNTERS of moe_product_kernel, set to 0.  large: the tiles are moe_product_kernel's, listed run by run of the 8 that
// an XCD takes each, experts of many rows first and dealt to the runs in turn: what is left at the end is small
__global__ __launch_bounds__(1024) void moe_group_kernel(const int* __restrict__ idx, int n_pairs, int E, int tile_rows,
                                                         int* __restrict__ rows, int* __restrict__ offs,
                                                         int* __restrict__ tile_expert, int* __restrict__ n_tiles,
                                                         int* __restrict__ counters, int large) {
    __shared__ int counts[MOE_MAX_EXPERTS], order[MOE_MAX_EXPERTS];
    __shared__ int pair_sum[16], tile_sum[16];
    const int e = threadIdx.x, lane = e & 63, wave = e >> 6;
    counts[e] = 0;
    if (e < MOE_PRODUCT_COUNTERS) counters[e] = 0;
    __syncthreads();
    for (int p = threadIdx.x; p < n_pairs; p += 1024)
        if (idx[p] < E) atomicAdd(&counts[idx[p]], 1);              // identity experts have no tiles
    __syncthreads();
    // running sums of pairs and tiles over the experts, one expert a thread
    const int c = counts[e];
    int mine = e;                                                       // the expert whose tiles this thread lists
    if (large) {
        if (e < E) {
            int rank = 0;                                               // experts with more rows, or as many and a lower number
            for (int i = 0; i < E; ++i) rank += counts[i] > c || (counts[i] == c && i < e);
            const int run = rank & 7, each = E / 8, more = E % 8;       // runs 0 .. more - 1 have one expert more
            order[run * each + min(run, more) + (rank >> 3)] = e;
        }
        __syncthreads();
        if (e < E) mine = order[e];
    }
    const int nt = (counts[mine] + tile_rows - 1) / tile_rows;
    int pairs = c, tiles = nt;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int a = __shfl_up(pairs, d, 64), b = __shfl_up(tiles, d, 64);
        if (lane >= d) {
            pairs += a;
            tiles += b;
        }
    }
    if (lane == 63) {
        pair_sum[wave] = pairs;
        tile_sum[wave] = tiles;
    }
    __syncthreads();
    for (int w = 0; w < wave; ++w) {
        pairs += pair_sum[w];
        tiles += tile_sum[w];
    }
    if (e < E) {
        offs[e] = pairs - c;
        if (e == E - 1) {
            offs[E] = pairs;
            *n_tiles = tiles;
        }
        for (int i = 0; i < nt; ++i) tile_expert[tiles - nt + i] = mine + 1024 * i;
    }
    counts[e] = pairs - c;
    __syncthreads();
    for (int p = threadIdx.x; p < n_pairs; p += 1024) {
        const int x = idx[p];
        if (x < E) rows[atomicAdd(&counts[x], 1)] = p;
    }
}

// Workgroups of 4 wavefronts; a tile of up to 64 rows against 128 weight rows (GATED: 64 features, gate and up row of
// each), a wavefront all rows and 32 weight rows (GATED: 16 features).  Pieces of 64 columns of both go through LDS in
// two buffers, the next piece on its way to registers meanwhile (with both operands straight from memory every wavefront
// fetched all of the rows for itself, 16 bytes of a row an access, and the address unit, not HBM or the matrix cores,
// was the bound).  A piece's row is 8 chunks of 16 bytes, chunk c of row r at place c ^ (r % 8): 8 neighbouring lanes
// then read all banks.  The tile's rows beyond the last 16 (beyond 32: 32) in use are neither loaded nor multiplied.
// K is the rows' width, N the number of features; in: h rows by token (GATED, PLAIN: pair / top) or act rows by pair.
// Measured (64 experts, width 4,096, 6 a token; us): 24 tokens, gated experts of 1,408 182 + 93 (their 58 experts' matrices
// at 6 to 7 TB/s); most weights are read once and streamed past the caches.  Two pieces on their way at once: one took 234 +
// 122.  Results leave through LDS as whole lines.
// The grid is dealt to the 8 XCDs in turn; each takes one run of the tasks, ordered expert by expert and within an expert
// weight rows by weight rows, so that the tiles that share weights meet in one L2.
template <int KIND>
__global__ __launch_bounds__(256, 2) void moe_tile_kernel(const bf16_t* __restrict__ in, long ldi,
                                                          const bf16_t* __restrict__ w, const int* __restrict__ rows,
                                                          const int* __restrict__ offs, const int* __restrict__ tile_expert,
                                                          const int* __restrict__ n_tiles, bf16_t* __restrict__ out, int K, int N, int top, int tile_rows,
                                                          int act_fn, float act_limit) {
    constexpr int BM = MOE_TILE, FEATURES = KIND == MOE_GATED ? 64 : 128;
    __shared__ mu32x4_t lds[2][(BM + 128) * 8];
    const int nts = (N + FEATURES - 1) / FEATURES;
    const int tasks = *n_tiles * nts, per = (tasks + 7) / 8;
    const int task = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || task >= tasks) return;
    const int q = task / nts, te = tile_expert[q], e = te & 1023;
    const int start = offs[e], cnt = offs[e + 1] - start;
    const int m = (cnt + tile_rows - 1) / tile_rows, rpt = ((cnt + m - 1) / m + 15) & ~15;
    const int local = task - (q - (te >> 10)) * nts, mt = local % m, f0 = local / m * FEATURES;
    const int row0 = start + mt * rpt, n_rows = min(rpt, cnt - mt * rpt);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int chunk = threadIdx.x & 7, lrow = threadIdx.x >> 3;       // what this thread brings: chunk of rows lrow + 32 i
    const bf16_t* wp[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        // weight row 32 w + 16 j + x of the tile: GATED feature f0 + 16 w + x, gate (j = 0) or up (j = 1)
        const int row = lrow + 32 * i;
        const int f = min(f0 + (KIND == MOE_GATED ? (row >> 5) * 16 + (row & 15) : row), N - 1);
        wp[i] = w + ((long)e * (KIND == MOE_GATED ? 2 : 1) * N + (KIND == MOE_GATED && (row & 16) ? N : 0) + f) * K + chunk * 8;
    }
    const int place = lrow * 8 + (chunk ^ (lrow & 7));                // rows 32 apart have the same place in their 256

    const bool whole = (uintptr_t)out % 16 == 0;                      // (pair outputs may start anywhere)
    auto product = [&](auto groups) {
        constexpr int NRT = decltype(groups)::value, AP = (NRT + 1) / 2;
        const bf16_t* ap[AP];
#pragma unroll
        for (int i = 0; i < AP; ++i) {
            const int pair = rows[row0 + min(lrow + 32 * i, n_rows - 1)];
            ap[i] = in + (long)(KIND == MOE_DOWN ? pair : pair / top) * ldi + chunk * 8;
        }
        struct Piece { mu32x4_t a[AP], w[4]; } p0, p1;                // on their way: this piece and the next
        auto fetch = [&](Piece& p, int k0) {
            const int k = min(k0, K - 8 - chunk * 8);                 // beyond the row's end: its last columns, zeroed below
#pragma unroll
            for (int i = 0; i < 4; ++i) p.w[i] = __builtin_nontemporal_load((const mu32x4_t*)(wp[i] + k));
#pragma unroll
            for (int i = 0; i < AP; ++i) p.a[i] = *(const mu32x4_t*)(ap[i] + k);
        };
        mfloatx4_t acc[NRT][2];
#pragma unroll
        for (int rt = 0; rt < NRT; ++rt) acc[rt][0] = acc[rt][1] = mfloatx4_t{0.f, 0.f, 0.f, 0.f};
        auto step = [&](Piece& p, int k0, int buf, auto last) {
            // (only behind the loop: a branch here would make every step wait for all loads in flight)
            if (decltype(last)::value && k0 + chunk * 8 >= K) {       // K % 8 == 0: the whole chunk lies beyond the end
                const mu32x4_t zero = {0u, 0u, 0u, 0u};
#pragma unroll
                for (int i = 0; i < 4; ++i) p.w[i] = zero;
#pragma unroll
                for (int i = 0; i < AP; ++i) p.a[i] = zero;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) lds[buf][BM * 8 + 256 * i + place] = p.w[i];
#pragma unroll
            for (int i = 0; i < AP; ++i)
                if (NRT % 2 == 0 || i + 1 < AP || lrow < 16) lds[buf][256 * i + place] = p.a[i];
            if (!decltype(last)::value) fetch(p, k0 + 128);
            __syncthreads();
            mbf16x8_t a[2][NRT], b[2][2];
            auto read = [&](int kk) {
                const int at = (kk * 4 + g) ^ (r & 7);
#pragma unroll
                for (int j = 0; j < 2; ++j) b[kk][j] = *(const mbf16x8_t*)&lds[buf][(BM + wave * 32 + j * 16 + r) * 8 + at];
#pragma unroll
                for (int rt = 0; rt < NRT; ++rt) a[kk][rt] = *(const mbf16x8_t*)&lds[buf][(rt * 16 + r) * 8 + at];
            };
            read(0);
            read(1);
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[rt][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[kk][rt], b[kk][j], acc[rt][j], 0, 0, 0);
        };
        fetch(p0, 0);
        fetch(p1, 64);
        int k0 = 0;
        for (; k0 + 128 <= K; k0 += 128) {
            step(p0, k0, 0, std::false_type());
            step(p1, k0 + 64, 1, std::false_type());
        }
        if (k0 < K) step(p0, k0, 0, std::true_type());
        if (k0 + 64 < K) step(p1, k0 + 64, 1, std::true_type());
        // lane (weight row r, g): acc[rt][j][i] belongs to the tile's row rt * 16 + 4 g + i.  The results pass through LDS, so
        // that 8 or 16 neighbouring lanes write a row's 16-byte chunks
        constexpr int LINE = FEATURES + 8;
        bf16_t* stage = (bf16_t*)lds;
        __syncthreads();
#pragma unroll
        for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                bf16_t* to = stage + (rt * 16 + 4 * g + i) * LINE + wave * (FEATURES / 4) + r;
                if (KIND == MOE_GATED) {
                    float gt = acc[rt][0][i], up = acc[rt][1][i];
                    gate_prepare(gt, up, act_fn, act_limit);
                    *to = f32_to_bf16(gate_act(gt, act_fn) * up);
                } else {
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        to[j * 16] = f32_to_bf16(KIND == MOE_PLAIN ? plain_act(acc[rt][j][i], act_fn) : acc[rt][j][i]);
                }
            }
        __syncthreads();
        constexpr int CHUNKS = FEATURES / 8;
        const int c = threadIdx.x % CHUNKS * 8;
        if (f0 + c < N)                                               // (N % 8 == 0: the whole chunk)
            for (int row = threadIdx.x / CHUNKS; row < n_rows; row += 256 / CHUNKS) {
                bf16_t* to = out + (long)rows[row0 + row] * N + f0 + c;
                const bf16_t* from = stage + row * LINE + c;
                if (whole) {
                    *(mu32x4_t*)to = *(const mu32x4_t*)from;
                } else {
#pragma unroll
                    for (int j = 0; j < 8; ++j) to[j] = from[j];
                }
            }
    };
    if (n_rows > 32) product(std::integral_constant<int, 4>());
    else if (n_rows > 16) product(std::integral_constant<int, 2>());
    else product(std::integral_constant<int, 1>());
}

// The same products for steps that give an expert many rows (cpmcu_moe_experts_mfma has the rule; the largest of them go to
// moe_product_kernel): tiles of up to 128 rows
// against 128 weight rows (GATED: 64 features), workgroups of 4 wavefronts, two a CU, a wavefront half of the rows and 64 weight rows.  Pieces of 64 columns go
// from memory to LDS without passing registers, the weights in three buffers and the rows in two (80 KB), with the swizzle of
// the kernel above in the column that each lane asks for.  The workgroup meets once a piece, in the middle of its products:
// what the second half multiplies has been read by then, and while it does, the next piece's first operands are read and the
// pieces behind it are on their way.  (Through registers, with the meeting before the products, LDS reads and matrix
// instructions took turns.)  An expert whose rows fill one tile streams its weights past the caches; where tiles share
// them they stay (all past the caches: 476 instead of 407 us; none: the passes of 347 tokens 282 instead of 254).
// What bounds it: weights alone take 290 us of about 400 at 2,048 tokens and even routing (5.1 TB/s), products alone 250,
// rows alone 130; a CU is busy 75 to 80% of the time, since experts' tiles are uneven.
// Kernel times, us, up + down, the kernel through registers (tiles of 128, under 48 pairs an expert of 64) -> this:
//   64 experts of 1,408 gated at width 4,096, routers with random weights (from none to 2,000 of 2,048 tokens an expert):
//     2,048 tokens 465 + 270 -> 424 + 246, 16 of 80 identity 427 + 246 -> 407 + 230, 347 tokens 275 + 157 -> 254 + 145
//   even routing: 2,048 477 + 269 -> 443 + 252, 768 317 + 177 -> 306 + 167, 512 298 + 167 -> 269 + 156, 280 256 + 146 -> 241 +
//     132 (on another day and with more shapes level: see the rule); of 2,112 without a gate, 2,048 372 + 372 -> 350 + 344, 512 246 +
//     240 -> 229 + 226
//   64 of 1,024 gated at 1,024, 2,048 tokens with 4 each 89 + 52 -> 75 + 45; 16 of 768 at 2,048 85 + 51 -> 75 + 47
// Taken back: workgroups of 8 wavefronts, one a CU, with tiles of 256 weight rows and 128, 192 or 256 rows (LDS reads a
// fifth fewer, weights asked for once: as fast with even routing, 0 to 5% slower with a router's); every XCD a share of all
// experts' features, for balance (rows no longer meet in an L2: 5% slower).
template <int KIND>
__global__ __launch_bounds__(256, 2) void moe_wide_kernel(const bf16_t* __restrict__ in, long ldi,
                                                          const bf16_t* __restrict__ w, const int* __restrict__ rows,
                                                          const int* __restrict__ offs, const int* __restrict__ tile_expert,
                                                          const int* __restrict__ n_tiles, bf16_t* __restrict__ out, int K, int N, int top, int tile_rows,
                                                          int act_fn, float act_limit) {
    constexpr int BM = MOE_WIDE, FEATURES = KIND == MOE_GATED ? 64 : 128;
    constexpr int WSTAGE = 128 * 8;                                   // 16-byte chunks of a piece's weights; three pieces
    __shared__ mu32x4_t lds[3 * WSTAGE + 2 * BM * 8];
    const int nts = (N + FEATURES - 1) / FEATURES;
    const int tasks = *n_tiles * nts, per = (tasks + 7) / 8;
    const int task = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || task >= tasks) return;
    const int q = task / nts, te = tile_expert[q], e = te & 1023;
    const int start = offs[e], cnt = offs[e + 1] - start;
    const int m = (cnt + tile_rows - 1) / tile_rows, rpt = ((cnt + m - 1) / m + 31) & ~31;
    const int local = task - (q - (te >> 10)) * nts, mt = local % m, f0 = local / m * FEATURES;
    const int row0 = start + mt * rpt, n_rows = min(rpt, cnt - mt * rpt);     // (never empty: rpt <= tile_rows)
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int chunk = ((lane & 7) ^ (lane >> 3)) * 8;                 // a lane brings place lane % 8 of row lane / 8 of 8 rows
    const unsigned base = lds_byte(lds);
    const int half = wave & 1, side = wave >> 1;
    const bool whole = (uintptr_t)out % 16 == 0;
    const bf16_t* wp[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = wave * 32 + i * 8 + (lane >> 3);              // weight row 32 w + 16 j + x, as above
        const int f = min(f0 + (KIND == MOE_GATED ? (row >> 5) * 16 + (row & 15) : row), N - 1);
        wp[i] = w + ((long)e * (KIND == MOE_GATED ? 2 : 1) * N + (KIND == MOE_GATED && (row & 16) ? N : 0) + f) * K;
    }
    auto product = [&](auto groups) {
        constexpr int NRT = decltype(groups)::value, HRT = NRT / 2;
        constexpr int AP = NRT / 2;                                   // groups of 8 rows a wavefront brings
        constexpr int RSTAGE = 16 * NRT * 8, ROWS = 3 * WSTAGE;
        const bf16_t* ap[AP];
#pragma unroll
        for (int i = 0; i < AP; ++i) {
            const int pair = rows[row0 + min((i * 4 + wave) * 8 + (lane >> 3), n_rows - 1)];
            ap[i] = in + (long)(KIND == MOE_DOWN ? pair : pair / top) * ldi;
        }
        auto fetch_w = [&](int p, int stage) {
            const int k = min(p * 64 + chunk, K - 8);
            const unsigned to = base + (stage * WSTAGE + wave * 256) * 16;
            if (m == 1) {
#pragma unroll
                for (int i = 0; i < 4; ++i) stream16(wp[i] + k, to + i * 1024);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) bring16(wp[i] + k, to + i * 1024);
            }
        };
        auto fetch_r = [&](int p) {
            const int k = min(p * 64 + chunk, K - 8);
            const unsigned to = base + (ROWS + (p & 1) * RSTAGE) * 16;
#pragma unroll
            for (int i = 0; i < AP; ++i) bring16(ap[i] + k, to + (i * 4 + wave) * 1024);
        };
        mfloatx4_t acc[HRT][4];
#pragma unroll
        for (int rt = 0; rt < HRT; ++rt)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[rt][j] = mfloatx4_t{0.f, 0.f, 0.f, 0.f};
        const int pieces = (K + 63) / 64;
        mbf16x8_t a[2][HRT], b[2][4];
        auto read = [&](int p, int stage, int kk) {
            const int at = (kk * 4 + g) ^ (r & 7);
            const mu32x4_t* ws = lds + stage * WSTAGE + side * 512;
            const mu32x4_t* rs = lds + ROWS + (p & 1) * RSTAGE + half * (HRT * 128);
#pragma unroll
            for (int j = 0; j < 4; ++j) b[kk][j] = *(const mbf16x8_t*)&ws[(j * 16 + r) * 8 + at];
#pragma unroll
            for (int rt = 0; rt < HRT; ++rt) a[kk][rt] = *(const mbf16x8_t*)&rs[(rt * 16 + r) * 8 + at];
        };
        auto multiply = [&](int kk) {
#pragma unroll
            for (int rt = 0; rt < HRT; ++rt)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[rt][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[kk][rt], b[kk][j], acc[rt][j], 0, 0, 0);
        };
        // columns beyond the row's end (K % 8 == 0: whole chunks) are nothing; asked for were the row's last ones
        auto blank = [&](int p, int stage) {
            if (p + 1 < pieces || K % 64 == 0) return;
            for (int i = threadIdx.x; i < WSTAGE + RSTAGE; i += 256) {
                mu32x4_t* to = i < WSTAGE ? lds + stage * WSTAGE + i : lds + ROWS + (p & 1) * RSTAGE + i - WSTAGE;
                if (((i & 7) ^ (i >> 3 & 7)) >= K % 64 / 8) *to = mu32x4_t{0u, 0u, 0u, 0u};
            }
            __syncthreads();
        };
        fetch_w(0, 0);
        fetch_r(0);
        if (pieces > 1) {
            fetch_w(1, 1);
            fetch_r(1);
        }
        if (pieces > 2) {
            fetch_w(2, 2);
            landed<8 + AP>();                                         // behind the first piece: w, rows, w
        } else {
            landed<0>();
        }
        blank(0, 0);
        read(0, 0, 0);
        int p = 0, stage = 0;
        for (; p + 2 < pieces; ++p) {
            read(p, stage, 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(0);
            landed<4>();                                              // behind piece p + 1: the weights of p + 2; p is free
            fetch_r(p + 2);
            if (p + 3 < pieces) fetch_w(p + 3, stage);
            stage = stage == 2 ? 0 : stage + 1;
            read(p + 1, stage, 0);
            __builtin_amdgcn_sched_barrier(0);
            multiply(1);
        }
        for (; p < pieces; ++p) {
            read(p, stage, 1);
            multiply(0);
            if (p + 1 < pieces) {
                landed<0>();
                stage = stage == 2 ? 0 : stage + 1;
                blank(p + 1, stage);
                read(p + 1, stage, 0);
            }
            multiply(1);
        }
        constexpr int LINE = FEATURES + 8;
        bf16_t* out_stage = (bf16_t*)lds;
        __syncthreads();
#pragma unroll
        for (int rt = 0; rt < HRT; ++rt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                bf16_t* to = out_stage + ((half * HRT + rt) * 16 + 4 * g + i) * LINE + side * (FEATURES / 2) + r;
                if (KIND == MOE_GATED) {
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        float gt = acc[rt][2 * j][i], up = acc[rt][2 * j + 1][i];
                        gate_prepare(gt, up, act_fn, act_limit);
                        to[j * 16] = f32_to_bf16(gate_act(gt, act_fn) * up);
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        to[j * 16] = f32_to_bf16(KIND == MOE_PLAIN ? plain_act(acc[rt][j][i], act_fn) : acc[rt][j][i]);
                }
            }
        __syncthreads();
        constexpr int CHUNKS = FEATURES / 8;
        const int c = threadIdx.x % CHUNKS * 8;
        if (f0 + c < N)
            for (int row = threadIdx.x / CHUNKS; row < n_rows; row += 256 / CHUNKS) {
                bf16_t* to = out + (long)rows[row0 + row] * N + f0 + c;
                const bf16_t* from = out_stage + row * LINE + c;
                if (whole) {
                    *(mu32x4_t*)to = *(const mu32x4_t*)from;
                } else {
#pragma unroll
                    for (int j = 0; j < 8; ++j) to[j] = from[j];
                }
            }
    };
    if (n_rows > 96) product(std::integral_constant<int, 8>());
    else if (n_rows > 64) product(std::integral_constant<int, 6>());
    else if (n_rows > 32) product(std::integral_constant<int, 4>());
    else product(std::integral_constant<int, 2>());
}

// V neighbouring columns a thread (4: 8-byte loads of a pair's row)
template <typename ST, int V>
__global__ __launch_bounds__(256) void moe_combine_kernel(const bf16_t* __restrict__ y, const float* __restrict__ w,
                                                          const ST* __restrict__ shared, int shared_parts,
                                                          long shared_stride, const float* __restrict__ sg,
                                                          const int* __restrict__ idx, const bf16_t* __restrict__ h, long ldh,
                                                          int E, float* __restrict__ out, long total, int H, int top, Join join) {
    auto load = [](const bf16_t* p, float* v) {
        if (V == 4) {
            const uint2 u = *(const uint2*)p;
            v[0] = __uint_as_float(u.x << 16); v[1 % V] = __uint_as_float(u.x & 0xffff0000u);
            v[2 % V] = __uint_as_float(u.y << 16); v[3 % V] = __uint_as_float(u.y & 0xffff0000u);
        } else {
            v[0] = to_f32(*p);
        }
    };
    for (long i = V * ((long)blockIdx.x * 256 + threadIdx.x); i < total; i += V * (long)gridDim.x * 256) {
        const long t = i / H;
        const int c = (int)(i - t * H);
        float s[V];
#pragma unroll
        for (int e = 0; e < V; ++e) s[e] = 0.f;
#pragma unroll 2
        for (int k = 0; k < top; ++k) {
            float v[V];
            load(idx[t * top + k] < E ? y + (t * top + k) * H + c : h + t * ldh + c, v);
#pragma unroll
            for (int e = 0; e < V; ++e) s[e] += w[t * top + k] * v[e];
        }
#pragma unroll
        for (int e = 0; e < V; ++e) {
            if (shared) {
                float v = 0.f;
                for (int p = 0; p < shared_parts; ++p) v += to_f32(shared[(long)p * shared_stride + i + e]);
                s[e] += (sg ? sg[t] : 1.0f) * v;
            }
            if (join.x) {
                s[e] += join.x[i + e] + (join.a_bias ? join.a_bias[c + e] : 0.f);
                for (int p = 0; p < join.a_parts; ++p) s[e] += join_part(join, p, i + e);
            }
        }
        float* dst = join.x ? join.x : out;
        if (V == 4) *(float4*)(dst + i) = make_float4(s[0], s[1 % V], s[2 % V], s[3 % V]);
        else dst[i] = s[0];
        if (join.copy) {
#pragma unroll
            for (int e = 0; e < V; ++e) ((bf16_t*)join.copy)[i + e] = f32_to_bf16(s[e]);
        }
    }
}

// The same sums for up to 8 experts a token, a workgroup 2,048 columns of a token, 8 neighbouring ones a thread: the token's
// experts and weights are scalars, and all TOP rows are asked for before the first is added (the kernel above has two in flight).
// 2,048 tokens, 6 experts, width 4,096: 39.3 -> 22.5 us (100 MB of rows in, 34 out: 6 TB/s); in a pass that joins the shared
// experts' result and the residual, read and written, on its way 47 to 50.
template <typename ST, int TOP>
__global__ __launch_bounds__(256) void moe_combine_token_kernel(const bf16_t* __restrict__ y, const float* __restrict__ w,
                                                                const ST* __restrict__ shared, int shared_parts,
                                                                long shared_stride, const float* __restrict__ sg,
                                                                const int* __restrict__ idx, const bf16_t* __restrict__ h, long ldh,
                                                                int E, float* __restrict__ out, int H, int pieces, Join join) {
    const long t = blockIdx.x / pieces;
    const int c = (int)(blockIdx.x % pieces) * 2048 + threadIdx.x * 8;
    if (c >= H) return;
    const long at = t * H + c;
    mu32x4_t v[TOP];
#pragma unroll
    for (int k = 0; k < TOP; ++k)
        v[k] = *(const mu32x4_t*)(idx[t * TOP + k] < E ? y + (t * TOP + k) * H + c : h + t * ldh + c);
    float s[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) s[e] = 0.f;
#pragma unroll
    for (int k = 0; k < TOP; ++k) {
        const float wk = w[t * TOP + k];
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] += wk * __uint_as_float(e & 1 ? v[k][e / 2] & 0xffff0000u : v[k][e / 2] << 16);
    }
    if (shared) {
        const float g = sg ? sg[t] : 1.0f;
        float a[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) a[e] = 0.f;
        for (int p = 0; p < shared_parts; ++p)
#pragma unroll
            for (int e = 0; e < 8; ++e) a[e] += to_f32(shared[(long)p * shared_stride + at + e]);
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] += g * a[e];
    }
    if (join.x) {
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] += join.x[at + e] + (join.a_bias ? join.a_bias[c + e] : 0.f);
        for (int p = 0; p < join.a_parts; ++p)
#pragma unroll
            for (int e = 0; e < 8; ++e) s[e] += join_part(join, p, at + e);
    }
    float* dst = (join.x ? join.x : out) + at;
    *(float4*)dst = make_float4(s[0], s[1], s[2], s[3]);
    *(float4*)(dst + 4) = make_float4(s[4], s[5], s[6], s[7]);
    if (join.copy) {
        bf16_t* copy = (bf16_t*)join.copy + at;
#pragma unroll
        for (int e = 0; e < 8; ++e) copy[e] = f32_to_bf16(s[e]);
    }
}

// scratch: rows int [max_tiles * 64] (the pairs by expert; at its end moe_product_kernel's counters and the experts' offsets), tile_expert int
// [max_tiles], n_tiles int [1], y bf16 [n * top, H];
// max_tiles = ceil(n * top / 64) + E
extern "C" const char* cpmcu_moe_experts_mfma(const void* h, long ldh, const void* wgu, const void* wd, const int* idx,
                                              const float* w, const void* shared, int shared_dtype, int shared_parts,
                                              long shared_stride, const float* sg, void* act, void* y, int* rows,
                                              int* tile_expert, int* n_tiles, int max_tiles, float* out, int n, int H,
                                              int F, int E, int top, int gated, int act_fn, float act_limit, float* x, const void* a,
                                              int a_dtype, int a_parts, long a_stride, const float* a_bias, void* copy,
                                              hipStream_t stream) {
    const Join join{x, a, a_dtype == CPMCU_BF16, a ? a_parts : 0, a_stride, a_bias, copy};
    if (const char* m = join_check(join, out)) return m;
    CPMCU_REQUIRE(n > 0 && H > 0 && F > 0 && E > 0 && top > 0, "moe_experts_mfma: empty shape");
    CPMCU_REQUIRE(gated ? CPMCU_ACT_KNOWN(act_fn) : CPMCU_PLAIN_ACT_KNOWN(act_fn), "moe_experts_mfma: unknown nonlinearity %d", act_fn);
    CPMCU_REQUIRE(E <= MOE_MAX_EXPERTS, "moe_experts_mfma: %d experts (up to %d are taken)", E, MOE_MAX_EXPERTS);
    CPMCU_REQUIRE(H % 8 == 0 && F % 8 == 0 && ldh % 8 == 0 && (uintptr_t)h % 16 == 0 && (uintptr_t)wgu % 16 == 0 &&
                  (uintptr_t)wd % 16 == 0 && (uintptr_t)act % 16 == 0,
                  "moe_experts_mfma: widths must be multiples of 8 and operands start on 16-byte borders (H=%d, F=%d)", H, F);
    const long pairs = (long)n * top;
    CPMCU_REQUIRE(max_tiles >= (pairs + MOE_TILE - 1) / MOE_TILE + E && max_tiles <= 65535,
                  "moe_experts_mfma: %d tiles of scratch for %ld pairs of %d experts (at most 65535)", max_tiles, pairs, E);
    // moe_wide_kernel from 48 pairs an expert on, and from 24 where the first product has four workgroups a CU (experts x blocks of 128 weight
    // rows).  Up + down in us, moe_tile_kernel / moe_wide_kernel; experts of width x size, gated unless said otherwise:
    //   from 48 on, against the tiles of 128 rows through registers that it replaced: 7% faster in the mean of 308 shapes (4 to 64
    //     experts, 512 x 256 to 4,096 x 2,112); the worst 32 of 2,048 x 1,408 at 100 pairs 131/142 (rows in steps of 32 instead of 16)
    //   24 to 47 pairs, four workgroups a CU or more: 64 of 4,096 x 1,408 even routing 28 pairs 375/371, 36 389/390; 64 of
    //     4,096 x 2,112 uneven 28 553/495; the same without a gate 28 390/341, 36 442/377, even 24 381/391
    //   fewer: one round of 512 workgroups where moe_tile_kernel has one of 768, and tiles of up to 128 rows behind which the CUs
    //     are idle.  32 of 4,096 x 1,408 28 pairs 201/228; 32 of 1,024 x 512 44 pairs 35/41, without a gate 30/35, 8 of them 26/32;
    //     32 of 512 x 256 without a gate 24 to 44 pairs 19/25
    // Without a gate the first product of up to 64 tokens alone takes it, on the tiles of the other, where every CU has one workgroup
    // at most and pieces enough to be ahead (1,024 columns): 8 of 4,096 x 1,408 at 6 pairs 37.2/32.2, 16 of 2,048 x 768 21.9/19.6, 4 of
    // 1,024 x 512 at 16 13.3/12.0; 512 x 256 at 2 8.0/8.4.  With more workgroups it is slower: of 530 steps (8 to 128 experts, 1.5 to 23
    // pairs) by 3% in the mean with 256 to 512, by 18% with 576 to 768, which moe_tile_kernel takes in one round (32 of 4,096 x 2,112 at 6
    // 126/131, 64 at 1.5 108/125), 3% faster with 800 to 1,000 and slower again beyond (64 at 4, even, 176/194); how many there
    // are is the router's choice.
    // The scratch is sized for tiles of 64: it holds the pairs without gaps and, at its end, the counters and the experts' offsets.
    const long fb = (F + 127) / 128, up_blocks = (gated ? (F + 63) / 64 : fb) * E;
    const bool wide = pairs >= 48L * E || (pairs >= 24L * E && up_blocks >= 1024);
    const bool wide_up = wide || (!gated && n <= MOE_TILE && H >= 1024 && fb * (pairs < E ? pairs : E) <= 256);
    // moe_product_kernel from 64 pairs an expert, 16 experts and 14e9 products of a matrix's numbers with rows on (21e9 of narrow experts), of widths
    // that it takes.
    // Up + down + the rest of the call, us, moe_wide_kernel / moe_product_kernel:
    //   64 of 4,096 x 1,408 gated, 6 a token, uneven: 2,048 tokens 670/612, even routing 688/555, 16 of 80 identity 640/542, 1,200 572/473, 700 (66 an
    //     expert) 468/408; 512 (48, even) 413/436.  Of 4,096 x 2,112 without a gate 2,048 720/664, 300 (28) 402/414
    //   92 drawn steps of this rule (16 to 160 experts of 1,600 to 4,700 x 512 to 2,500, even routing to a few experts with most rows): 8% faster in
    //     the mean, 25% at most; 11 slower, all but one of fewer than 20e9 products: 16 to 24 experts of which a few have most rows 2 to 34%,
    //     others up to 11% (of 24 steps of 14e9 to 21e9 half are faster, up to 22%)
    //   fewer than 1,600 columns (24 pieces a tile): below 21e9 level to 18% slower (64 of 1,088 x 576 at 351 an expert 184/197), above 2 to 15% faster
    //   smaller: 64 of 2,048 x 512, 16 pieces and 700 tasks for 256 CUs, 144/168 at 128 an expert (8.6e9), 123/140 at 176 without a gate
    //     (11.8e9), 2,048 x 1,408 260/237 at 87 (16e9); 16 of 1,024 x 1,536 75/89 at 180 (4.5e9)
    //   8 experts: 264 tasks are two rounds, 4,096 x 1,408 at 455 an expert 177/210
    const bool many = pairs >= 64L * E && E >= 16 && pairs * H >= (H < 1600 ? 21000000000L : 14000000000L) / F;
    const bool large = wide && many && moe_product_takes(H, F, gated, n, ldh, pairs, top) && moe_product_takes(F, H, false, pairs, F, pairs, top) &&
                       (uintptr_t)y % 16 == 0;
    const int tile_rows = large ? MOE_PRODUCT_ROWS : wide ? MOE_WIDE : MOE_TILE;
    const long tiles = (pairs + tile_rows - 1) / tile_rows + E;
    const long behind = (long)max_tiles * MOE_TILE - (E + 1) - MOE_PRODUCT_COUNTERS;      // pairs <= behind: max_tiles covers 64 E rows more
    int* counters = rows + behind;
    int* offs = counters + MOE_PRODUCT_COUNTERS;
    CPMCU_REQUIRE(pairs <= behind && (long)max_tiles * MOE_TILE < (1L << 31), "moe_experts_mfma: scratch of %d tiles for %ld pairs", max_tiles, pairs);
    moe_group_kernel<<<1, 1024, 0, stream>>>(idx, (int)pairs, E, tile_rows, rows, offs, tile_expert, n_tiles, counters, large);
    CPMCU_LAUNCH_CHECK("moe_group");
#define TILES(KIND, wide, in, ldi, w, out, K, N, act, limit)                                                              \
    do {                                                                                                                  \
        const long blocks = (tiles * (((N) + (KIND == MOE_GATED ? 63 : 127)) / (KIND == MOE_GATED ? 64 : 128)) + 7) / 8 * 8;   \
        CPMCU_REQUIRE(blocks < (1L << 31), "moe_experts_mfma: %ld workgroups exceed the launch grid", blocks);             \
        auto* const kernel = wide ? moe_wide_kernel<KIND> : moe_tile_kernel<KIND>;                                         \
        kernel<<<(unsigned)blocks, 256, 0, stream>>>(in, ldi, (const bf16_t*)(w), rows, offs, tile_expert, n_tiles,        \
                                                     (bf16_t*)(out), K, N, top, tile_rows, act, limit);                    \
    } while (0)
    if (large) {
        if (const char* m = moe_product(gated ? MOE_GATED : MOE_PLAIN, (const bf16_t*)h, ldh, (const bf16_t*)wgu, rows, offs, tile_expert,
                                        n_tiles, counters, (bf16_t*)act, pairs, H, F, top, tiles, act_fn, act_limit, stream)) return m;
        if (const char* m = moe_product(MOE_DOWN, (const bf16_t*)act, F, (const bf16_t*)wd, rows, offs, tile_expert, n_tiles,
                                        counters + 8, (bf16_t*)y, pairs, F, H, top, tiles, 0, 0.f, stream)) return m;
    } else {
        if (gated) TILES(MOE_GATED, wide, (const bf16_t*)h, ldh, wgu, act, H, F, act_fn, act_limit);
        else TILES(MOE_PLAIN, wide_up, (const bf16_t*)h, ldh, wgu, act, H, F, act_fn, act_limit);
        CPMCU_LAUNCH_CHECK("moe_up_tiles");
        TILES(MOE_DOWN, wide, (const bf16_t*)act, (long)F, wd, y, F, H, 0, 0.f);
        CPMCU_LAUNCH_CHECK("moe_down_tiles");
    }
#undef TILES
    const long total = (long)n * H;
    const bool vec = H % 4 == 0 && ldh % 4 == 0 && (uintptr_t)y % 16 == 0 && (uintptr_t)(x ? x : out) % 16 == 0;
    const long work = vec ? total / 4 : total;
    const int blocks = (int)((work + 255) / 256 < 8192 ? (work + 255) / 256 : 8192);
    // (the token kernel's rows start on 16-byte borders: H % 8 == 0, and y and the result are looked at here)
    if (top <= 8 && (uintptr_t)y % 16 == 0 && (uintptr_t)(x ? x : out) % 16 == 0 && (long)n * ((H + 2047) / 2048) < (1L << 31)) {
        const int pieces = (H + 2047) / 2048;
#define TOKENS(STv, TOPv)                                                                                                  \
    case TOPv:                                                                                                             \
        moe_combine_token_kernel<STv, TOPv><<<(unsigned)((long)n * pieces), 256, 0, stream>>>(                             \
            (const bf16_t*)y, w, (const STv*)shared, shared_parts, shared_stride, sg, idx, (const bf16_t*)h, ldh, E, out, H, pieces, join); \
        break
#define BY_TOP(STv)                                                                                                        \
    switch (top) { TOKENS(STv, 1); TOKENS(STv, 2); TOKENS(STv, 3); TOKENS(STv, 4); TOKENS(STv, 5); TOKENS(STv, 6); TOKENS(STv, 7); TOKENS(STv, 8); }
        if (!shared || shared_dtype == CPMCU_F32) BY_TOP(float)
        else BY_TOP(bf16_t)
#undef BY_TOP
#undef TOKENS
        CPMCU_LAUNCH_CHECK("moe_combine");
        return nullptr;
    }
#define COMBINE(STv, Vv)                                                                                              \
    moe_combine_kernel<STv, Vv><<<blocks, 256, 0, stream>>>((const bf16_t*)y, w, (const STv*)shared, shared_parts,   \
                                                            shared_stride, sg, idx, (const bf16_t*)h, ldh, E, out,  \
                                                            total, H, top, join)
    if (!shared || shared_dtype == CPMCU_F32) {
        if (vec) COMBINE(float, 4);
        else COMBINE(float, 1);
    } else {
        if (vec) COMBINE(bf16_t, 4);
        else COMBINE(bf16_t, 1);
    }
#undef COMBINE
    CPMCU_LAUNCH_CHECK("moe_combine");
    return nullptr;
}
