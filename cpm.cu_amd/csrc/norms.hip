// Norms beyond the residual RMSNorm of elementwise.hip, all with float statistics:
//
//  * rms_norm_groups_kernel: RMS norm of a row cut into equal groups, each by its own root mean square,
//    optionally after a SiLU gate (y <- y * silu(z), the gate before the norm) or followed by a sigmoid gate
//    (out <- norm(y) * w * sigmoid(z), the gate after the norm).  Rows may be slices of wider
//    rows (leading dimensions), so the first columns of a projection are normed where they lie.
//  * branch_norm_add_norm_kernel: a branch that has a norm of its own before it joins the residual
//    (x += rmsnorm(b) * wb), then the norm of the next sub-layer on the sum (out = rmsnorm(x) * w): the
//    arrangement "norm before and after every sub-layer" in one pass over the row.
//  * poly_norm_kernel: the PolyNorm activation a N(z) + b N(z^2) + c N(z^3) + e, N = division by the root mean
//    square of the row's values (powers element by element).
//
// RMS norm here always means x / sqrt(mean(x^2) + eps), eps inside the root.
#include "common.h"
#include "vec4.h"

template <typename T>
__device__ inline float sum_slices(const T* p, int nparts, long stride) {
    float v = 0.f;
    for (int i = 0; i < nparts; ++i) v += to_f32(p[(long)i * stride]);
    return v;
}

__device__ inline float silu_f(float z) { return z / (1.0f + expf(-z)); }

// grid (rows, groups); out[r, g*W + c] = v * rsqrt(mean_g(v^2) + eps) * weight[g*W + c], v = x * silu(z) if z and
// gate_after == 0; with gate_after the statistics are those of x alone and the result is multiplied by sigmoid(z)
// (gate_after == 1) or by silu(z) (gate_after == 2)
template <typename XT, typename ZT, typename OT>
__global__ __launch_bounds__(1024) void rms_norm_groups_kernel(const XT* __restrict__ x, long ldx,
                                                              const ZT* __restrict__ z, long ldz,
                                                              const float* __restrict__ weight, OT* __restrict__ out,
                                                              long ldo, int W, float eps, int gate_after,
                                                              const float* __restrict__ divisor) {
    __shared__ float red[17];
    const long r = blockIdx.x;
    const int g = blockIdx.y;
    const XT* xr = x + r * ldx + (long)g * W;
    const ZT* zr = z ? z + r * ldz + (long)g * W : nullptr;
    const bool before = zr && !gate_after;
    // divisor: one number a (row, group) by which the group's values are divided first
    const float pre = divisor ? 1.0f / divisor[r * gridDim.y + g] : 1.0f;
    float ss = 0.f;
    for (int c = threadIdx.x; c < W; c += blockDim.x) {
        float v = to_f32(xr[c]) * pre;
        if (before) v *= silu_f(to_f32(zr[c]));
        ss += v * v;
    }
    ss = block_sum(ss, red);
    const float rs = 1.0f / sqrtf(ss / (float)W + eps);
    OT* orow = out + r * ldo + (long)g * W;
    for (int c = threadIdx.x; c < W; c += blockDim.x) {
        float v = to_f32(xr[c]) * pre;
        if (before) v *= silu_f(to_f32(zr[c]));
        v *= rs;
        if (weight) v *= weight[(long)g * W + c];
        if (zr && gate_after) v *= gate_after == 2 ? silu_f(to_f32(zr[c])) : 1.0f / (1.0f + expf(-to_f32(zr[c])));
        orow[c] = from_f32<OT>(v);
    }
}

// The same with 16-byte accesses and a group's values kept in registers between the sum and the result, 4 NQ a thread: THREADS 64
// (up to 1,024 columns): a wavefront a group, four groups a workgroup, no barrier; 256 (up to 4,096): a workgroup a group.  All of a
// group's loads are in flight at once.  The bytes bound it: 2,048 rows of 8 groups of 1,024, float in, bf16 gate and result,
// 65 -> 32 us (134 MB); 1,500 rows of 16 groups of 256 31 -> 15, 2,048 rows of 4,096 27 -> 19.
template <typename XT, typename ZT, typename OT, int THREADS, int NQ>
__global__ __launch_bounds__(256) void rms_norm_groups_vec_kernel(const XT* __restrict__ x, long ldx, const ZT* __restrict__ z,
                                                                  long ldz, const float* __restrict__ weight, OT* __restrict__ out,
                                                                  long ldo, int W, int groups, int total, float eps, int gate_after,
                                                                  const float* __restrict__ divisor) {
    __shared__ float red[17];
    __shared__ float4 held[THREADS == 64 ? 4 : 1][64 * NQ * (THREADS / 64)];     // the groups' values
    const int at = THREADS == 64 ? blockIdx.x * 4 + (threadIdx.x >> 6) : blockIdx.x, t = threadIdx.x % THREADS;
    if (at >= total) return;
    const long r = at / groups;
    const int g = at % groups;
    const XT* xr = x + r * ldx + (long)g * W;
    const ZT* zr = z ? z + r * ldz + (long)g * W : nullptr;
    const bool before = zr && !gate_after;
    const float pre = divisor ? 1.0f / divisor[at] : 1.0f;
    float4 v[NQ], gt[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) v[i] = load4(xr + min((t + i * THREADS) * 4, W - 4));
    if (zr) {
#pragma unroll
        for (int i = 0; i < NQ; ++i) gt[i] = load4(zr + min((t + i * THREADS) * 4, W - 4));
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
        float* e = (float*)&v[i];
        const float* q = (const float*)&gt[i];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            e[j] *= pre;
            if (before) e[j] *= silu_f(q[j]);
        }
    }
    // the squares are added as rms_norm_groups_kernel's 256 threads add them, to the last bit
    float4* const own = held[THREADS == 64 ? threadIdx.x >> 6 : 0];
#pragma unroll
    for (int i = 0; i < NQ; ++i) own[t + i * THREADS] = v[i];
    const float* const vs = (const float*)own;
    if (THREADS == 64) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");       // (a wavefront's LDS accesses keep their order)
#pragma unroll
        for (int part = 0; part < 4; ++part) {
            float sq = 0.f;
#pragma unroll
            for (int i = 0; i < NQ; ++i) {
                const int c = 64 * part + t + 256 * i;
                if (c < W) sq += vs[c] * vs[c];
            }
            ss += wave_sum(sq);
        }
    } else {
        __syncthreads();
        for (int c = t; c < W; c += 256) ss += vs[c] * vs[c];
        ss = block_sum(ss, red);
    }
    const float rs = 1.0f / sqrtf(ss / (float)W + eps);
    OT* orow = out + r * ldo + (long)g * W;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
        const int c = (t + i * THREADS) * 4;
        if (c >= W) continue;
        float* e = (float*)&v[i];
        const float* q = (const float*)&gt[i];
        const float4 w4 = weight ? load4(weight + (long)g * W + c) : make_float4(1.f, 1.f, 1.f, 1.f);
        const float* w = (const float*)&w4;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            e[j] *= rs;
            if (weight) e[j] *= w[j];
            if (zr && gate_after) e[j] *= gate_after == 2 ? silu_f(q[j]) : 1.0f / (1.0f + expf(-q[j]));
        }
        store4(orow + c, e[0], e[1], e[2], e[3]);
    }
}

extern "C" const char* cpmcu_rms_norm_groups(const void* x, long ldx, int x_dtype, const void* z, long ldz, int z_dtype,
                                             const float* weight, void* out, long ldo, int out_dtype, int n, int groups,
                                             int W, float eps, int gate_after, const float* divisor,
                                             hipStream_t stream) {
    CPMCU_REQUIRE(n > 0 && groups > 0 && W > 0, "rms_norm_groups: empty shape rows=%d groups=%d width=%d", n, groups, W);
    CPMCU_REQUIRE(groups <= 65535, "rms_norm_groups: %d groups exceed the launch grid", groups);
    CPMCU_REQUIRE(ldx >= (long)groups * W && ldo >= (long)groups * W && (!z || ldz >= (long)groups * W),
                  "rms_norm_groups: leading dimensions too small for %d groups of %d", groups, W);
    dim3 grid(n, groups);
    // a group as wide as a model (one norm over all heads) on few rows is a handful of workgroups, each a chain of
    // dependent passes over its row: 1,024 threads shorten the chain
    const int block = (W >= 2048 && (long)n * groups < 1024) ? 1024 : (W >= 256 ? 256 : 64);
    const int zd = z ? z_dtype : x_dtype;
    const auto off = [](const void* p, int dtype) { return (uintptr_t)p % (dtype == CPMCU_F32 ? 16 : 8) != 0; };
    // The vector kernel where it was the faster one.  256 columns at any number of groups (us, general / here: 5 groups 2.8/2.2, 160
    // 3.1/3.2, 2,200 5.2/4.1) and more than 1,024 (7 groups of 1,280 5.4/4.8, 380 of 1,536 9.2/5.1).  Between, a wavefront's own chain
    // is longer than a workgroup's of one load a lane, and only many groups make up for it: 24 of 768 4.2/5.3, 224 of 320 3.6/4.4, 823 of
    // 264 4.2/5.4, 1,176 of 516 5.6/8.2, 1,336 of 516 6.1/7.2; 1,560 and more level (1,568 of 1,024 9.2/9.0) to 2.7 times
    // as fast, 1,128 of 448 to 1,376 of 1,024 on both sides.  Groups under 256 columns would leave lanes of their wavefront idle and
    // few wide ones have 1,024 threads: the general kernel's.  The others' results are its own.
    const bool pays = W == 256 || W > 1024 || (long)n * groups >= 1536;
    const bool vec = W % 4 == 0 && W >= 256 && W <= 4096 && block == 256 && pays && ldx % 4 == 0 && ldo % 4 == 0 && (!z || ldz % 4 == 0) && (long)n * groups < (1L << 31) &&
                     !off(x, x_dtype) && !off(out, out_dtype) && !(z && off(z, zd)) && (uintptr_t)weight % 16 == 0;
    const int total = vec ? n * groups : 0;
#define VEC(XT, ZT, OT, THREADS, NQ)                                                                          \
    rms_norm_groups_vec_kernel<XT, ZT, OT, THREADS, NQ><<<(unsigned)(THREADS == 64 ? ((long)total + 3) / 4 : total), 256, 0, stream>>>( \
        (const XT*)x, ldx, (const ZT*)z, ldz, weight, (OT*)out, ldo, W, groups, total, eps, gate_after, divisor)
#define LAUNCH(XT, ZT, OT)                                                                                     \
    do {                                                                                                       \
        if (vec && W <= 256) VEC(XT, ZT, OT, 64, 1);                                                           \
        else if (vec && W <= 512) VEC(XT, ZT, OT, 64, 2);                                                      \
        else if (vec && W <= 1024) VEC(XT, ZT, OT, 64, 4);                                                     \
        else if (vec) VEC(XT, ZT, OT, 256, 4);                                                                 \
        else                                                                                                   \
            rms_norm_groups_kernel<XT, ZT, OT><<<grid, block, 0, stream>>>((const XT*)x, ldx, (const ZT*)z, ldz, weight, \
                                                                           (OT*)out, ldo, W, eps, gate_after, divisor); \
    } while (0)
    if (x_dtype == CPMCU_F32 && zd == CPMCU_F32 && out_dtype == CPMCU_F32) LAUNCH(float, float, float);
    else if (x_dtype == CPMCU_F32 && zd == CPMCU_F32 && out_dtype == CPMCU_BF16) LAUNCH(float, float, bf16_t);
    else if (x_dtype == CPMCU_F32 && zd == CPMCU_BF16 && out_dtype == CPMCU_BF16) LAUNCH(float, bf16_t, bf16_t);
    else if (x_dtype == CPMCU_BF16 && zd == CPMCU_BF16 && out_dtype == CPMCU_BF16) LAUNCH(bf16_t, bf16_t, bf16_t);
    else if (x_dtype == CPMCU_BF16 && zd == CPMCU_BF16 && out_dtype == CPMCU_F32) LAUNCH(bf16_t, bf16_t, float);
    else CPMCU_FAIL("rms_norm_groups: unsupported dtypes x=%d z=%d out=%d", x_dtype, zd, out_dtype);
#undef LAUNCH
#undef VEC
    CPMCU_LAUNCH_CHECK("rms_norm_groups");
    return nullptr;
}

// One workgroup a row.  b may come as float partial sums [nparts][n][H].  With `rows` only those rows are
// computed, into out[R, H], and x stays as it was (the final norm on the wanted rows).
template <typename BT, typename OT>
__global__ __launch_bounds__(256) void branch_norm_add_norm_kernel(float* __restrict__ x, const BT* __restrict__ b,
                                                                   int nparts, long part_stride,
                                                                   const float* __restrict__ wb, float eps_b,
                                                                   const float* __restrict__ w, float eps,
                                                                   OT* __restrict__ out, const int* __restrict__ rows,
                                                                   int H) {
    __shared__ float red[17];
    const long r = rows ? rows[blockIdx.x] : blockIdx.x;
    float* xr = x + r * H;
    const BT* br = b + r * H;
    float sb = 0.f;
    for (int c = threadIdx.x; c < H; c += blockDim.x) {
        const float v = sum_slices(br + c, nparts, part_stride);
        sb += v * v;
    }
    sb = block_sum(sb, red);
    const float rb = 1.0f / sqrtf(sb / (float)H + eps_b);
    float sx = 0.f;
    for (int c = threadIdx.x; c < H; c += blockDim.x) {
        const float v = xr[c] + sum_slices(br + c, nparts, part_stride) * rb * wb[c];
        if (!rows) xr[c] = v;
        sx += v * v;
    }
    if (!out) return;
    sx = block_sum(sx, red);
    const float rx = 1.0f / sqrtf(sx / (float)H + eps);
    OT* orow = out + (long)blockIdx.x * H;
    for (int c = threadIdx.x; c < H; c += blockDim.x) {
        const float v = rows ? xr[c] + sum_slices(br + c, nparts, part_stride) * rb * wb[c] : xr[c];
        orow[c] = from_f32<OT>(v * rx * w[c]);
    }
}

// The same with the row held in registers (H <= 1024 * VPT): one trip to memory for the branch's slices and the
// residual, all loads of a thread in flight together (a loop of dependent passes over the row costs a step of
// few rows ten times as much).
template <typename BT, typename OT, int VPT>
__global__ __launch_bounds__(1024) void branch_norm_add_norm_reg_kernel(float* __restrict__ x, const BT* __restrict__ b,
                                                                        int nparts, long part_stride,
                                                                        const float* __restrict__ wb, float eps_b,
                                                                        const float* __restrict__ w, float eps,
                                                                        OT* __restrict__ out,
                                                                        const int* __restrict__ rows, int H) {
    __shared__ float red[17];
    const long r = rows ? rows[blockIdx.x] : blockIdx.x;
    float* xr = x + r * H;
    const BT* br = b + r * H;
    float bv[VPT], xv[VPT], wbv[VPT], wv[VPT];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int c = threadIdx.x + i * 1024;
        bv[i] = 0.f;
        xv[i] = c < H ? xr[c] : 0.f;
        wbv[i] = c < H ? wb[c] : 0.f;
        wv[i] = (c < H && out) ? w[c] : 0.f;
    }
    // four slices' loads are issued before any of them is added
    int p = 0;
    for (; p + 4 <= nparts; p += 4) {
        float t4[4][VPT];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int i = 0; i < VPT; ++i) {
                const int c = min((int)threadIdx.x + i * 1024, H - 1);  // clamped: no load in a branch
                t4[u][i] = to_f32(br[(long)(p + u) * part_stride + c]);
            }
#pragma unroll
        for (int i = 0; i < VPT; ++i) bv[i] += (t4[0][i] + t4[1][i]) + (t4[2][i] + t4[3][i]);
    }
    for (; p < nparts; ++p) {
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            const int c = min((int)threadIdx.x + i * 1024, H - 1);
            bv[i] += to_f32(br[(long)p * part_stride + c]);
        }
    }
    float sb = 0.f;
#pragma unroll
    for (int i = 0; i < VPT; ++i)
        if ((int)threadIdx.x + i * 1024 >= H) bv[i] = 0.f;
#pragma unroll
    for (int i = 0; i < VPT; ++i) sb += bv[i] * bv[i];
    sb = block_sum(sb, red);
    const float rb = 1.0f / sqrtf(sb / (float)H + eps_b);
    float sx = 0.f;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int c = threadIdx.x + i * 1024;
        xv[i] += bv[i] * rb * wbv[i];
        if (!rows && c < H) xr[c] = xv[i];
        sx += xv[i] * xv[i];
    }
    if (!out) return;
    sx = block_sum(sx, red);
    const float rx = 1.0f / sqrtf(sx / (float)H + eps);
    OT* orow = out + (long)blockIdx.x * H;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int c = threadIdx.x + i * 1024;
        if (c < H) orow[c] = from_f32<OT>(xv[i] * rx * wv[i]);
    }
}

// The same for steps of many rows, up to 1,024 NQ columns and a branch that is one tensor: 256 threads a row, 4 neighbouring columns
// NQ times each, with 16-byte accesses.  Its bytes bound it; with 4-byte accesses and 1,024 threads behind every barrier 2,048
// rows of 4,096 took 28.9 us, here 16.4 (bf16 branch and result, 100 MB); 300 rows 13.1 -> 8.4, 1,000 of 6,144 19.9 -> 12.6.
template <typename BT, typename OT, int NQ>
__global__ __launch_bounds__(256) void branch_norm_add_norm_vec_kernel(float* __restrict__ x, const BT* __restrict__ b,
                                                                       const float* __restrict__ wb, float eps_b,
                                                                       const float* __restrict__ w, float eps,
                                                                       OT* __restrict__ out, int H) {
    __shared__ float red[17];
    const long r = blockIdx.x;
    float4 bv[NQ], xv[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
        const int c = min((int)(threadIdx.x + i * 256) * 4, H - 4);
        bv[i] = load4(b + r * H + c);
        xv[i] = load4(x + r * H + c);
    }
    float sb = 0.f;
#pragma unroll
    for (int i = 0; i < NQ; ++i)
        if ((int)(threadIdx.x + i * 256) * 4 < H) sb += (bv[i].x * bv[i].x + bv[i].y * bv[i].y) + (bv[i].z * bv[i].z + bv[i].w * bv[i].w);
    sb = block_sum(sb, red);
    const float rb = 1.0f / sqrtf(sb / (float)H + eps_b);
    float sx = 0.f;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
        const int c = (threadIdx.x + i * 256) * 4;
        if (c >= H) continue;
        const float4 g = load4(wb + c);
        xv[i].x += bv[i].x * rb * g.x; xv[i].y += bv[i].y * rb * g.y;
        xv[i].z += bv[i].z * rb * g.z; xv[i].w += bv[i].w * rb * g.w;
        store4(x + r * H + c, xv[i].x, xv[i].y, xv[i].z, xv[i].w);
        sx += (xv[i].x * xv[i].x + xv[i].y * xv[i].y) + (xv[i].z * xv[i].z + xv[i].w * xv[i].w);
    }
    if (!out) return;
    sx = block_sum(sx, red);
    const float rx = 1.0f / sqrtf(sx / (float)H + eps);
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
        const int c = (threadIdx.x + i * 256) * 4;
        if (c >= H) continue;
        const float4 g = load4(w + c);
        store4(out + r * H + c, xv[i].x * rx * g.x, xv[i].y * rx * g.y, xv[i].z * rx * g.z, xv[i].w * rx * g.w);
    }
}

extern "C" const char* cpmcu_branch_norm_add_norm(float* x, const void* b, int b_dtype, int nparts, long part_stride,
                                                  const float* wb, float eps_b, const float* w, float eps, void* out,
                                                  int out_dtype, const int* rows, int n_out, int H,
                                                  hipStream_t stream) {
    CPMCU_REQUIRE(n_out > 0 && H > 0 && nparts >= 1, "branch_norm_add_norm: empty shape rows=%d width=%d", n_out, H);
    CPMCU_REQUIRE(x && b && wb && (!out || w), "branch_norm_add_norm: a pointer is missing");
    CPMCU_REQUIRE(!rows || out, "branch_norm_add_norm: a list of rows needs an output");
    // From a row for every CU on; fewer rows end sooner with 1,024 threads each.
    const auto off = [](const void* p, int dtype) { return (uintptr_t)p % (dtype == CPMCU_F32 ? 16 : 8) != 0; };
    const bool vec = !rows && nparts == 1 && n_out >= 256 && H % 4 == 0 && H <= 8192 && !off(x, CPMCU_F32) && !off(b, b_dtype) &&
                     !off(out, out_dtype) && !off(wb, CPMCU_F32) && !off(w, CPMCU_F32);
#define VEC(BT, OT, NQ) branch_norm_add_norm_vec_kernel<BT, OT, NQ><<<n_out, 256, 0, stream>>>(x, (const BT*)b, wb, eps_b, w, eps, (OT*)out, H)
#define LAUNCH(BT, OT)                                                                                              \
    do {                                                                                                            \
        if (vec && H <= 2048) VEC(BT, OT, 2);                                                                       \
        else if (vec && H <= 4096) VEC(BT, OT, 4);                                                                  \
        else if (vec) VEC(BT, OT, 8);                                                                               \
        else if (H <= 2048)                                                                                         \
            branch_norm_add_norm_reg_kernel<BT, OT, 2><<<n_out, 1024, 0, stream>>>(                                 \
                x, (const BT*)b, nparts, part_stride, wb, eps_b, w, eps, (OT*)out, rows, H);                        \
        else if (H <= 4096)                                                                                         \
            branch_norm_add_norm_reg_kernel<BT, OT, 4><<<n_out, 1024, 0, stream>>>(                                 \
                x, (const BT*)b, nparts, part_stride, wb, eps_b, w, eps, (OT*)out, rows, H);                        \
        else if (H <= 8192)                                                                                         \
            branch_norm_add_norm_reg_kernel<BT, OT, 8><<<n_out, 1024, 0, stream>>>(                                 \
                x, (const BT*)b, nparts, part_stride, wb, eps_b, w, eps, (OT*)out, rows, H);                        \
        else                                                                                                        \
            branch_norm_add_norm_kernel<BT, OT><<<n_out, 256, 0, stream>>>(x, (const BT*)b, nparts, part_stride, wb, \
                                                                           eps_b, w, eps, (OT*)out, rows, H);       \
    } while (0)
    if (b_dtype == CPMCU_F32 && out_dtype == CPMCU_F32) LAUNCH(float, float);
    else if (b_dtype == CPMCU_F32 && out_dtype == CPMCU_BF16) LAUNCH(float, bf16_t);
    else if (b_dtype == CPMCU_BF16 && out_dtype == CPMCU_BF16) LAUNCH(bf16_t, bf16_t);
    else if (b_dtype == CPMCU_BF16 && out_dtype == CPMCU_F32) LAUNCH(bf16_t, float);
    else CPMCU_FAIL("branch_norm_add_norm: unsupported dtypes branch=%d out=%d", b_dtype, out_dtype);
#undef LAUNCH
#undef VEC
    CPMCU_LAUNCH_CHECK("branch_norm_add_norm");
    return nullptr;
}

// out = a z / rms(z) + b z^2 / rms(z^2) + c z^3 / rms(z^3) + e;  coef = (a, b, c, e) on the device.
// z may come as float partial sums [nparts][n][F].
template <typename ZT, typename OT>
__global__ __launch_bounds__(256) void poly_norm_kernel(const ZT* __restrict__ z, int nparts, long part_stride,
                                                        const float* __restrict__ coef, OT* __restrict__ out, int F,
                                                        float eps) {
    __shared__ float red[17];
    const long r = blockIdx.x;
    const ZT* zr = z + r * F;
    float s2 = 0.f, s4 = 0.f, s6 = 0.f;
    for (int c = threadIdx.x; c < F; c += blockDim.x) {
        const float v = sum_slices(zr + c, nparts, part_stride);
        const float v2 = v * v;
        s2 += v2;
        s4 += v2 * v2;
        s6 += v2 * v2 * v2;
    }
    s2 = block_sum(s2, red);
    s4 = block_sum(s4, red);
    s6 = block_sum(s6, red);
    const float inv = 1.0f / (float)F;
    const float a = coef[0] / sqrtf(s2 * inv + eps), b = coef[1] / sqrtf(s4 * inv + eps),
                cc = coef[2] / sqrtf(s6 * inv + eps), e = coef[3];
    OT* orow = out + r * F;
    for (int c = threadIdx.x; c < F; c += blockDim.x) {
        const float v = sum_slices(zr + c, nparts, part_stride);
        orow[c] = from_f32<OT>(((cc * v + b) * v + a) * v + e);
    }
}

// The same with the row held in registers (F <= 1024 * VPT).
template <typename ZT, typename OT, int VPT>
__global__ __launch_bounds__(1024) void poly_norm_reg_kernel(const ZT* __restrict__ z, int nparts, long part_stride,
                                                             const float* __restrict__ coef, OT* __restrict__ out,
                                                             int F, float eps) {
    __shared__ float red[17];
    const long r = blockIdx.x;
    const ZT* zr = z + r * F;
    float zv[VPT];
#pragma unroll
    for (int i = 0; i < VPT; ++i) zv[i] = 0.f;
    for (int p = 0; p < nparts; ++p) {
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            const int c = threadIdx.x + i * 1024;
            if (c < F) zv[i] += to_f32(zr[(long)p * part_stride + c]);
        }
    }
    float s2 = 0.f, s4 = 0.f, s6 = 0.f;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const float v2 = zv[i] * zv[i];
        s2 += v2;
        s4 += v2 * v2;
        s6 += v2 * v2 * v2;
    }
    s2 = block_sum(s2, red);
    s4 = block_sum(s4, red);
    s6 = block_sum(s6, red);
    const float inv = 1.0f / (float)F;
    const float a = coef[0] / sqrtf(s2 * inv + eps), b = coef[1] / sqrtf(s4 * inv + eps),
                cc = coef[2] / sqrtf(s6 * inv + eps), e = coef[3];
    OT* orow = out + r * F;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int c = threadIdx.x + i * 1024;
        if (c < F) orow[c] = from_f32<OT>(((cc * zv[i] + b) * zv[i] + a) * zv[i] + e);
    }
}

// The same for 16-bit rows of whole 16-byte pieces (a prompt's): PIECES pieces a thread stay in registers as they came, and
// the three sums cross the workgroup together, behind one barrier.  Memory bounds it; with 2-byte accesses a row's 1,024
// threads waited for the address unit and at six barriers.  2,048 rows of 11,008: 48 -> 21 us; 4,096 wide 22 -> 12; 8 rows the same.
// Built for 1, 3 and 4 pieces; widths of 4,097 to 8,192 take three, the last of them empty, and gain as the others do (2,048
// rows that stay in the caches, us: 4,096 18 -> 11, 4,608 24 -> 14, 6,144 27 -> 15, 8,192 31 -> 15, 11,008 35 -> 16).
#define POLY_WIDE_THREADS 512
template <int PIECES>
__global__ __launch_bounds__(POLY_WIDE_THREADS) void poly_norm_wide_kernel(const bf16_t* __restrict__ z,
                                                                           const float* __restrict__ coef,
                                                                           bf16_t* __restrict__ out, int F, float eps) {
    constexpr int WAVES = POLY_WIDE_THREADS / 64;
    __shared__ float red[3][WAVES];
    const uint4* zr = (const uint4*)(z + (long)blockIdx.x * F);
    uint4* orow = (uint4*)(out + (long)blockIdx.x * F);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, pieces = F / 8;
    uint4 held[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        const int c = threadIdx.x + i * POLY_WIDE_THREADS;
        held[i] = c < pieces ? zr[c] : make_uint4(0, 0, 0, 0);
    }
    const float a0 = coef[0], b0 = coef[1], c0 = coef[2], e = coef[3];
    float s[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        const uint32_t w[4] = {held[i].x, held[i].y, held[i].z, held[i].w};
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float v = __uint_as_float(j & 1 ? w[j / 2] & 0xffff0000u : w[j / 2] << 16), v2 = v * v;
            s[0] += v2;
            s[1] += v2 * v2;
            s[2] += v2 * v2 * v2;
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        s[k] = wave_sum(s[k]);
        if (lane == 0) red[k][wave] = s[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        s[k] = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) s[k] += red[k][w];
    }
    const float inv = 1.0f / (float)F;
    const float a = a0 / sqrtf(s[0] * inv + eps), b = b0 / sqrtf(s[1] * inv + eps), cc = c0 / sqrtf(s[2] * inv + eps);
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        const int c = threadIdx.x + i * POLY_WIDE_THREADS;
        const uint32_t w[4] = {held[i].x, held[i].y, held[i].z, held[i].w};
        uint32_t o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float lo = __uint_as_float(w[j] << 16), hi = __uint_as_float(w[j] & 0xffff0000u);
            o[j] = (uint32_t)f32_to_bf16(((cc * lo + b) * lo + a) * lo + e).v |
                   (uint32_t)f32_to_bf16(((cc * hi + b) * hi + a) * hi + e).v << 16;
        }
        if (c < pieces) orow[c] = make_uint4(o[0], o[1], o[2], o[3]);
    }
}

extern "C" const char* cpmcu_poly_norm(const void* z, int z_dtype, int nparts, long part_stride, const float* coef,
                                       void* out, int out_dtype, int n, int F, float eps, hipStream_t stream) {
    CPMCU_REQUIRE(n > 0 && F > 0 && nparts >= 1, "poly_norm: empty shape rows=%d width=%d", n, F);
#define LAUNCH(ZT, OT)                                                                                          \
    do {                                                                                                        \
        if (F <= 4096)                                                                                          \
            poly_norm_reg_kernel<ZT, OT, 4><<<n, 1024, 0, stream>>>((const ZT*)z, nparts, part_stride, coef,    \
                                                                    (OT*)out, F, eps);                          \
        else if (F <= 16384)                                                                                    \
            poly_norm_reg_kernel<ZT, OT, 16><<<n, 1024, 0, stream>>>((const ZT*)z, nparts, part_stride, coef,   \
                                                                     (OT*)out, F, eps);                         \
        else                                                                                                    \
            poly_norm_kernel<ZT, OT><<<n, 256, 0, stream>>>((const ZT*)z, nparts, part_stride, coef, (OT*)out,  \
                                                            F, eps);                                            \
    } while (0)
    if (z_dtype == CPMCU_F32 && out_dtype == CPMCU_F32) LAUNCH(float, float);
    else if (z_dtype == CPMCU_F32 && out_dtype == CPMCU_BF16) LAUNCH(float, bf16_t);
    else if (z_dtype == CPMCU_BF16 && out_dtype == CPMCU_BF16 && nparts == 1 && F % 8 == 0 && F <= 4 * 8 * POLY_WIDE_THREADS &&
             (uintptr_t)z % 16 == 0 && (uintptr_t)out % 16 == 0) {
#define WIDE(P) poly_norm_wide_kernel<P><<<n, POLY_WIDE_THREADS, 0, stream>>>((const bf16_t*)z, coef, (bf16_t*)out, F, eps)
        if (F <= 8 * POLY_WIDE_THREADS) WIDE(1);
        else if (F <= 3 * 8 * POLY_WIDE_THREADS) WIDE(3);
        else WIDE(4);
#undef WIDE
    } else if (z_dtype == CPMCU_BF16 && out_dtype == CPMCU_BF16) LAUNCH(bf16_t, bf16_t);
    else CPMCU_FAIL("poly_norm: unsupported dtypes in=%d out=%d", z_dtype, out_dtype);
#undef LAUNCH
    CPMCU_LAUNCH_CHECK("poly_norm");
    return nullptr;
}
