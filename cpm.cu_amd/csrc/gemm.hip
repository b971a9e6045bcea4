// Matrix products of the linear layers:  Y[m,N] = alpha * X[m,K] . W[N,K]^T
// with weights stored [out, in] row-major as in the checkpoint (reference:
// src/model/linear.cuh:9-37 calls a library product with fp32 accumulation).
//
//  * gemm_tiled_kernel: LDS-tiled product with scalar float FMAs, any size: the plain twin of the bf16 products.
//  * gemm_f32_split_kernel, gemm_f32_shares_kernel, gemm_f32_mfma_kernel, gemm_f32_rows_kernel: the whole 32-bit engine's
//    product on the matrix cores, any size: with every float as the exact sum of three bf16, or on the float instruction.
#include "common.h"

#define GT_BM 64
#define GT_BN 64
#define GT_BK 16

template <typename XT, typename WT, typename OT>
__global__ __launch_bounds__(256) void gemm_tiled_kernel(const XT* __restrict__ X, long ldx,
                                                         const WT* __restrict__ W, long ldw, OT* __restrict__ Y,
                                                         long ldy, int M, int N, int K, float alpha) {
    __shared__ float xs[GT_BK][GT_BM + 1];
    __shared__ float ws[GT_BK][GT_BN + 1];
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    const int m0 = blockIdx.y * GT_BM, n0 = blockIdx.x * GT_BN;
    float acc[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += GT_BK) {
        // 64 rows x 16 k of each operand: 1024 elements, 4 per thread
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = threadIdx.x + i * 256;
            const int r = e / GT_BK, kk = e % GT_BK;
            const int k = k0 + kk;
            xs[kk][r] = (m0 + r < M && k < K) ? to_f32(X[(long)(m0 + r) * ldx + k]) : 0.f;
            ws[kk][r] = (n0 + r < N && k < K) ? to_f32(W[(long)(n0 + r) * ldw + k]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < GT_BK; ++kk) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = xs[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = ws[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] += a[i] * b[j];
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + ty * 4 + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + tx * 4 + j;
            if (n < N) Y[(long)m * ldy + n] = from_f32<OT>(alpha * acc[i][j]);
        }
    }
}

// ---------------------------------------------------------------------------
// The 32-bit product on the matrix cores.  v_mfma_f32_16x16x4_f32 takes float operands as they are and adds in float
// (32 multiply-adds a cycle and SIMD, 157 TFLOP/s on the chip); v_mfma_f32_16x16x32_bf16 does 16 times as many, so that eight
// of its products, which a float as three bf16 asks for (below), still are twice as fast.
//
// gemm_f32_mfma_kernel: the float instruction, for few columns.  256 threads, 2 x 2 wavefronts of 32 x 32 outputs each; 32 columns
// of both operands go through LDS in two buffers, the next ones on their way to registers meanwhile, one barrier a piece.  A row
// of a piece is 8 chunks of 16 bytes, chunk c of row r at place c ^ (r % 8), so that 8 neighbouring lanes (8 rows, one chunk) read
// all banks.  A lane's 16 bytes serve four instructions: in instruction s, lane group g stands for column 4 g + s of the 16, in
// both operands alike (a sum over columns may take them in any order).  Tiles of 32 x 32 outputs and 64 columns are level up to
// 130 x 8,192 and slower beyond (us, rows x outputs x columns: 2,048 x 4,096 x 32 22.3 -> 12.7, 523 x 8,192 x 48 12.4 -> 11.2).
// ---------------------------------------------------------------------------
typedef float gfloatx4_t __attribute__((ext_vector_type(4)));

// columns k .. k + 3 of a row of K, zero beyond its end; VEC: K % 4 == 0 and rows on 16-byte borders
template <bool VEC>
__device__ inline gfloatx4_t f32_piece(const float* __restrict__ row, int k, int K) {
    gfloatx4_t v = {0.f, 0.f, 0.f, 0.f};
    if (VEC) {
        const gfloatx4_t in = *(const gfloatx4_t*)(row + min(k, K - 4));     // no branch around the load
        if (k < K) v = in;
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (k + i < K) v[i] = row[k + i];
    }
    return v;
}

template <bool VEC>
__global__ __launch_bounds__(256) void gemm_f32_mfma_kernel(const float* __restrict__ X, long ldx,
                                                            const float* __restrict__ W, long ldw, float* __restrict__ Y,
                                                            long ldy, int M, int N, int K, float alpha) {
    constexpr int TM = 2, TN = 2, BK = 32, BM = 32 * TM, BN = 32 * TN, CH = BK / 4, PIECES = (BM + BN) * CH / 256;
    __shared__ float lds[2][(BM + BN) * BK];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    // rows beyond the matrices read the last one; their results are not stored
    const float* src[PIECES];
    int place[PIECES];
    const int chunk = threadIdx.x % CH;
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        const int row = threadIdx.x / CH + 256 / CH * i;
        src[i] = row < BM ? X + (long)min(m0 + row, M - 1) * ldx : W + (long)min(n0 + row - BM, N - 1) * ldw;
        place[i] = row * BK + ((chunk ^ (row & 7)) << 2);
    }
    gfloatx4_t next[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) next[i] = f32_piece<VEC>(src[i], chunk * 4, K);
    gfloatx4_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = gfloatx4_t{0.f, 0.f, 0.f, 0.f};
    const int row_a = (wave & 1) * 16 * TM + r, row_b = BM + (wave >> 1) * 16 * TN + r;
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += BK, buf ^= 1) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) *(gfloatx4_t*)&lds[buf][place[i]] = next[i];
        __syncthreads();
        if (k0 + BK < K) {
#pragma unroll
            for (int i = 0; i < PIECES; ++i) next[i] = f32_piece<VEC>(src[i], k0 + BK + chunk * 4, K);
        }
#pragma unroll
        for (int kb = 0; kb < BK / 16; ++kb) {
            const int at = ((kb * 4 + g) ^ (r & 7)) << 2;
            gfloatx4_t a[TM], b[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) a[i] = *(const gfloatx4_t*)&lds[buf][(row_a + 16 * i) * BK + at];
#pragma unroll
            for (int j = 0; j < TN; ++j) b[j] = *(const gfloatx4_t*)&lds[buf][(row_b + 16 * j) * BK + at];
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][s], b[j][s], acc[i][j], 0, 0, 0);
        }
    }
    // lane (column r, g): acc[i][j][e] is row 4 g + e of its 16 x 16 outputs
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int m = m0 + (wave & 1) * 16 * TM + 16 * i + 4 * g + e;
            if (m >= M) continue;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = n0 + (wave >> 1) * 16 * TN + 16 * j + r;
                if (n < N) Y[(long)m * ldy + n] = alpha * acc[i][j][e];
            }
        }
}

// ---------------------------------------------------------------------------
// The same product with every float as the sum of three bf16, x = h + m + l: the upper 8 bits, the upper 8 of what is left
// and the rest, exact for all that a float holds (down to 2^-110, where the last part ends below the smallest bf16).  Eight of
// the nine products go through v_mfma_f32_16x16x32_bf16; the last parts' own, below 2^-30 of a product, is left out.  That
// instruction cuts its sums' last bits where a float addition rounds them (all terms into one accumulator: sums of positive
// products 4e-7 too small), so a piece of 32 columns has two sums that start from zero, hh and the seven others, which end 2^-7
// below it, and meets the sum of the pieces in float additions.  Distance from a product in double, float instruction -> here:
// 1,024 columns 5.7e-7 -> 7.9e-8, 4,096 columns 1.15e-6 -> 1.0e-7; positive numbers 4.9e-7 -> 5.2e-8; rows of which one element is not zero 2.5e-8 in both, four 4.0e-8 -> 2.7e-8.
// Infinities, NaNs, inputs whose parts do not hold all of them and very small results are worked out on the float instruction
// (f32_finish_tile).
//
// gemm_f32_split_kernel: 64 rows against 64 TN outputs a workgroup.  X's piece of 32 columns is split once and its parts go
// through LDS in two buffers; a wavefront splits its own 16 TN rows of W in registers, which nobody else needs.  Two pieces on
// their way to registers (of 48 outputs a wavefront one).
// gemm_f32_shares_kernel: for outputs that give too few such workgroups: every one of 8 wavefronts has the whole tile of
// 16 TM x 16 TN outputs and an eighth of the columns, no barrier until their sums meet in LDS.  Pieces are brought
// whole lines a row (8 lanes each) and turned into operands through the wavefront's own LDS: loads straight into the operand's
// order, where 64 neighbouring lanes ask for 64 rows, pass one lane a cycle (523 x 1,024 x 4,096: 59.5 -> 46.2 us).
// What bounds both: a piece's vector instructions (352 of conversions for 64 x 64 outputs, 128 of sums) take about as long as its
// 128 matrix instructions, and the two overlap little; then grids that 256 CUs do not divide.
// Measured (us, tiles on the float instruction -> here; rows x outputs x columns): 523 x 8,192 x 1,024 108 -> 87 (101 TFLOP/s),
// 523 x 1,024 x 4,096 72 -> 52, 523 x 1,024 x 1,024 21.2 -> 16.5, 523 x 1,280 x 1,024 22.3 -> 18.0, 700 x 8,192 x 1,024 121 -> 94,
// 2,048 x 4,096 x 4,096 535 -> 517, 2,048 x 1,024 x 4,096 157 -> 149, 130 x 8,192 x 1,024 37.4 -> 38.1, 130 x 1,024 x 4,096 42 -> 27,
// 40 x 8,192 x 1,024 16.7 -> 14.1, 17 x 1,024 x 4,096 42 -> 24, 64 x 73,448 x 1,024 121 -> 105, 1 x 73,448 x 1,024 66 -> 60.
// ---------------------------------------------------------------------------
typedef __bf16 gbf16x8_t __attribute__((ext_vector_type(8)));
struct Split8 {      // eight floats as three bf16 each: upper, middle, last
    gbf16x8_t part[3];
};
// the upper halves of two floats, a's first
__device__ inline uint32_t f32_upper(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }
// (lost: its lower half gathers what a last part has no room for)
__device__ inline Split8 f32_split(const gfloatx4_t& x, const gfloatx4_t& y, uint32_t& lost) {
    union { uint32_t u[4]; gbf16x8_t v; } part[3];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t a = __float_as_uint(i < 2 ? x[2 * i] : y[2 * i - 4]), b = __float_as_uint(i < 2 ? x[2 * i + 1] : y[2 * i - 3]);
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            part[p].u[i] = f32_upper(a, b);
            if (p < 2) {
                a = __float_as_uint(__uint_as_float(a) - __uint_as_float(a & 0xffff0000u));
                b = __float_as_uint(__uint_as_float(b) - __uint_as_float(b & 0xffff0000u));
            }
        }
        lost |= a | b;
    }
    return {{part[0].v, part[1].v, part[2].v}};
}

// acc[i] += a piece of 32 columns of tile i's rows (x(p, i): part p of them) times w's.  The bf16 instruction cuts what its sum
// leaves below a float's last bit, so the products that reach there have a sum of their own, and every piece is added as floats.
template <int TM, typename XP>
__device__ inline void f32_multiply(const XP& x, const Split8& w, gfloatx4_t (&acc)[TM]) {
    constexpr int P[7] = {1, 2, 2, 0, 1, 1, 0}, Q[7] = {2, 1, 0, 2, 1, 0, 1};
    gfloatx4_t small[TM], big[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) small[i] = gfloatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 7; ++t)
#pragma unroll
        for (int i = 0; i < TM; ++i) small[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x(P[t], i), w.part[Q[t]], small[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < TM; ++i) big[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x(0, i), w.part[0], gfloatx4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[i] += big[i] + small[i];
}

// One 16 x 16 tile of a split product as it is stored.  A result is worked out again on the float instruction if an input of its
// rows has bits that its last part has no room for (odd: some row of the workgroup's has), if it is no finite number, which may
// stand for an infinity (whose parts are an infinity and no numbers), and if it is below 2^-64, where a product of parts may lie
// below the smallest float.  (A sum of exactly 0 is taken as it is: K 2^-126 at most are lost.)  The other results of the tile
// stay, so that none depends on its neighbours.
__device__ inline uint32_t f32_rest(float x) {
#pragma unroll
    for (int p = 0; p < 2; ++p) x -= __uint_as_float(__float_as_uint(x) & 0xffff0000u);
    return __float_as_uint(x) & 0xffff;
}
template <bool VEC>
__device__ inline void f32_finish_tile(gfloatx4_t sum, const float* __restrict__ X, long ldx, const float* __restrict__ W, long ldw,
                                       float* __restrict__ Y, long ldy, int M, int N, int K, float alpha, int m0, int n0,
                                       bool odd) {
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    bool again[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        again[e] = !(fabsf(sum[e]) < __builtin_inff()) || (fabsf(sum[e]) < 0x1p-64f && sum[e] != 0.f);
        odd |= again[e];
    }
    if (__any(odd)) {
        const float* xr = X + (long)min(m0 + r, M - 1) * ldx;
        const float* wr = W + (long)min(n0 + r, N - 1) * ldw;
        gfloatx4_t whole = {0.f, 0.f, 0.f, 0.f};
        uint32_t rest_x = 0, rest_w = 0;                             // of row r of each
        for (int k = 0; k < K; k += 16) {
            const gfloatx4_t a = f32_piece<VEC>(xr, k + 4 * g, K), b = f32_piece<VEC>(wr, k + 4 * g, K);
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                whole = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b[s], whole, 0, 0, 0);
                rest_x |= f32_rest(a[s]);
                rest_w |= f32_rest(b[s]);
            }
        }
#pragma unroll
        for (int d = 16; d < 64; d *= 2) {
            rest_x |= __shfl_xor(rest_x, d);
            rest_w |= __shfl_xor(rest_w, d);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t rest = rest_w | __shfl(rest_x, 4 * g + e);        // (by all lanes)
            if (again[e] || rest) sum[e] = whole[e];
        }
    }
    // lane (column r, g): sum[e] is row 4 g + e
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int m = m0 + 4 * g + e, n = n0 + r;
        if (m < M && n < N) Y[(long)m * ldy + n] = alpha * sum[e];
    }
}

// Which tile a workgroup takes: workgroups go to the 8 XCDs in turn, and neighbouring tiles (same outputs, other rows) to
// one XCD, whose L2 then reads their weights once.
__device__ inline int tile_of_workgroup(int wg, int tiles) {
    const int per = tiles / 8, more = tiles % 8, x = wg % 8;
    return x * per + min(x, more) + wg / 8;
}

// The pieces of a share of the columns, an eighth.  Every kernel here adds a share's pieces in their order and then the shares, and
// so a row's result does not depend on how many rows there are.
__device__ inline int f32_share(int K) { return ((K + 31) / 32 + 7) / 8; }

template <int TM, int TN, bool VEC>
__global__ __launch_bounds__(256, 2) void gemm_f32_split_kernel(
    const float* __restrict__ X, long ldx, const float* __restrict__ W, long ldw, float* __restrict__ Y, long ldy, int M, int N,
    int K, float alpha, int m_tiles, int tiles) {
    constexpr int TASKS = TM / 4, PLANE = TM * 16 * 64, BUF = 3 * PLANE;
    constexpr bool AHEAD = TN < 3;       // two pieces of W on their way (of 48 outputs a wavefront one: registers)
    __shared__ __attribute__((aligned(16))) char lds[2 * BUF];
    __shared__ gfloatx4_t total[TN * TM][256];               // the sum of whole shares, a thread's own
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int t = tile_of_workgroup(blockIdx.x, tiles);
    const int m0 = t % m_tiles * 16 * TM, n0 = (t / m_tiles * 4 + wave) * 16 * TN;
    const float *xr[TASKS], *wr[TN];
    int place[TASKS];
    const int chunk = threadIdx.x & 3;
#pragma unroll
    for (int i = 0; i < TASKS; ++i) {
        const int row = (threadIdx.x >> 2) + 64 * i;
        xr[i] = X + (long)min(m0 + row, M - 1) * ldx;
        place[i] = row * 64 + ((chunk ^ ((row >> 1) & 3)) << 4);
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) wr[j] = W + (long)min(n0 + 16 * j + r, N - 1) * ldw;
    struct Piece { gfloatx4_t x[TASKS][2], w[TN][2]; } p0, p1;
    const auto fetch = [&](const float* row, int k, gfloatx4_t (&v)[2]) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            if (VEC) v[c] = *(const gfloatx4_t*)(row + min(k + 16 * c, K - 4));
            else v[c] = f32_piece<false>(row, k + 16 * c, K);
        }
    };
    const auto fetch_x = [&](Piece& p, int k) {
#pragma unroll
        for (int i = 0; i < TASKS; ++i) fetch(xr[i], k + 4 * chunk, p.x[i]);
    };
    const auto fetch_w = [&](Piece& p, int k) {
#pragma unroll
        for (int j = 0; j < TN; ++j) fetch(wr[j], k + 4 * g, p.w[j]);
    };
    uint32_t lost = 0;
    const auto stage = [&](Piece& p, int k, int buf) {
#pragma unroll
        for (int i = 0; i < TASKS; ++i) {
            // beyond the last column X's are zeros, so that W's need not be: a clamped load's stand there, and what is not finite
            // among them is not finite in the row either
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (VEC) p.x[i][c][e] = k + 4 * chunk + 16 * c < K ? p.x[i][c][e] : 0.f;
            const Split8 x = f32_split(p.x[i][0], p.x[i][1], lost);
#pragma unroll
            for (int c = 0; c < 3; ++c) *(gbf16x8_t*)(lds + buf + c * PLANE + place[i]) = x.part[c];
        }
    };
    gfloatx4_t acc[TN][TM];
    const auto start = [&]() {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int i = 0; i < TM; ++i) acc[j][i] = gfloatx4_t{0.f, 0.f, 0.f, 0.f};
    };
    start();
    const int per = f32_share(K);
    int shares = 0, left = per;
    const int at = r * 64 + ((g ^ ((r >> 1) & 3)) << 4);
    // p: piece k (its rows of X in lds[buf]); q: piece k + 32, whose rows go to the other buffer
    const auto step = [&](Piece& p, Piece& q, int k, int buf) {
        __syncthreads();
        gbf16x8_t x[3][TM];
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int i = 0; i < TM; ++i) x[c][i] = *(const gbf16x8_t*)(lds + buf + c * PLANE + at + i * 1024);
        fetch_x(p, k + 64);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            gfloatx4_t (&v)[2] = AHEAD ? p.w[j] : p0.w[j];
            const Split8 w = f32_split(v[0], v[1], lost);
            fetch(wr[j], k + (AHEAD ? 64 : 32) + 4 * g, v);
            f32_multiply<TM>([&](int c, int i) { return x[c][i]; }, w, acc[j]);
        }
        if (--left == 0 && k + 32 < K) {                     // (the last share stays in registers)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    gfloatx4_t& sum = total[j * TM + i][threadIdx.x];
                    sum = shares ? sum + acc[j][i] : acc[j][i];
                }
            start();
            ++shares;
            left = per;
        }
        stage(q, k + 32, BUF - buf);
    };
    fetch_x(p0, 0);
    fetch_w(p0, 0);
    fetch_x(p1, 32);
    if (AHEAD) fetch_w(p1, 32);
    stage(p0, 0, 0);
    int k = 0;
    for (; k + 32 < K; k += 64) {
        step(p0, p1, k, 0);
        step(p1, p0, k + 32, BUF);
    }
    if (k < K) step(p0, p1, k, 0);
    const bool odd = __syncthreads_or(lost & 0xffff);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const gfloatx4_t sum = shares ? total[j * TM + i][threadIdx.x] + acc[j][i] : acc[j][i];
            f32_finish_tile<VEC>(sum, X, ldx, W, ldw, Y, ldy, M, N, K, alpha, m0 + 16 * i, n0 + 16 * j, odd);
        }
}

template <int TM, int TN, int NW, bool VEC>
__global__ __launch_bounds__(NW * 64, 2) void gemm_f32_shares_kernel(
    const float* __restrict__ X, long ldx, const float* __restrict__ W, long ldw, float* __restrict__ Y, long ldy, int M, int N,
    int K, float alpha, int m_tiles, int tiles) {
    constexpr int PER = (TM * TN + NW - 1) / NW, ROWS = 16 * (TM + TN), LOADS = ROWS / 8;
    constexpr int REGION = (TM + TN) * 2 > TM * TN ? (TM + TN) * 128 : TM * TN * 64;       // a wavefront's, in 16 bytes
    __shared__ gfloatx4_t lds[NW * REGION];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    gfloatx4_t* own = lds + wave * REGION;
    const int t = tile_of_workgroup(blockIdx.x, tiles);
    const int m0 = t % m_tiles * 16 * TM, n0 = t / m_tiles * 16 * TN;
    // a piece: 32 columns of the tile's rows, X's before W's; a load brings 8 rows, 8 lanes a row
    const int chunk = lane & 7, row8 = lane >> 3;
    const float *xb = X + (long)m0 * ldx, *wb = W + (long)n0 * ldw;
    uint32_t off[LOADS];                                                                   // floats from there
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int row = 8 * i + row8;
        off[i] = i < 2 * TM ? min(row, M - 1 - m0) * (uint32_t)ldx : min(row - 16 * TM, N - 1 - n0) * (uint32_t)ldw;
    }
    gfloatx4_t next[LOADS];
    const auto fetch = [&](int k0) {
        const int k = VEC ? min(k0 + 4 * chunk, K - 4) : k0 + 4 * chunk;                   // beyond the end: cleared below
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const float* base = i < 2 * TM ? xb : wb;
            if (VEC) next[i] = *(const gfloatx4_t*)(base + (off[i] + (uint32_t)k));
            else next[i] = f32_piece<false>(base + off[i], k, K);
        }
    };
    gfloatx4_t acc[TN][TM];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) acc[j][i] = gfloatx4_t{0.f, 0.f, 0.f, 0.f};
    const int place = row8 * 8 + (chunk ^ row8), at0 = r * 8 + (g ^ (r & 7)), at1 = at0 ^ 4;
    uint32_t lost = 0;
    static_assert(NW == 8, "a share a wavefront");
    const int per = f32_share(K) * 32, end = min((wave + 1) * per, K);
    fetch(wave * per);
    for (int k = wave * per; k < end; k += 32) {
        if (VEC && k + 32 > K && k + 4 * chunk >= K) {
#pragma unroll
            for (int i = 0; i < LOADS; ++i) next[i] = gfloatx4_t{0.f, 0.f, 0.f, 0.f};
        }
        // (a wavefront's LDS accesses keep their order: no barrier)
#pragma unroll
        for (int i = 0; i < LOADS; ++i) own[64 * i + place] = next[i];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        fetch(k + 32);
        Split8 x[TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) x[i] = f32_split(own[128 * i + at0], own[128 * i + at1], lost);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const Split8 w = f32_split(own[128 * (TM + j) + at0], own[128 * (TM + j) + at1], lost);
            f32_multiply<TM>([&](int c, int i) { return x[i].part[c]; }, w, acc[j]);
        }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) own[(i * TN + j) * 64 + lane] = acc[j][i];
    const bool odd = __syncthreads_or(lost & 0xffff);
#pragma unroll
    for (int f = 0; f < PER; ++f) {
        const int tile = wave * PER + f, i = tile / TN, j = tile % TN;
        if (tile >= TM * TN) break;
        gfloatx4_t sum = lds[tile * 64 + lane];
#pragma unroll
        for (int w = 1; w < NW; ++w) sum += lds[w * REGION + tile * 64 + lane];
        f32_finish_tile<VEC>(sum, X, ldx, W, ldw, Y, ldy, M, N, K, alpha, m0 + 16 * i, n0 + 16 * j, odd);
    }
}

// The same for at most 16 rows (decode steps), where the weight's bytes are the bound: a workgroup owns 16 outputs a row
// over all of K, its NW wavefronts take 16 columns each in turn, operands straight from memory, and add up through LDS.
template <int NW, bool VEC>
__global__ __launch_bounds__(NW * 64) void gemm_f32_rows_kernel(const float* __restrict__ X, long ldx,
                                                                const float* __restrict__ W, long ldw,
                                                                float* __restrict__ Y, long ldy, int M, int N, int K,
                                                                float alpha) {
    __shared__ gfloatx4_t part[NW][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16;
    const float* xr = X + (long)min(r, M - 1) * ldx;
    const float* wr = W + (long)min(n0 + r, N - 1) * ldw;
    gfloatx4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int k = wave * 16 + 4 * g; k < K + 4 * g; k += NW * 16) {
        const gfloatx4_t a = f32_piece<VEC>(xr, k, K), b = f32_piece<VEC>(wr, k, K);
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b[s], acc, 0, 0, 0);
    }
    part[wave][lane] = acc;
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int w = 1; w < NW; ++w) acc += part[w][lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int m = 4 * g + e;
            if (m < M && n0 + r < N) Y[(long)m * ldy + n0 + r] = alpha * acc[e];
        }
    }
}

template <bool VEC>
static void gemm_f32_launch(const float* X, long ldx, const float* W, long ldw, float* Y, long ldy, int M, int N, int K,
                            float alpha, hipStream_t stream) {
    const auto up = [](int a, int b) { return (a + b - 1) / b; };
    // Up to 16 rows the weight's bytes bound the product: every workgroup takes 16 outputs over all of K (1 x 1,024 x
    // 4,096: 12 us, 43 us in tiles of 32 x 32).  Beyond 32,768 outputs there are tiles enough, and the kernels for
    // more rows read x once for 32 outputs instead of 16 (16 x 73,448 x 1,024: 66 against 83 us).
    if (M <= 16 && N <= 32768) {
        gemm_f32_rows_kernel<16, VEC><<<up(N, 16), 1024, 0, stream>>>(X, ldx, W, ldw, Y, ldy, M, N, K, alpha);
        return;
    }
    // (few columns, up to two pieces: 523 x 8,192 x 48 11.2 us, 13.9 in three parts; 2,048 x 4,096 x 32 12.7, 16.4; 523 x 1,024 x 32 6.8, 7.2)
    if (K < 64) {
        gemm_f32_mfma_kernel<VEC><<<dim3(up(N, 64), up(M, 64)), 256, 0, stream>>>(X, ldx, W, ldw, Y, ldy, M, N, K, alpha);
        return;
    }
    // Columns shared out while the tiles are at most one a CU: the smallest tile for which that holds (its wavefronts' pieces cost
    // the least).  Beyond, 64 rows by as many outputs as still leave one and a half workgroups a CU, which then overlap (tiles of
    // 64 / 128 / 192 outputs: 523 x 8,192 x 1,024 88/98/87, 700 x 8,192 x 1,024 107/101/93, 2,048 x 4,096 x 4,096 549/486/518).
    // (up to 32 rows of very many outputs: the weight's bytes are the bound, 32 x 73,448 x 1,024 70 us in the smallest tile, 86 in 64 rows)
    const int few = N > 32768 ? 32 : 0;
    const bool near = 80 * (ldx > ldw ? ldx : ldw) < (1L << 32);      // (a tile's rows are within reach of 32-bit offsets)
#define SHARES(TM, TN)                                                                                                   \
    if (near && (up(M, 16 * TM) * (long)up(N, 16 * TN) <= 256 || M <= few)) {                                            \
        const int tiles = up(M, 16 * TM) * up(N, 16 * TN);                                                               \
        gemm_f32_shares_kernel<TM, TN, 8, VEC><<<tiles, 512, 0, stream>>>(X, ldx, W, ldw, Y, ldy, M, N, K, alpha, up(M, 16 * TM), tiles); \
        return;                                                                                                          \
    }
    SHARES(2, 2);
    SHARES(2, 4);
    SHARES(5, 2);
    SHARES(3, 4);
    SHARES(4, 4);
#undef SHARES
#define SPLIT(TN)                                                                                                        \
    if (TN == 1 || up(M, 64) * (long)up(N, 64 * TN) >= 384) {                                                            \
        const int tiles = up(M, 64) * up(N, 64 * TN);                                                                    \
        gemm_f32_split_kernel<4, TN, VEC><<<tiles, 256, 0, stream>>>(X, ldx, W, ldw, Y, ldy, M, N, K, alpha, up(M, 64), tiles); \
        return;                                                                                                          \
    }
    SPLIT(3);
    SPLIT(2);
    SPLIT(1);
#undef SPLIT
}

extern "C" const char* cpmcu_gemm_nt_plain(const void* X, long ldx, const void* W, long ldw, void* Y, long ldy,
                                           int in_dtype, int out_dtype, int M, int N, int K, float alpha,
                                           hipStream_t stream) {
    CPMCU_REQUIRE(M > 0 && N > 0 && K > 0, "gemm: empty shape M=%d N=%d K=%d", M, N, K);
    CPMCU_REQUIRE(ldx >= K && ldw >= K && ldy >= N, "gemm: leading dimensions %ld %ld %ld too small for K=%d N=%d",
                  ldx, ldw, ldy, K, N);
    dim3 grid((N + GT_BN - 1) / GT_BN, (M + GT_BM - 1) / GT_BM);
    CPMCU_REQUIRE(grid.y <= 65535, "gemm: M=%d too large for one launch", M);
    if (in_dtype == CPMCU_F32 && out_dtype == CPMCU_F32) {
        const bool vec = K % 4 == 0 && ldx % 4 == 0 && ldw % 4 == 0 && (uintptr_t)X % 16 == 0 && (uintptr_t)W % 16 == 0;
        const float *x = (const float*)X, *w = (const float*)W;
        if (vec) gemm_f32_launch<true>(x, ldx, w, ldw, (float*)Y, ldy, M, N, K, alpha, stream);
        else gemm_f32_launch<false>(x, ldx, w, ldw, (float*)Y, ldy, M, N, K, alpha, stream);
        CPMCU_LAUNCH_CHECK("gemm_nt_plain");
        return nullptr;
    }
#define LAUNCH(T, OT)                                                                                     \
    gemm_tiled_kernel<T, T, OT><<<grid, 256, 0, stream>>>((const T*)X, ldx, (const T*)W, ldw, (OT*)Y, ldy, \
                                                          M, N, K, alpha)
    if (in_dtype == CPMCU_BF16 && out_dtype == CPMCU_BF16) LAUNCH(bf16_t, bf16_t);
    else if (in_dtype == CPMCU_BF16 && out_dtype == CPMCU_F32) LAUNCH(bf16_t, float);
    else CPMCU_FAIL("gemm: unsupported dtypes in=%d out=%d", in_dtype, out_dtype);
#undef LAUNCH
    CPMCU_LAUNCH_CHECK("gemm_nt_plain");
    return nullptr;
}

// ---------------------------------------------------------------------------
// The same product head by head: Y[m, h, :] = X[m, h, :] . W[h]^T for H heads with a weight [N, K] each (W is
// [H, N, K]); head h's run of a row starts at h * hsx (X) and h * hsy (Y), so inputs and outputs may be slices
// of wider rows.  With `gate` the rows of head h are multiplied by sigmoid(gate[m * ldg + h]) (an output gate
// of one number a head), or, gate_wide, element by element with sigmoid(gate[m * ldg + h * N + n]).  blockIdx.z is
// the head.
// ---------------------------------------------------------------------------
template <typename XT, typename WT, typename OT>
__global__ __launch_bounds__(256) void gemm_heads_kernel(const XT* __restrict__ X, long ldx, long hsx,
                                                         const WT* __restrict__ W, OT* __restrict__ Y, long ldy,
                                                         long hsy, const XT* __restrict__ gate, long ldg,
                                                         int gate_wide, int M, int N, int K) {
    __shared__ float xs[GT_BK][GT_BM + 1];
    __shared__ float ws[GT_BK][GT_BN + 1];
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    const int m0 = blockIdx.y * GT_BM, n0 = blockIdx.x * GT_BN, h = blockIdx.z;
    X += (long)h * hsx;
    Y += (long)h * hsy;
    W += (long)h * N * K;
    float acc[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += GT_BK) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = threadIdx.x + i * 256;
            const int r = e / GT_BK, kk = e % GT_BK;
            const int k = k0 + kk;
            xs[kk][r] = (m0 + r < M && k < K) ? to_f32(X[(long)(m0 + r) * ldx + k]) : 0.f;
            ws[kk][r] = (n0 + r < N && k < K) ? to_f32(W[(long)(n0 + r) * K + k]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < GT_BK; ++kk) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = xs[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = ws[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] += a[i] * b[j];
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + ty * 4 + i;
        if (m >= M) continue;
        float gs = 1.f;
        if (gate && !gate_wide) gs = 1.0f / (1.0f + expf(-to_f32(gate[(long)m * ldg + h])));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + tx * 4 + j;
            if (n >= N) continue;
            if (gate_wide) gs = 1.0f / (1.0f + expf(-to_f32(gate[(long)m * ldg + (long)h * N + n])));
            Y[(long)m * ldy + n] = from_f32<OT>(gs * acc[i][j]);
        }
    }
}

extern "C" const char* cpmcu_gemm_nt_heads(const void* X, long ldx, long hsx, const void* W, void* Y, long ldy, long hsy,
                                           const void* gate, long ldg, int gate_wide, int in_dtype, int out_dtype, int M,
                                           int H, int N, int K, hipStream_t stream) {
    CPMCU_REQUIRE(M > 0 && H > 0 && N > 0 && K > 0, "gemm_heads: empty shape M=%d heads=%d N=%d K=%d", M, H, N, K);
    CPMCU_REQUIRE(ldx >= (H - 1) * hsx + K && ldy >= (H - 1) * hsy + N && (!gate || ldg >= (gate_wide ? (long)H * N : H)),
                  "gemm_heads: rows of %ld / %ld elements cannot hold %d heads", ldx, ldy, H);
    dim3 grid((N + GT_BN - 1) / GT_BN, (M + GT_BM - 1) / GT_BM, H);
    CPMCU_REQUIRE(grid.y <= 65535 && H <= 65535, "gemm_heads: M=%d or heads=%d too large for one launch", M, H);
#define LAUNCH(T, OT)                                                                                          \
    gemm_heads_kernel<T, T, OT><<<grid, 256, 0, stream>>>((const T*)X, ldx, hsx, (const T*)W, (OT*)Y, ldy, hsy, \
                                                          (const T*)gate, ldg, gate && gate_wide, M, N, K)
    if (in_dtype == CPMCU_F32 && out_dtype == CPMCU_F32) LAUNCH(float, float);
    else if (in_dtype == CPMCU_BF16 && out_dtype == CPMCU_BF16) LAUNCH(bf16_t, bf16_t);
    else if (in_dtype == CPMCU_BF16 && out_dtype == CPMCU_F32) LAUNCH(bf16_t, float);
    else CPMCU_FAIL("gemm_heads: unsupported dtypes in=%d out=%d", in_dtype, out_dtype);
#undef LAUNCH
    CPMCU_LAUNCH_CHECK("gemm_nt_heads");
    return nullptr;
}

// The product head by head in bf16 on the matrix cores (v_mfma_f32_16x16x32_bf16).  A workgroup of 4
// wavefronts owns, for one head, 64 rows x 64 columns (WM = 4: a wavefront a tile of 16 rows, NT = 4 tiles of 16
// columns) or 16 rows x 64 columns (WM = 1, steps of few rows: a wavefront 16 columns, NT = 1, so that a head's weight
// is spread over as many wavefronts as it has strips of 16 columns).
// Operands come straight from memory, 16 bytes a lane: lane (r, g) of a tile reads row r, columns k0 + 8g .. + 8,
// of X and of W alike (W [N, K] row-major is the transposed operand as it lies).  K is a multiple of 8 and
// rows start on 16-byte borders (the launcher checks).  No load stands in a branch: rows and columns beyond the end
// repeat the last one (their results are not written), features beyond K read the step's first ones and are zeroed.
typedef __bf16 hbf16x8_t __attribute__((ext_vector_type(8)));
typedef float hfloatx4_t __attribute__((ext_vector_type(4)));

template <int WM, int NT>
__global__ __launch_bounds__(256) void gemm_heads_mfma_kernel(const bf16_t* __restrict__ X, long ldx, long hsx,
                                                              const bf16_t* __restrict__ W, bf16_t* __restrict__ Y,
                                                              long ldy, long hsy, const bf16_t* __restrict__ gate,
                                                              long ldg, int gate_wide, int M, int N, int K) {
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int h = blockIdx.z;
    const int m0 = blockIdx.y * (WM == 4 ? 64 : 16) + (WM == 4 ? wave * 16 : 0);
    const int n0 = blockIdx.x * 64 + (WM == 4 ? 0 : wave * 16 * NT);
    if (m0 >= M || n0 >= N) return;
    const bf16_t* xp = X + (long)h * hsx + (long)min(m0 + r, M - 1) * ldx;
    const bf16_t* wp = W + (long)h * N * K;
    hfloatx4_t acc[NT];
    long wrow[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        acc[j] = hfloatx4_t{0.f, 0.f, 0.f, 0.f};
        wrow[j] = (long)min(n0 + 16 * j + r, N - 1) * K;
    }
    // the gate's numbers of this lane's results are asked for before the product's operands
    float gs[4][NT];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            gs[i][j] = 0.f;
            if (gate) {
                const long m = min(m0 + 4 * g + i, M - 1);
                gs[i][j] = to_f32(gate[m * ldg + (gate_wide ? (long)h * N + min(n0 + 16 * j + r, N - 1) : h)]);
            }
        }
    const hbf16x8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll (NT == 1 ? 8 : 2)
    for (int k0 = 0; k0 < K; k0 += 32) {
        const bool k_ok = k0 + g * 8 < K;
        const int kk = k0 + (k_ok ? g * 8 : 0);
        hbf16x8_t a = *(const hbf16x8_t*)(xp + kk);
        a = k_ok ? a : zero8;
        hbf16x8_t b[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) b[j] = *(const hbf16x8_t*)(wp + wrow[j] + kk);
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, k_ok ? b[j] : zero8, acc[j], 0, 0, 0);
    }
    // lane (column r, g): acc[j][i] is the result of row m0 + 4g + i, column n0 + 16j + r
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + 4 * g + i;
        if (m >= M) continue;
        bf16_t* yr = Y + (long)h * hsy + (long)m * ldy;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int n = n0 + 16 * j + r;
            if (n < N) yr[n] = f32_to_bf16(gate ? acc[j][i] / (1.0f + expf(-gs[i][j])) : acc[j][i]);
        }
    }
}

// The same for many rows: 128 rows x 128 columns of a head a workgroup, a wavefront 64 x 64, pieces of 64 columns of both
// operands through two LDS buffers with the next piece on its way to registers.  With operands straight from memory every
// wavefront fetched rows and weights for itself, 16 bytes of a row an access, and the address unit was the bound (105
// TFLOP/s): 2,048 rows, 32 heads, 128 features to 512 columns 88 -> 63 us, 512 to 128 88 -> 31 us.  A piece's row is 8 chunks of 16 bytes,
// chunk c of row r at place c ^ (r % 8), so that 8 neighbouring lanes read all banks.  W takes the first operand's place: a
// lane then holds 4 neighbouring columns of a row of Y and writes them together.
typedef unsigned hu32x4_t __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void gemm_heads_tile_kernel(const bf16_t* __restrict__ X, long ldx, long hsx,
                                                              const bf16_t* __restrict__ W, bf16_t* __restrict__ Y,
                                                              long ldy, long hsy, const bf16_t* __restrict__ gate,
                                                              long ldg, int gate_wide, int M, int N, int K, int pairs) {
    __shared__ hu32x4_t lds[2][256 * 8];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int h = blockIdx.z, m0 = blockIdx.y * 128, n0 = blockIdx.x * 128;
    const int chunk = threadIdx.x & 7, lrow = threadIdx.x >> 3;
    const int place = lrow * 8 + (chunk ^ (lrow & 7));
    const bf16_t *xp[4], *wp[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        xp[i] = X + (long)h * hsx + (long)min(m0 + lrow + 32 * i, M - 1) * ldx + chunk * 8;
        wp[i] = W + ((long)h * N + min(n0 + lrow + 32 * i, N - 1)) * K + chunk * 8;
    }
    hu32x4_t nx[4], nw[4];
    auto fetch = [&](int k0) {
        const int k = min(k0, K - 8 - chunk * 8);                  // beyond the row's end: its last columns, zeroed below
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            nx[i] = *(const hu32x4_t*)(xp[i] + k);
            nw[i] = *(const hu32x4_t*)(wp[i] + k);
        }
    };
    hfloatx4_t acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = hfloatx4_t{0.f, 0.f, 0.f, 0.f};
    const int mw = (wave & 1) * 64, nw0 = (wave >> 1) * 64;
    fetch(0);
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += 64, buf ^= 1) {
        if (k0 + chunk * 8 >= K) {                                 // K % 8 == 0: the whole chunk lies beyond the end
#pragma unroll
            for (int i = 0; i < 4; ++i) nx[i] = nw[i] = hu32x4_t{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            lds[buf][256 * i + place] = nx[i];
            lds[buf][1024 + 256 * i + place] = nw[i];
        }
        __syncthreads();
        if (k0 + 64 < K) fetch(k0 + 64);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int at = (kk * 4 + g) ^ (r & 7);
            hbf16x8_t x[4], w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[i] = *(const hbf16x8_t*)&lds[buf][(mw + 16 * i + r) * 8 + at];
                w[i] = *(const hbf16x8_t*)&lds[buf][1024 + (nw0 + 16 * i + r) * 8 + at];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j], x[i], acc[i][j], 0, 0, 0);
        }
    }
    // lane (row r, g): acc[i][j][e] is row m0 + mw + 16 i + r, column n0 + nw0 + 16 j + 4 g + e
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + mw + 16 * i + r;
        if (m >= M) continue;
        const float one = gate && !gate_wide ? to_f32(gate[(long)m * ldg + h]) : 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + nw0 + 16 * j + 4 * g;
            if (n >= N) continue;
            bf16_t o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = acc[i][j][e];
                if (gate) v /= 1.0f + expf(-(gate_wide ? to_f32(gate[(long)m * ldg + (long)h * N + min(n + e, N - 1)]) : one));
                o[e] = f32_to_bf16(v);
            }
            bf16_t* to = Y + (long)h * hsy + (long)m * ldy + n;
            if (pairs && n + 4 <= N) {                             // rows and heads of Y start on 8-byte borders
                *(uint2*)to = make_uint2((uint32_t)o[0].v | (uint32_t)o[1].v << 16, (uint32_t)o[2].v | (uint32_t)o[3].v << 16);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) to[e] = o[e];
            }
        }
    }
}

// Whether tiles of 128 x 128 are the faster ones: where there is one for every CU, features enough to pay for the two
// barriers a piece, and rows and columns that fill them.  What fills them is how many 64 x 64 tiles they replace, four
// each at most.  Measured (us, tiles of 64 / of 128; heads, rows: columns x features):
//   4       256, 128: 128 x 128 15.5/10.6   64, 512: 128 x 64 9.7/9.8   16, 2,048: 512 x 128 43/25   32, 2,048: 512 x 32 28/37
//   3       256, 65: 192 x 256 30/15   64, 160: 512 x 128 20.6/14.5   128, 160: 256 x 64 13.2/11.2   256, 160: 512 x 64 34/39
//           with 256 tiles: 32, 160: 512 x 128 10.2/10.6   128, 65: 136 x 128 8.1/9.9   128, 128: 192 x 256 20/13
//   2, 1.5  256, 64: 128 x 512 24/17   256, 65: 64 x 512 23/15   256, 64: 192 x 256 20/15   256, 24: 192 x 256 11.2/11.0
//           256, 17: 192 x 256 10.6/10.9   256, 64: 128 x 128 9.0/9.8   128, 136: 136 x 128 14/13
//   1       256, 64: 64 x 512 13.5/14.7   256, 17: 8 x 8 3.7/4.3
static bool heads_in_tiles(int M, int H, int N, int K) {
    const auto up = [](int a, int b) { return (long)((a + b - 1) / b); };
    const long tiles = up(M, 128) * up(N, 128) * H, small = up(M, 64) * up(N, 64) * H;
    if (tiles < 256 || M < 24 || N < 64 || K < 64) return false;
    if (small == 4 * tiles) return true;
    if (K >= 256) return 2 * small >= 3 * tiles;
    return small >= 3 * tiles && tiles >= 512 && (K >= 128 || tiles < 1024);
}

extern "C" const char* cpmcu_gemm_nt_heads_mfma(const void* X, long ldx, long hsx, const void* W, void* Y, long ldy,
                                                long hsy, const void* gate, long ldg, int gate_wide, int M, int H, int N,
                                                int K, hipStream_t stream) {
    CPMCU_REQUIRE(M > 0 && H > 0 && N > 0 && K > 0, "gemm_heads_mfma: empty shape M=%d heads=%d N=%d K=%d", M, H, N, K);
    CPMCU_REQUIRE(K % 8 == 0 && ldx % 8 == 0 && hsx % 8 == 0 && ((uintptr_t)X % 16 == 0) && ((uintptr_t)W % 16 == 0),
                  "gemm_heads_mfma: K, the row stride and the head stride of X must be multiples of 8 elements and "
                  "the operands start on 16-byte borders (K=%d, %ld, %ld)", K, ldx, hsx);
    CPMCU_REQUIRE(ldx >= (H - 1) * hsx + K && ldy >= (H - 1) * hsy + N && (!gate || ldg >= (gate_wide ? (long)H * N : H)),
                  "gemm_heads_mfma: rows of %ld / %ld elements cannot hold %d heads", ldx, ldy, H);
    CPMCU_REQUIRE(H <= 65535, "gemm_heads_mfma: %d heads exceed the launch grid", H);
    if (M <= 16) {
        dim3 grid((N + 63) / 64, 1, H);
        gemm_heads_mfma_kernel<1, 1><<<grid, 256, 0, stream>>>((const bf16_t*)X, ldx, hsx, (const bf16_t*)W, (bf16_t*)Y, ldy,
                                                               hsy, (const bf16_t*)gate, ldg, gate && gate_wide, M, N, K);
    } else if (heads_in_tiles(M, H, N, K)) {
        dim3 grid((N + 127) / 128, (M + 127) / 128, H);
        CPMCU_REQUIRE(grid.y <= 65535, "gemm_heads_mfma: M=%d too large for one launch", M);
        const int pairs = ldy % 4 == 0 && hsy % 4 == 0 && (uintptr_t)Y % 8 == 0;
        gemm_heads_tile_kernel<<<grid, 256, 0, stream>>>((const bf16_t*)X, ldx, hsx, (const bf16_t*)W, (bf16_t*)Y, ldy, hsy,
                                                         (const bf16_t*)gate, ldg, gate && gate_wide, M, N, K, pairs);
    } else {
        dim3 grid((N + 63) / 64, (M + 63) / 64, H);
        CPMCU_REQUIRE(grid.y <= 65535, "gemm_heads_mfma: M=%d too large for one launch", M);
        gemm_heads_mfma_kernel<4, 4><<<grid, 256, 0, stream>>>((const bf16_t*)X, ldx, hsx, (const bf16_t*)W, (bf16_t*)Y, ldy,
                                                               hsy, (const bf16_t*)gate, ldg, gate && gate_wide, M, N, K);
    }
    CPMCU_LAUNCH_CHECK("gemm_nt_heads_mfma");
    return nullptr;
}

// ===========================================================================
// Skinny product for decode steps (bf16, at most 64 rows of X):
//   Y[m,N] = alpha * X[m,K] . W[N,K]^T
// The step is bound by reading W once from HBM, so W streams from global memory
// straight into MFMA operand registers (v_mfma_f32_16x16x32_bf16: 16 rows of W
// by 32 of K an instruction), four K-blocks of 128 ahead of their use, while X
// (small, shared by all rows of W) is staged through LDS 512 columns at a time.
// For the i-th MFMA of a K-block of 128 the lane group g = lane/16 holds columns
// [32i + 8g, 32i + 8g + 8) of its row, so the four lanes of a row read 64
// contiguous bytes an instruction; X is read from LDS with the same mapping.
// TILED: W comes re-laid for this kernel (made once when the weights are bound):
// [strip of 16 rows][K-block of 128][MFMA i][lane][8 elements], rows and K padded with
// zeros, so every load instruction of a wavefront reads 1 KiB of consecutive memory and
// a wavefront streams one contiguous region.  Measured on the MI355X this lifts the large
// products from about 4.9 to 5.8-6.1 TB/s (a plain read kernel reaches 6.3).
//   MODE 0: Y (float or bf16) = alpha * product
//   MODE 1: float partial sums of a K-split, part[blockIdx.y][m][N]
//   MODE 2: rows come in pairs (gate j, up I+j): Y[m][j] = act(gate) * up  (bf16; act: SiLU or the tanh form of GELU)
//   MODE 3: Y (bf16) = act(product), a nonlinearity without a gate
// ===========================================================================
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));

#define SK_XC 512            // K columns of X staged at a time
#define SK_XS (SK_XC + 8)    // LDS row stride in elements (16 bytes of padding)

template <int MT, int MODE, typename OT, int SPW, int NW, bool TILED>
__global__ __launch_bounds__(NW * 64) void gemm_skinny_kernel(const bf16_t* __restrict__ X, long ldx,
                                                             const bf16_t* __restrict__ W, long ldw,
                                                             OT* __restrict__ Y, long ldy, int M, int N, int K, int KS,
                                                             float alpha, int I, long part_stride,
                                                             const float* __restrict__ row_ss, int ss_slices,
                                                             float eps, int act, float act_limit) {
    static_assert(MODE != 2 || SPW == 2, "gated output pairs a gate strip with an up strip");
    // whether the x operands are read from LDS a step ahead (below): it pays for 4 tiles of rows in the split and
    // plain products (64 rows, us without/with: q/k/v 17.0/14.3, down 31.0/28.9, head 134/130, o 11.7/12.0), not
    // for the gated product (53.8/55.3) and not for 2 tiles (q/k/v 12.5/11.4 but down 24.4/25.8)
    constexpr bool AHEAD = MT >= 4 && MODE != 2;
    constexpr int NT = NW * 64;
    constexpr int XV = MT * 16 * 64 / NT;     // 16-byte vectors of X a thread stages per chunk
    constexpr int BPW = 4;                    // K-blocks of a chunk
    __shared__ __attribute__((aligned(16))) bf16_t xs[MT * 16 * SK_XS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int k_begin = blockIdx.y * KS;
    const int k_end = min(K, k_begin + KS);
    const int nkb = (k_end - k_begin + 127) / 128;

    // the strips of 16 rows of W this wave owns
    int out_base[SPW];
    const bf16_t* wp[SPW];
    const long nkb_total = (K + 127) / 128;       // K-blocks of a tiled row strip
    const int n_strips = (N + 15) / 16;
    if (MODE == 2) {
        const int p = blockIdx.x * (NW * 16) + wave * 16;
        out_base[0] = out_base[SPW - 1] = p;
        if (TILED) {                              // I is a multiple of 16: up strip = gate strip + I/16
            const long gs = min(p / 16, I / 16 - 1);
            wp[0] = W + gs * nkb_total * 2048 + lane * 8;
            wp[SPW - 1] = W + (gs + I / 16) * nkb_total * 2048 + lane * 8;
        } else {
            const int pr = min(p + r, I - 1);
            wp[0] = W + (long)pr * ldw;
            wp[SPW - 1] = W + ((long)I + pr) * ldw;
        }
    } else {
        const int n0 = blockIdx.x * (NW * SPW * 16) + wave * (SPW * 16);
#pragma unroll
        for (int s = 0; s < SPW; ++s) {
            out_base[s] = n0 + s * 16;
            if (TILED) wp[s] = W + (long)min(n0 / 16 + s, n_strips - 1) * nkb_total * 2048 + lane * 8;
            else wp[s] = W + (long)min(n0 + s * 16 + r, N - 1) * ldw;
        }
    }

    // In the main loop no load stands in a branch: the compiler waits for every load in flight where such a
    // branch ends, and the weights asked for a chunk ahead would have to be there before the chunk's x is stored
    // (that wait cost the 64-row products a trip to memory a chunk).  Only the slice's last chunks (`guard`) ask
    // whether a block or a column exists.
    bf16x8_t a[BPW][SPW][4];                  // a chunk's blocks of the wavefront's strips
    auto load_w = [&](int kb, bf16x8_t (&dst)[SPW][4], const bool guard) {
        if (guard && kb >= nkb) {             // uniform; the block is multiplied by zeros of x or not at all
#pragma unroll
            for (int s = 0; s < SPW; ++s)
#pragma unroll
                for (int i = 0; i < 4; ++i) dst[s][i] = bf16x8_t{0, 0, 0, 0, 0, 0, 0, 0};
            return;
        }
        const int k = k_begin + kb * 128 + g * 8;
#pragma unroll
        for (int s = 0; s < SPW; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (TILED)                    // one 128-block of a strip is 2048 elements: [i][lane][8]
                    dst[s][i] = __builtin_nontemporal_load((const bf16x8_t*)(wp[s] + ((long)(k_begin / 128 + kb) * 4 + i) * 512));
                else                          // columns beyond K repeat the row's last 8 and meet zeros of x
                    dst[s][i] = __builtin_nontemporal_load((const bf16x8_t*)(wp[s] + min(k + i * 32, K - 8)));
            }
    };
    // rows beyond the step repeat its last row (their results are not written); columns beyond the slice are
    // read from the row's end and replaced by zeros when the chunk is stored
    bf16x8_t xr[XV];
    auto load_x = [&](int chunk) {
        const int k0 = k_begin + chunk * SK_XC;
#pragma unroll
        for (int v = 0; v < XV; ++v) {
            const int idx = tid + v * NT;
            const int xrow = idx >> 6, vec = idx & 63;
            xr[v] = *(const bf16x8_t*)(X + (long)min(xrow, M - 1) * ldx + min(k0 + vec * 8, K - 8));
        }
    };
    auto store_x = [&](int chunk, const bool guard) {
        const int k0 = k_begin + chunk * SK_XC;
#pragma unroll
        for (int v = 0; v < XV; ++v) {
            const int idx = tid + v * NT;
            const int xrow = idx >> 6, vec = idx & 63;
            const bf16x8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
            *(bf16x8_t*)(xs + xrow * SK_XS + vec * 8) = (!guard || k0 + vec * 8 < k_end) ? xr[v] : zero;
        }
    };

    floatx4_t acc[SPW][MT];
#pragma unroll
    for (int s = 0; s < SPW; ++s)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[s][t] = floatx4_t{0.f, 0.f, 0.f, 0.f};

    // x first: loads return in the order of their issue, and the loop's first store of x must not wait for more
    // weights than its later ones do (the compiler takes the stricter of the two for all)
    load_x(0);
#pragma unroll
    for (int jj = 0; jj < BPW; ++jj) load_w(min(jj, nkb - 1), a[jj], false);   // beyond a short slice: its last block again
    // X may be x * w of a norm whose row factor is still to come (common.h: row_scales); the loop's first
    // barrier makes rs_s visible
    __shared__ float rs_s[MT * 16];
    if (row_ss) row_scales<NT, MT * 16>(row_ss, ss_slices, M, 1.0f / (float)K, eps, rs_s);
    const int nchunk = (nkb + 3) / 4, nfull = nkb / 4;       // chunks in all, chunks of 4 whole blocks
    // a block's weights are asked for again, a chunk ahead, as soon as the block is multiplied
    auto one_chunk = [&](int c, bf16x8_t (&ap)[BPW][SPW][4], const bool guard) {
        __syncthreads();
        store_x(c, guard);
        __syncthreads();
        if (!guard || c + 1 < nchunk) load_x(c + 1);
        if (!AHEAD) {
#pragma unroll
            for (int jj = 0; jj < BPW; ++jj) {
                const int j = jj;
                // consecutive matrix instructions go to different accumulators (tiles of rows, then strips)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
#pragma unroll
                    for (int t = 0; t < MT; ++t) {
                        const bf16x8_t b = *(const bf16x8_t*)(xs + (t * 16 + r) * SK_XS + j * 128 + g * 8 + i * 32);
#pragma unroll
                        for (int s = 0; s < SPW; ++s)
                            acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ap[jj][s][i], b, acc[s][t], 0, 0, 0);
                    }
                }
                load_w((c + 1) * 4 + j, ap[jj], guard);
            }
            return;
        }
        // the x operands of a step (32 columns) are read from LDS a step ahead of the matrix instructions that use
        // them; with one or two wavefronts a SIMD nothing else hides that latency
        auto read_b = [&](int jj, int i, bf16x8_t (&b)[MT]) {
            const int j = jj;
#pragma unroll
            for (int t = 0; t < MT; ++t) b[t] = *(const bf16x8_t*)(xs + (t * 16 + r) * SK_XS + j * 128 + g * 8 + i * 32);
        };
        bf16x8_t bq[2][MT];
        read_b(0, 0, bq[0]);
#pragma unroll
        for (int jj = 0; jj < BPW; ++jj) {
            const int j = jj;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int step = jj * 4 + i;
                if (step + 1 < BPW * 4) read_b((step + 1) / 4, (step + 1) % 4, bq[(step + 1) & 1]);
#pragma unroll
                for (int t = 0; t < MT; ++t)
#pragma unroll
                    for (int s = 0; s < SPW; ++s)
                        acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ap[jj][s][i], bq[step & 1][t], acc[s][t], 0, 0, 0);
            }
            load_w((c + 1) * 4 + j, ap[jj], guard);
        }
        if (!guard) {
            // the order the scheduler is to keep: x of the next chunk asked for, then step by step the next
            // step's operands read from LDS before this step's matrix instructions, a block's weights asked for
            // again when its last step is through (left alone, the scheduler reads each operand just before its
            // use to save registers)
            __builtin_amdgcn_sched_group_barrier(0x020, XV, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, MT, 0);
#pragma unroll
            for (int step = 0; step < BPW * 4; ++step) {
                if (step + 1 < BPW * 4) __builtin_amdgcn_sched_group_barrier(0x100, MT, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, MT * SPW, 0);
                if (step % 4 == 3) __builtin_amdgcn_sched_group_barrier(0x020, SPW * 4, 0);
            }
        }
    };
    int c0 = 0;
    for (; c0 + 2 <= nfull; ++c0) one_chunk(c0, a, false);   // this chunk, the next x and the blocks asked for are whole
    for (; c0 < nchunk; ++c0) one_chunk(c0, a, true);        // the slice's end
    // lane (r, g) of tile t holds token t*16 + r, rows 4g .. 4g+3 of each strip
    OT* Yp = Y + (MODE == 1 ? (long)blockIdx.y * part_stride : 0);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int tok = t * 16 + r;
        if (tok >= M) continue;
        const float rs_t = row_ss ? rs_s[tok] : 1.0f;
        if (MODE == 2) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int col = out_base[0] + 4 * g + i;
                if (col < I) {
                    float gt = acc[0][t][i] * rs_t, up = acc[SPW - 1][t][i] * rs_t;
                    gate_prepare(gt, up, act, act_limit);
                    Yp[(long)tok * ldy + col] = from_f32<OT>(gate_act(gt, act) * up);
                }
            }
        } else {
#pragma unroll
            for (int s = 0; s < SPW; ++s)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int col = out_base[s] + 4 * g + i;
                    if (col < N) {
                        const float v = alpha * rs_t * acc[s][t][i];
                        Yp[(long)tok * ldy + col] = from_f32<OT>(MODE == 3 ? plain_act(v, act) : v);
                    }
                }
        }
    }
}

// The same for at most 16 rows of X and a tiled weight, a wavefront a workgroup: 16 rows of W over all of K, x straight from L2
// into the operand, PF blocks of 128 columns asked for ahead.  The sums are the kernel's above, in its order, to the last bit.
// Four times the workgroups of the kernel above, which has 96 of them for 6,144 weight rows on 256 CUs, and no barriers.
// Measured in a chain of launches over weights that no cache holds (us at 1 / 8 / 16 rows, above -> here):
//   4,096 x 4,096 13.4/13.9/14.3 -> 8.0/8.4/9.7     6,144 x 4,096 16.3/16.6/17.0 -> 11.0/12.1/14.4     9,280 x 4,096 17.2/18.0/19.0 -> 16.5/17.0/18.8
//   16,384 x 4,096 25.9/26.2/26.7 -> 24.5/24.5/27.5 73,448 x 4,096 101/102/105 -> 92.6/100/122         4,096 x 16,384 45.8/47.1/49.2 -> 24.2/25.3/29.7
//   1,024 x 1,024 4.2/4.4/4.8 -> 2.9/3.2/3.6        8,192 x 1,024 5.1/5.2/5.5 -> 4.5/4.7/5.3           73,448 x 1,024 25.3/26.2 -> 23.8/26.1
//   1,024 x 128 3.0/3.2/3.5 -> 2.5/2.9/3.2          8,192 x 128 3.2/3.3/3.6 -> 2.7/3.0/3.5             4,096 x 2,048 7.1/7.3/7.8 -> 4.7/5.0/5.5
// K is a multiple of 128 (nothing is padded).  ACT: Y (bf16) = act(alpha * product).
template <int PF, typename OT, bool ACT>
__global__ __launch_bounds__(64) void gemm_strip_kernel(const bf16_t* __restrict__ X, long ldx, const bf16_t* __restrict__ W,
                                                        OT* __restrict__ Y, long ldy, int M, int N, int K, float alpha,
                                                        const float* __restrict__ row_ss, int ss_slices, float eps, int act) {
    __shared__ float rs_s[16];
    const int lane = threadIdx.x, r = lane & 15, g = lane >> 4;
    const int nkb = K / 128;
    const bf16_t* wp = W + (long)blockIdx.x * nkb * 2048 + lane * 8;
    const bf16_t* xp = X + (long)min(r, M - 1) * ldx + g * 8;             // rows beyond the step repeat its last one
    bf16x8_t w[PF][4], x[PF][4];
    auto load = [&](int kb, bf16x8_t (&wd)[4], bf16x8_t (&xd)[4]) {       // no branch around a load: the last block again
        const int at = min(kb, nkb - 1);
#pragma unroll
        for (int i = 0; i < 4; ++i) wd[i] = __builtin_nontemporal_load((const bf16x8_t*)(wp + ((long)at * 4 + i) * 512));
#pragma unroll
        for (int i = 0; i < 4; ++i) xd[i] = *(const bf16x8_t*)(xp + at * 128 + i * 32);
    };
    floatx4_t acc = {0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](bf16x8_t (&wd)[4], bf16x8_t (&xd)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wd[i], xd[i], acc, 0, 0, 0);
    };
#pragma unroll
    for (int j = 0; j < PF; ++j) load(j, w[j], x[j]);
    if (row_ss) {
#pragma unroll
        for (int p = 0; p < 4; ++p)                                       // 16 lanes a row, as 256 threads share 16 rows
            row_scale<16>(row_ss, ss_slices, M, 1.0f / (float)K, eps, 4 * p + (lane >> 4), lane & 15, rs_s);
        __syncthreads();
    }
    int kb = 0;
    for (; kb + 2 * PF <= nkb; kb += PF) {
#pragma unroll
        for (int j = 0; j < PF; ++j) {
            multiply(w[j], x[j]);
            load(kb + j + PF, w[j], x[j]);
        }
    }
    for (; kb < nkb; kb += PF) {
#pragma unroll
        for (int j = 0; j < PF; ++j) {
            if (kb + j < nkb) multiply(w[j], x[j]);
            if (kb + j + PF < nkb) load(kb + j + PF, w[j], x[j]);
        }
    }
    // lane (row r of X, g): acc[e] is row 4 g + e of the strip
    if (r >= M) return;
    const float rs = row_ss ? rs_s[r] : 1.0f;
    OT* y = Y + (long)r * ldy + blockIdx.x * 16 + 4 * g;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float v = alpha * rs * acc[e];
        if (blockIdx.x * 16 + 4 * g + e < N) y[e] = from_f32<OT>(ACT ? plain_act(v, act) : v);
    }
}

// out_mode: 0 = Y[m,N] in out_dtype; 1 = float partial sums Y[ksplit][m][N]; 2 = gated (N = 2*I rows of W, Y[m,I] bf16);
// 3 = Y[m,N] bf16 with a nonlinearity without a gate
// row_ss (or null): X is x * w of a norm cut by columns, whose sums of squares [M][ss_slices] these are (a
// slice for every 64 columns after add_norm_columns, for every 16 after proj_add_norm); the output is multiplied
// by rsqrt(sum of the row's slices / K + eps) row by row.
// Workgroups that measured best on the MI355X: 4 wavefronts of one strip each (more, smaller workgroups balance
// better over 256 CUs); for the gated output 2 wavefronts of a gate and an up strip each at every number of rows
// (32,768 x 4,096, us with 4 wavefronts / 2 / two groups of 4 that share the staged x: 17 rows 50.9/46.5/52.9,
// 32 rows 49.5/46.1/52.2, 64 rows 51.9/49.5/52.8).
extern "C" const char* cpmcu_gemm_skinny(const void* X, long ldx, const void* W, long ldw, void* Y, long ldy,
                                         int out_dtype, int out_mode, int M, int N, int K, int ksplit, float alpha,
                                         int tiled, const float* row_ss, int ss_slices, float eps, int act,
                                         float act_limit, hipStream_t stream) {
    CPMCU_REQUIRE(out_mode == 3 ? CPMCU_PLAIN_ACT_KNOWN(act) : CPMCU_ACT_KNOWN(act), "gemm_skinny: unknown nonlinearity %d", act);
    CPMCU_REQUIRE(M > 0 && M <= 64, "gemm_skinny: %d rows (1..64 are taken; more rows belong to the tiled product)", M);
    CPMCU_REQUIRE(N > 0 && K > 0 && K % 8 == 0, "gemm_skinny: K=%d must be a positive multiple of 8 (N=%d)", K, N);
    CPMCU_REQUIRE(ldx % 8 == 0 && ldx >= K && (tiled || (ldw % 8 == 0 && ldw >= K)),
                  "gemm_skinny: leading dimensions %ld %ld must be multiples of 8 and >= K", ldx, ldw);
    CPMCU_REQUIRE(!tiled || out_mode != 2 || (N / 2) % 16 == 0,
                  "gemm_skinny: gated output from tiled weights needs a multiple of 16 gate rows, got %d", N / 2);
    CPMCU_REQUIRE(((uintptr_t)X % 16 == 0) && ((uintptr_t)W % 16 == 0), "gemm_skinny: operands must be 16-byte aligned");
    CPMCU_REQUIRE(ksplit >= 1 && (out_mode == 1 || ksplit == 1), "gemm_skinny: a K-split (%d) needs partial-sum output", ksplit);
    CPMCU_REQUIRE(out_mode != 2 || N % 2 == 0, "gemm_skinny: gated output needs an even number of rows, got %d", N);
    int KS = (K + ksplit - 1) / ksplit;
    KS = (KS + 127) / 128 * 128;
    const int splits = (K + KS - 1) / KS;
    CPMCU_REQUIRE(splits == ksplit, "gemm_skinny: K=%d cannot be cut into %d slices of whole 128-blocks (would be %d)", K, ksplit, splits);
    const int MT = (M + 15) / 16 == 3 ? 4 : (M + 15) / 16;
    const int I = N / 2;
    const long part_stride = (long)M * ldy;
    // One wavefront a strip where that is the faster one: up to 8 rows everywhere, up to 16 where the kernel below leaves CUs
    // without a workgroup of 64 weight rows (beyond, every strip's own copy of x costs more, and with few columns, where a wavefront's
    // strip is short, its start does: 40,000 x 256 6.8 -> 10.3, 32,768 x 512 7.1 -> 7.3, 16,384 x 1,024 7.0 in both).  Blocks in flight:
    // 8 where a CU has few strips, and where so many weights are streamed that only memory counts.
    if (tiled && M <= (N <= 8192 ? 16 : K >= 1024 ? 8 : 0) && (out_mode == 0 || out_mode == 3) && K % 128 == 0 &&
        (out_mode == 3 || out_dtype == CPMCU_F32 || out_dtype == CPMCU_BF16)) {
#define STRIPS(PFv, OT, ACTv)                                                                                        \
    gemm_strip_kernel<PFv, OT, ACTv><<<(N + 15) / 16, 64, 0, stream>>>((const bf16_t*)X, ldx, (const bf16_t*)W, (OT*)Y, ldy, M, \
                                                                       N, K, alpha, row_ss, ss_slices, eps, act)
#define BY_SIZE(OT, ACTv)                                       \
    do {                                                        \
        if (N <= 4096 || N > 32768) STRIPS(8, OT, ACTv);        \
        else STRIPS(4, OT, ACTv);                               \
    } while (0)
        if (out_mode == 3) BY_SIZE(bf16_t, true);
        else if (out_dtype == CPMCU_F32) BY_SIZE(float, false);
        else BY_SIZE(bf16_t, false);
#undef BY_SIZE
#undef STRIPS
        CPMCU_LAUNCH_CHECK("gemm_strips");
        return nullptr;
    }
#define LAUNCH(MTv, MODEv, OT, SPW, NW)                                                                           \
    do {                                                                                                          \
        const int rows_wg = (MODEv == 2) ? NW * 16 : NW * SPW * 16;                                               \
        dim3 grid(((MODEv == 2 ? I : N) + rows_wg - 1) / rows_wg, ksplit);                                        \
        if (tiled)                                                                                                \
            gemm_skinny_kernel<MTv, MODEv, OT, SPW, NW, true><<<grid, NW * 64, 0, stream>>>(                      \
                (const bf16_t*)X, ldx, (const bf16_t*)W, ldw, (OT*)Y, ldy, M, N, K, KS, alpha, I, part_stride,    \
                row_ss, ss_slices, eps, act, act_limit);                                                               \
        else                                                                                                      \
            gemm_skinny_kernel<MTv, MODEv, OT, SPW, NW, false><<<grid, NW * 64, 0, stream>>>(                     \
                (const bf16_t*)X, ldx, (const bf16_t*)W, ldw, (OT*)Y, ldy, M, N, K, KS, alpha, I, part_stride,    \
                row_ss, ss_slices, eps, act, act_limit);                                                               \
    } while (0)
#define BY_MT(MODEv, OT, SPW, NW)                     \
    do {                                              \
        if (MT == 1) LAUNCH(1, MODEv, OT, SPW, NW);   \
        else if (MT == 2) LAUNCH(2, MODEv, OT, SPW, NW); \
        else LAUNCH(4, MODEv, OT, SPW, NW);           \
    } while (0)
    if (out_mode == 0 && out_dtype == CPMCU_F32) BY_MT(0, float, 1, 4);
    else if (out_mode == 0 && out_dtype == CPMCU_BF16) BY_MT(0, bf16_t, 1, 4);
    else if (out_mode == 1) BY_MT(1, float, 1, 4);
    else if (out_mode == 2) BY_MT(2, bf16_t, 2, 2);
    else if (out_mode == 3) BY_MT(3, bf16_t, 1, 4);
    else CPMCU_FAIL("gemm_skinny: unknown output mode %d / dtype %d", out_mode, out_dtype);
#undef BY_MT
#undef LAUNCH
    CPMCU_LAUNCH_CHECK("gemm_skinny");
    return nullptr;
}
