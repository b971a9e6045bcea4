// Products of steps of many tokens (bf16, from 65 rows on): out [M, N] = X [M, K] . W [N, K]^T, summed in float, written in bf16,
// or with the gate's nonlinearity on the float sums (W: gate rows, then up rows), so that neither half is rounded, written and read again.
//
// A workgroup of 4 wavefronts (2 x 2) holds a tile of 32 RT rows by 32 CT weight rows in its accumulators, 256 x 256 at most: 256
// registers a lane, and as many left.  Pieces of 64 columns go from memory to LDS without passing registers (rows of X in SA stages, W in
// SB: HBM is further away), rows of 128 bytes whose 16-byte places are swapped by the row's number, so that 16 lanes that read 16 rows
// meet no bank twice.  A wavefront reads half a piece's operands while it multiplies the half before, a read and at most one fetch
// for two matrix instructions; the workgroup meets once a piece, in the middle.  At most 256 workgroups, one a CU, go from tile to
// tile: the pieces of the next tile are fetched while the last is multiplied and written.  XCD b % 8 has a run of neighbouring
// tiles, rows fastest: 32 at a time that share their operands in its L2.
//
// What bounds it: matrix instructions alone reach 2,090 TFLOP/s with random numbers (2,460 with zeros: that part is the chip's power), this kernel
// with tiles of 256 x 256 in whole rounds 1,310 to 1,400 at 2.0 GHz, the library 1,430 to 1,480; on half the CUs (2,048 x 4,096 x 16,384)
// it takes 2,600 cycles a piece for 2,048 of matrix instructions.  Smaller tiles are bound by what L2 hands a CU (32 bytes a cycle; 256 x 128
// in a prompt's pass 1,200 TFLOP/s, 192 x 128 1,050), a few tiles alone by what one CU is handed of memory (about 37 GB/s of W).
// The matrix instructions are written as asm with the accumulators in place: left to itself the compiler moved them between registers
// in some of these loops (124 moves a piece, 281 -> 434 us).
//
// us, the library -> here, weights that no cache holds:
//   2,048 rows: 22,016 x 4,096 402 -> 276, 4,096 x 4,096 59 to 75 -> 60 to 62, 4,096 x 16,384 223 -> 216, 6,176 x 4,096 89 -> 85;
//     whole rounds of 256 x 256: 16,384 x 4,096 191 -> 203, 32,768 x 4,096 377 -> 407
//   1,500: 22,016 x 4,096 292 -> 218, 4,096 x 11,008 128 -> 123; 1,040: 4,096 x 4,096 45.5 -> 40.3; 347: 22,016 x 4,096 75 -> 63
//   with the gate, against the library's product and the kernel for the nonlinearity (distance from 64 bits 3.1e-3 -> 1.7e-3): 11,008 gates x
//     4,096 at 2,048, 1,500, 1,040, 704 rows 429, 308, 180, 155 -> 285, 224, 174, 136; 2,816 91, 74, 59, 53 -> 78, 72, 51, 40; whole rounds:
//     16,384 at 2,048 397 -> 426, at 1,500 309 -> 331
//
// Where tiles are few for 256 CUs, K is cut into 2 or 4 equal shares if the costs below say so (cpmcu_product_plan; of up to 704 rows most
// products, of more those of long rows): every share's sums go out as floats, product_sum_kernel adds them in their order and applies the
// gate's nonlinearity.  us, the library (with the kernel for the nonlinearity) -> here, in 4 shares unless said otherwise:
//   4,096 x 16,384 at 65, 128, 256, 512, 704 rows 50, 81, 65, 105, 111 -> 42, 51, 53, 72, 92; without shares 116, 145, 142, 139, 126
//     768, 1,024 (2), 1,500 (2), 2,048 (1) 119, 143, 184, 218 -> 94, 123, 172, 222; without 142, 145, 178
//   4,096 x 11,008 38, 58, 49, 74, 81 -> 33, 38, 40, 53, 68; 1,024 (2) 104 -> 85; 2,048 x 16,384 at 1,040, 2,048 (2) 114, 135 -> 74, 117
//   4,096 x 4,096 16, 24, 23, 30 (2), 32 (1) -> 16, 19, 23, 30, 35; 12,288 x 4,096 at 256, 512, 704 (1) 50, 55, 77 -> 44, 54, 64
//   2,816 gates x 4,096 26, 28, 44, 41 (1), 53 (1) -> 18, 20, 28, 39, 40
//   one share: 16,384 gates 67, 68, 82, 117, 171 -> 63, 65, 76, 111, 163; 11,008 gates 48 (2), 51, 68, 95, 155 -> 51, 52, 63, 95, 136
//
// The rule (ops.product_faster) over 1,056 products of 65 to 2,048 rows (23 shapes without a gate, 9 with one; shares as planned), against the library
// for all: without a gate 10% faster in the mean up to 704 rows and 6% beyond, with one 9% and 10%.  How fast the library is goes up and
// down with the sizes (4,096 x 4,096 at 160, 192, 224, 320 rows 27, 33, 22, 26; 4,096 x 16,384 at 1,536, 1,579 183, 393), so it is not always the
// slower one: 96 of the products are more than 2% slower here, half of them by up to 5%, four in five by up to 10%; the worst 128 x 2,048 x 16,384 37 -> 45,
// 1,400 x 32,768 x 4,096 268 -> 320 (with the gate 294 -> 331), 768 and 1,500 rows of 4,096 x 2,816 and 2,048 x 4,096 26, 32 -> 30, 36.
//   Left to the library, us there / here: 11 to 16 million weights beyond 192 rows 17/20 (4,096 x 2,816 at 256), 24/25 (2,816 x 4,096 at 448); from 8,192
//   outputs on, up to 128 rows, 33/39 (16,384 x 4,096 at 65), 30/32 (12,288), though 38/25 (10,240); up to 1,024 outputs 58/80 (8,192 rows of
//   1,024 x 4,096); results below 2.88 million without shares 34/38 (1,280 x 2,048 x 4,096)
//
// 8 and 16 shares are slower than 4 but for 65 and 128 rows of 4,096 x 16,384 (38 and 41 us with 16).
// (reference: every linear layer is its vendor's library's, src/model/linear.cuh:9-37; the gate src/model/activation.cuh:6-18)
#include "product.h"

// (as the kernel that runs behind the library's product forms it)
__device__ inline float gate_fast(float g, int act) { return g * __builtin_amdgcn_rcpf(1.0f + __expf(-gate_arg(g, act))); }

enum { PRODUCT_PLAIN = 0, PRODUCT_GATED = 1, PRODUCT_PARTS = 2 };

template <int RT, int CT, int SA, int SB, int KIND>
__global__ __launch_bounds__(256, 1) void product_kernel(const bf16_t* __restrict__ X, int ldx, const bf16_t* __restrict__ W, int M,
                                                         int N, int K, void* __restrict__ out, int ldo, int mt, int nt, int act, float act_limit, int parts) {
    constexpr int BM = 32 * RT, BN = 32 * CT;
    constexpr int AS = BM * 8, BS = BN * 8, B0 = SA * AS;               // 16-byte chunks
    __shared__ ru32x4_t lds[SA * AS + SB * BS];
    // PRODUCT_PARTS: `parts` equal shares of K, each into a buffer of its own; units run tile by tile, share by share
    const int tiles = mt * nt * (KIND == PRODUCT_PARTS ? parts : 1), per = (tiles + 7) / 8;
    const int first = (blockIdx.x & 7) * per, last = min(first + per, tiles), stride = gridDim.x >> 3;
    int u = first + (blockIdx.x >> 3);
    if (u >= last) return;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int wm = wave & 1, wn = wave >> 1;
    const unsigned base = lds_byte(lds);
    const int pieces = KIND == PRODUCT_PARTS ? K / 64 / parts : K / 64;
    auto share_of = [&](int u) { return KIND == PRODUCT_PARTS ? u / (mt * nt) : 0; };
    unsigned ao[RT], bo[CT];
    auto aim_a = [&](int u) {
        int lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));                                  // (worked out again for every tile: no registers held)
        const int m0 = u % mt * BM, chunk = ((lane & 7) ^ (lane >> 3)) + share_of(u) * pieces * 8;
#pragma unroll
        for (int i = 0; i < RT; ++i) ao[i] = (unsigned)min(m0 + (i * 4 + wave) * 8 + (lane >> 3), M - 1) * (unsigned)(ldx * 2) + chunk * 16;
    };
    auto aim_b = [&](int u) {
        int lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));
        const int n0 = (u - share_of(u) * (mt * nt)) / mt * BN, chunk = ((lane & 7) ^ (lane >> 3)) + share_of(u) * pieces * 8;
#pragma unroll
        for (int i = 0; i < CT; ++i) {
            const int row = (i * 4 + wave) * 8 + (lane >> 3);
            int n;
            if (KIND == PRODUCT_GATED) n = min(n0 / 2 + (row >> 5) * 16 + (row & 15), N - 1) + (row & 16 ? N : 0);
            else n = min(n0 + row, N - 1);
            bo[i] = (unsigned)n * (unsigned)(K * 2) + chunk * 16;
        }
    };
    // what is fetched next: unit, piece, stage
    int ua = u, ub = u, fa = 0, fb = 0, sa = 0, sb = 0;
    const char* xa = (const char*)X;
    const char* wa = (const char*)W;
    auto fetch_a = [&](int i) { bring16_at(xa, ao[i], base + (sa * AS + (i * 4 + wave) * 64) * 16); };
    auto fetch_b = [&](int i) { bring16_at(wa, bo[i], base + (B0 + sb * BS + (i * 4 + wave) * 64) * 16); };
    auto next_a = [&]() {
        sa = sa + 1 == SA ? 0 : sa + 1;
        xa += 128;
        if (++fa == pieces) {
            fa = 0;
            xa = (const char*)X;
            if (ua + stride < last) { ua += stride; aim_a(ua); }
        }
    };
    auto next_b = [&]() {
        sb = sb + 1 == SB ? 0 : sb + 1;
        wa += 128;
        if (++fb == pieces) {
            fb = 0;
            wa = (const char*)W;
            if (ub + stride < last) { ub += stride; aim_b(ub); }
        }
    };
    rfloatx4_t acc[RT][CT];
    rbf16x8_t a[2][RT], b[2][CT];
    const int sw0 = r * 8 + (g ^ (r & 7)), sw1 = r * 8 + ((4 + g) ^ (r & 7));
    auto read_one = [&](int s, int i, const ru32x4_t* as, const ru32x4_t* bs) {      // a0 b0 .. b(CT-1) a1 ..
        const int sw = s ? sw1 : sw0;
        if (i == 0) a[s][0] = *(const rbf16x8_t*)&as[wm * (RT * 128) + sw];
        else if (i <= CT) b[s][i - 1] = *(const rbf16x8_t*)&bs[wn * (CT * 128) + (i - 1) * 128 + sw];
        else a[s][i - CT] = *(const rbf16x8_t*)&as[wm * (RT * 128) + (i - CT) * 128 + sw];
    };
    constexpr int READS = RT + CT, MM = RT * CT, STEPS = MM / 2;
    static_assert(READS <= STEPS && SB >= SA && SA >= 2 && CT % 2 == 0, "");
    auto half = [&](auto S, const ru32x4_t* as, const ru32x4_t* bs) {
        constexpr int s = decltype(S)::value;
#pragma unroll
        for (int i = 0; i < STEPS; ++i) {
            if (i < READS) read_one(s ^ 1, i, as, bs);
            if (s && i * READS / STEPS != (i + 1) * READS / STEPS) {
                const int f = i * READS / STEPS;
                if (f < RT) fetch_a(f);
                else fetch_b(f - RT);
            }
#pragma unroll
            for (int q = 2 * i; q < 2 * i + 2; ++q) {
                const int x = q / CT, y = x & 1 ? CT - 1 - q % CT : q % CT;
                multiply_into(acc[x][y], b[s][y], a[s][x]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);                            // lgkmcnt(0): here it is free, behind the next half's first read not
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    constexpr int STORES = KIND == PRODUCT_GATED ? MM / 4 : KIND == PRODUCT_PLAIN ? MM / 2 : MM;
    constexpr int BEHIND = (SB > SA ? CT : 0) + (SA - 2) * (RT + CT);
    constexpr int BEHIND_STORES = BEHIND + STORES < 63 ? BEHIND + STORES : 63;
    aim_a(u);
    aim_b(u);
#pragma unroll
    for (int i = 0; i < SB - SA; ++i) {
#pragma unroll
        for (int j = 0; j < CT; ++j) fetch_b(j);
        next_b();
    }
#pragma unroll
    for (int i = 0; i < SA; ++i) {
#pragma unroll
        for (int j = 0; j < RT; ++j) fetch_a(j);
        next_a();
#pragma unroll
        for (int j = 0; j < CT; ++j) fetch_b(j);
        next_b();
    }
    landed<BEHIND>();
#pragma unroll
    for (int i = 0; i < READS; ++i) read_one(0, i, lds, lds + B0);
    __builtin_amdgcn_s_waitcnt(0xC07F);
    bool written = false;
    int ra = 0, rb = 0;                                                // the stages of the piece that is multiplied
    for (;; u += stride) {
#pragma unroll
        for (int x = 0; x < RT; ++x)
#pragma unroll
            for (int y = 0; y < CT; ++y) acc[x][y] = rfloatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int x = 0; x < RT; ++x)
#pragma unroll
            for (int y = 0; y < CT; ++y) in_place(acc[x][y]);
        asm volatile("s_nop 7" ::: "memory");
        int p = 0;
        do {
            half(I0(), lds + ra * AS, lds + B0 + rb * BS);
            if (p == 0 && written) landed<BEHIND_STORES>();
            else landed<BEHIND>();
            __builtin_amdgcn_s_waitcnt(0xC07F);
            ra = ra + 1 == SA ? 0 : ra + 1;
            rb = rb + 1 == SB ? 0 : rb + 1;
            half(I1(), lds + ra * AS, lds + B0 + rb * BS);
            next_a();
            next_b();
        } while (++p < pieces);
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");             // the matrix instructions' results are there
        constexpr bool FLOATS = KIND == PRODUCT_PARTS;
        constexpr int EB = FLOATS ? 4 : 2;
        const int m0 = u % mt * BM + wm * 16 * RT, n0 = ((u - share_of(u) * (mt * nt)) / mt * BN + wn * 16 * CT) / (KIND == PRODUCT_GATED ? 2 : 1);
        int er = m0 + r, ec = FLOATS ? n0 + 4 * g : n0 + (g & 1) * 16 + (g >> 1) * 8;
        asm volatile("" : "+v"(er), "+v"(ec));
        void* const to = KIND == PRODUCT_PARTS ? (void*)((float*)out + (long)share_of(u) * M * ldo) : out;
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(to, 0, (int)(((unsigned)(M - 1) * (unsigned)ldo + (unsigned)N) * EB), 0x00020000);
#pragma unroll
        for (int x = 0; x < RT; ++x) {
            const unsigned line = (unsigned)(er + x * 16) * (unsigned)ldo;
            const bool ok = er + x * 16 < M;
            if (FLOATS) {
#pragma unroll
                for (int y = 0; y < CT; ++y) {
                    rfloatx4_t v;
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = sum_of(acc[x][y][i]);
                    const int col = ec + y * 16;
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(ru32x4_t, v), rsrc, ok && col < N ? (line + (unsigned)col) * 4u : 0xFFFFF000u, 0, 0);
                }
            } else {
#pragma unroll
                for (int y = 0; y < CT; y += KIND == PRODUCT_GATED ? 4 : 2) {
                    unsigned d[2][2];
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int i = 0; i < 2; ++i) {
                            float v[2];
#pragma unroll
                            for (int j = 0; j < 2; ++j) {
                                if (KIND == PRODUCT_GATED) {
                                    float gt = sum_of(acc[x][y + 2 * h][2 * i + j]), up = sum_of(acc[x][y + 2 * h + 1][2 * i + j]);
                                    gate_prepare(gt, up, act, act_limit);
                                    v[j] = gate_fast(gt, act) * up;
                                } else {
                                    v[j] = sum_of(acc[x][y + h][2 * i + j]);
                                }
                            }
                            d[h][i] = bf16_pair(v[0], v[1]);
                        }
                    const cpmcu_u32x2_t p0 = __builtin_amdgcn_permlane16_swap(d[0][0], d[1][0], false, false);
                    const cpmcu_u32x2_t p1 = __builtin_amdgcn_permlane16_swap(d[0][1], d[1][1], false, false);
                    const int col = ec + y * (KIND == PRODUCT_GATED ? 8 : 16);
                    __builtin_amdgcn_raw_buffer_store_b128(ru32x4_t{p0.x, p1.x, p0.y, p1.y}, rsrc, ok && col < N ? (line + (unsigned)col) * 2u : 0xFFFFF000u, 0, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (u + stride >= last) break;
        written = true;
    }
    landed<0>();
}

// What a product costs with a tile of 32 RT x 32 CT, in us: the launch, what a round of 256 tiles adds, a piece of 64 columns where few
// CUs are busy and what it takes longer with the share of them that is.  Fitted to 260 products of 65 to 2,048 rows (256 to 33,000
// outputs, 256 to 16,512 columns, every tile): 4 to 10% off in the mean; the tile chosen by it is 0.5% slower than the fastest.
struct ProductTile { int rt, ct; float launch, round, piece, shared; };
#define PRODUCT_TILES(DO)                                                                                                                  \
    DO(8, 8, 2, 3, 3.6f, 4.2f, 0.981f, 0.512f) DO(7, 8, 2, 3, 2.8f, 4.3f, 0.944f, 0.346f) DO(6, 8, 2, 3, 1.9f, 4.9f, 0.796f, 0.287f)       \
    DO(5, 8, 3, 3, 2.1f, 4.1f, 0.740f, 0.241f) DO(4, 8, 3, 3, 2.7f, 2.8f, 0.642f, 0.206f) DO(8, 4, 3, 4, 3.2f, 2.7f, 0.579f, 0.240f)       \
    DO(7, 4, 3, 4, 3.5f, 2.1f, 0.541f, 0.180f) DO(6, 4, 4, 4, 3.3f, 2.1f, 0.493f, 0.176f) DO(5, 4, 4, 5, 3.8f, 1.6f, 0.433f, 0.173f)       \
    DO(4, 4, 4, 5, 3.9f, 1.1f, 0.380f, 0.154f) DO(6, 6, 3, 3, 2.8f, 3.3f, 0.644f, 0.211f) DO(8, 6, 2, 4, 2.0f, 4.8f, 0.783f, 0.288f)       \
    DO(4, 6, 4, 4, 3.2f, 2.1f, 0.529f, 0.156f)
#define PRODUCT_ROW(RT, CT, SA, SB, a, b, c, d) {RT, CT, a, b, c, d},
static const ProductTile PRODUCT_SHAPES[] = {PRODUCT_TILES(PRODUCT_ROW)};
static const int PRODUCT_COUNT = sizeof(PRODUCT_SHAPES) / sizeof(PRODUCT_SHAPES[0]);

// out [M, N] of `parts` buffers [M, rows] of floats, part after part: their sum in bf16, or (gated: rows = 2 N) the gate's nonlinearity on the sums
template <bool GATED>
__global__ __launch_bounds__(256) void product_sum_kernel(const float* __restrict__ part, int parts, int M, int N, bf16_t* __restrict__ out, long ldo,
                                                          int act, float act_limit) {
    const int rows = GATED ? 2 * N : N, cols = N / 8;
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= (long)M * cols) return;
    const int m = (int)(i / cols), c = (int)(i % cols) * 8;
    const float* p = part + (long)m * rows + c;
    rfloatx4_t v[GATED ? 4 : 2] = {};
    for (int s = 0; s < parts; ++s, p += (long)M * rows)
#pragma unroll
        for (int j = 0; j < (GATED ? 4 : 2); ++j) v[j] += *(const rfloatx4_t*)(p + (j & 1) * 4 + (j >> 1) * N);
    if (GATED) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float gt = v[j][e], up = v[GATED ? j + 2 : j][e];
                gate_prepare(gt, up, act, act_limit);
                v[j][e] = gate_fast(gt, act) * up;
            }
    }
    *(ru32x4_t*)(out + m * ldo + c) = ru32x4_t{bf16_pair(v[0][0], v[0][1]), bf16_pair(v[0][2], v[0][3]), bf16_pair(v[1][0], v[1][1]), bf16_pair(v[1][2], v[1][3])};
}

static float product_us(const ProductTile& t, long M, long rows, int K, int parts = 1) {      // rows: of the weight
    const long tiles = ((M + 32 * t.rt - 1) / (32 * t.rt)) * ((rows + 32 * t.ct - 1) / (32 * t.ct)) * parts;
    const long per = (tiles + 7) / 8, rounds = (per + 31) / 32;               // of an XCD with 32 CUs
    return t.launch + rounds * t.round + K / 64 / parts * (rounds * t.piece + per / 32.0f * t.shared);
}
static int product_tile(long M, long rows, int K, bool gated, int parts = 1) {
    int best = -1;
    float least = 0.f;
    for (int i = 0; i < PRODUCT_COUNT; ++i) {
        if (gated && PRODUCT_SHAPES[i].ct % 4) continue;                          // gates and their up rows: 32 weight rows at a time
        const float us = product_us(PRODUCT_SHAPES[i], M, rows, K, parts);
        if (best < 0 || us < least) best = i, least = us;
    }
    return best;
}

// In how many shares of K a product takes least: each share more is M x rows floats that are written and read again (1.4 ps each) and, the
// first of them, a launch.
extern "C" int cpmcu_product_plan(int M, long rows, int K, int gated) {
    int best = 1;
    float least = 0.f;
    for (int parts = 1; parts <= 4; parts *= 2) {
        if (K / 64 % parts || (parts > 1 && (K / 64 / parts < 8 || (double)M * rows * parts >= 1 << 29 || rows * K >= 1L << 30))) continue;
        const int tile = product_tile(M, rows, K, gated && parts == 1, parts);
        const float us = product_us(PRODUCT_SHAPES[tile], M, rows, K, parts) + (parts > 1 ? 3.5f + 1.4e-6f * parts * M * rows : 0.f);
        if (parts == 1 || us < least) best = parts, least = us;
    }
    return best;
}

// out [M, N] = X [M, K] . W^T, W [N, K] and out bf16; PRODUCT_GATED: W [2 N, K] holds gate rows, then up rows, out =
// act(gate) * up in bf16.  tile: one of PRODUCT_TILES, or -1 for the rule's.
extern "C" const char* cpmcu_product(const void* X, long ldx, const void* W, int M, int N, int K, void* out, long ldo, int kind, int act,
                                     float act_limit, int tile, hipStream_t stream) {
    CPMCU_REQUIRE(kind == PRODUCT_PLAIN || kind == PRODUCT_GATED, "product: unknown kind %d", kind);
    CPMCU_REQUIRE(kind != PRODUCT_GATED || CPMCU_ACT_KNOWN(act), "product: unknown nonlinearity %d", act);
    CPMCU_REQUIRE(M > 0 && N > 0 && K > 0 && K % 64 == 0 && N % 8 == 0, "product: K=%d must be a multiple of 64, N=%d of 8", K, N);
    const long rows = (long)N * (kind == PRODUCT_GATED ? 2 : 1);
    CPMCU_REQUIRE((long)M * ldo < (1L << 30) - 4096 && (long)M * ldx < (1L << 31) && rows * K < (1L << 31),
                  "product: %d rows of %ld, %d x %d exceed 32-bit offsets", M, ldx, N, K);
    CPMCU_REQUIRE(ldx % 8 == 0 && ldo % 8 == 0 && ldx >= K && ldo >= N && X && W && out && (uintptr_t)X % 16 == 0 && (uintptr_t)W % 16 == 0 &&
                  (uintptr_t)out % 16 == 0, "product: rows must start on 16-byte borders");
    if (tile < 0) tile = product_tile(M, rows, K, kind == PRODUCT_GATED);
    CPMCU_REQUIRE(tile < PRODUCT_COUNT && (kind != PRODUCT_GATED || PRODUCT_SHAPES[tile].ct % 4 == 0), "product: no tile %d", tile);
    const int rt = PRODUCT_SHAPES[tile].rt, ct = PRODUCT_SHAPES[tile].ct;
    const int mt = (M + 32 * rt - 1) / (32 * rt), nt = (int)((rows + 32 * ct - 1) / (32 * ct));
    const long blocks = ((long)mt * nt + 7) / 8 * 8;
    const unsigned grid = (unsigned)(blocks < 256 ? blocks : 256);
#define PRODUCT_KIND(RT, CT, SA, SB, KINDv)                                                                                                \
    product_kernel<RT, CT, SA, SB, KINDv><<<grid, 256, 0, stream>>>((const bf16_t*)X, (int)ldx, (const bf16_t*)W, M, N, K, out, (int)ldo, mt, nt, \
                                                                    act, act_limit, 1)
#define PRODUCT_LAUNCH(RT, CT, SA, SB, a, b, c, d)                                                                                         \
    if (rt == RT && ct == CT) {                                                                                                            \
        if (kind == PRODUCT_PLAIN) PRODUCT_KIND(RT, CT, SA, SB, PRODUCT_PLAIN);                                                            \
        else if constexpr (CT % 4 == 0) PRODUCT_KIND(RT, CT, SA, SB, PRODUCT_GATED);                                                       \
    }
    PRODUCT_TILES(PRODUCT_LAUNCH)
#undef PRODUCT_LAUNCH
#undef PRODUCT_KIND
    CPMCU_LAUNCH_CHECK("product");
    return nullptr;
}

// The same by shares of K: `parts` partial sums in scratch (parts x M x rows floats, rows 2 N where gated), then their sum; K / 64 in equal shares
// of at least 4 pieces; bf16 results.
extern "C" const char* cpmcu_product_parts(const void* X, long ldx, const void* W, int M, int N, int K, void* out, long ldo, int gated, int act,
                                           float act_limit, float* scratch, int parts, int tile, hipStream_t stream) {
    CPMCU_REQUIRE(!gated || CPMCU_ACT_KNOWN(act), "product_parts: unknown nonlinearity %d", act);
    CPMCU_REQUIRE(M > 0 && N > 0 && K > 0 && K % 64 == 0 && N % 8 == 0, "product_parts: K=%d must be a multiple of 64, N=%d of 8", K, N);
    CPMCU_REQUIRE(parts > 0 && K / 64 % parts == 0 && K / 64 / parts >= 4, "product_parts: %d shares of K=%d", parts, K);
    const int rows = N * (gated ? 2 : 1);
    CPMCU_REQUIRE((long)M * rows * parts < (1L << 29) && (long)M * ldx < (1L << 31) && (long)N * K < (1L << 30),
                  "product_parts: %d rows of %ld, %d x %d exceed 32-bit offsets", M, ldx, N, K);
    CPMCU_REQUIRE(ldx % 8 == 0 && ldo % 8 == 0 && ldx >= K && ldo >= N && X && W && out && scratch && (uintptr_t)X % 16 == 0 && (uintptr_t)W % 16 == 0 &&
                  (uintptr_t)out % 16 == 0 && (uintptr_t)scratch % 16 == 0, "product_parts: rows must start on 16-byte borders");
    if (tile < 0) tile = product_tile(M, rows, K, false, parts);
    CPMCU_REQUIRE(tile < PRODUCT_COUNT, "product_parts: no tile %d", tile);
    const int rt = PRODUCT_SHAPES[tile].rt, ct = PRODUCT_SHAPES[tile].ct;
    const int mt = (M + 32 * rt - 1) / (32 * rt), nt = (rows + 32 * ct - 1) / (32 * ct);
    const long blocks = ((long)mt * nt * parts + 7) / 8 * 8;
    const unsigned grid = (unsigned)(blocks < 256 ? blocks : 256);
#define PRODUCT_LAUNCH(RT, CT, SA, SB, a, b, c, d)                                                                                         \
    if (rt == RT && ct == CT)                                                                                                              \
        product_kernel<RT, CT, SA, SB, PRODUCT_PARTS><<<grid, 256, 0, stream>>>((const bf16_t*)X, (int)ldx, (const bf16_t*)W, M, rows, K, scratch, rows, \
                                                                                mt, nt, 0, 0.f, parts);
    PRODUCT_TILES(PRODUCT_LAUNCH)
#undef PRODUCT_LAUNCH
    CPMCU_LAUNCH_CHECK("product_parts");
    const unsigned sums = (unsigned)(((long)M * (N / 8) + 255) / 256);
    if (gated) product_sum_kernel<true><<<sums, 256, 0, stream>>>(scratch, parts, M, N, (bf16_t*)out, ldo, act, act_limit);
    else product_sum_kernel<false><<<sums, 256, 0, stream>>>(scratch, parts, M, N, (bf16_t*)out, ldo, act, act_limit);
    CPMCU_LAUNCH_CHECK("product_sum");
    return nullptr;
}
