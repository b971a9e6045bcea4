// Products of routed experts of steps that give an expert many rows: the tiles of product.hip, expert by expert.
//
// A workgroup of 4 wavefronts (2 x 2), one a CU, holds up to 224 rows of an expert against 256 of its weight rows (GATED: gate and up
// rows of 128 features) in its accumulators; pieces of 64 columns go from memory to LDS without passing registers, rows in 2 stages,
// weights, past the caches, in 3 (with 256 rows nothing would be left of LDS for the rows' list).  A form of the loop for every 32
// rows of 96 to 224.  256 workgroups go from tile to tile, the pieces of the next tile on their way while the last is multiplied and
// written.  The tasks (expert by expert, weight rows by weight rows, an expert's tiles of rows side by side) are cut into 8 runs, one an
// XCD, whose workgroups take the next one from a counter; a run that has ended helps the run that has most left.  moe_group_kernel
// deals the experts to the runs by their rows, many rows first, so that what runs last is small.
//
// us (64 experts of 4,096 x 1,408 gated, 2,048 tokens with 6 each), tiles of 128 x 128 two a CU -> this, each product standing alone and the whole
// call: even routing 447 + 263 -> 346 + 189, 688 -> 555; uneven (up to 750 rows an expert, half with fewer than 80) 452 + 259 -> 385 + 221, 670 -> 612; a
// router with random weights (one expert of 1,700 rows, half with fewer than 10) 443 + 254 -> 366 + 214, 681 -> 604; with 16 of 80 identity 384 + 221 ->
// 319 + 192, 640 -> 542.  2,112 without a gate 337 + 340 -> 306 + 317.  In a pass of other layers the second product gains less, or nothing
// (Pemalorn's 2,048 tokens 214.5 -> 214).  The gate has the full precision of the other kernels; by the fast exponential and
// reciprocal the first product takes up to 4% less.
// What bounds it (the figures up to the end with the fast gate): even routing moves 1.47 + 0.74 GB of weights, a piece of 32 KB in 1.26 us a CU (6.6 TB/s together) beside
// 1,536 cycles of matrix instructions; with all operands in caches and nothing written 246 + 137 are left.  A tile costs 7 us beside its
// pieces (results 4, the next task and its list 2), the kernel's start 7, and at the end CUs wait for the last: a tenth of the time.
// Taken back: weights through the caches where tiles share them (592 -> 613 for the call, even routing 540 -> 551), runs taken
// from both ends, so that large tiles and small ones meet (594 -> 621, level with a router's load), forms for 96, 160 and 224 rows only (594 ->
// 606), experts in the order of their numbers (first product uneven 354 -> 344, of 1,200 tokens 315 -> 292 with the order).
#include "moe_product.h"
#include "product.h"

template <int KIND>
__global__ __launch_bounds__(256, 1) void moe_product_kernel(const bf16_t* __restrict__ in, int ldi, const bf16_t* __restrict__ w,
                                                             const int* __restrict__ rows, const int* __restrict__ offs,
                                                             const int* __restrict__ tile_expert, const int* __restrict__ n_tiles,
                                                             int* __restrict__ counters, bf16_t* __restrict__ out, int out_rows, int K, int N, unsigned by_top,
                                                             int act, float act_limit) {
    constexpr int CT = 8, SA = 2, SB = 3, MOST = MOE_PRODUCT_ROWS / 32;
    constexpr int AS = MOE_PRODUCT_ROWS * 8, BS = 256 * 8, B0 = SA * AS;   // 16-byte chunks
    constexpr int FEATURES = KIND == MOE_GATED ? 128 : 256;
    constexpr int STORES = 3 * CT / (KIND == MOE_GATED ? 4 : 2);           // of a tile of few rows: no tile has fewer
    __shared__ ru32x4_t lds[SA * AS + SB * BS];
    __shared__ int list[2][256];                                           // the pairs of this tile and of the next
    __shared__ int taken;
    const int nts = (N + FEATURES - 1) / FEATURES;
    const int tasks = *n_tiles * nts;
    const int home = blockIdx.x & 7;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int wm = wave & 1, wn = wave >> 1;
    const unsigned base = lds_byte(lds);
    const int pieces = K / 64;
    // the next task of the home run, then of the run that has most left; -1: none is left.  (Counters only grow: every round of the
    // loop takes a task or has seen one taken.)
    auto take = [&](int i) {                                              // i: what the home run's counter gave
        int per = (tasks + 7) / 8;
        asm volatile("" : "+s"(per));                                     // (worked out again for every tile: no registers held)
        auto length = [&](int run) { return max(min(per, tasks - run * per), 0); };
        if (i < length(home)) return home * per + i;
        for (;;) {
            int most = 0, at = 0;
#pragma unroll
            for (int x = 0; x < 8; ++x) {
                const int left = length(x) - __hip_atomic_load(&counters[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (left > most) most = left, at = x;
            }
            if (most == 0) return -1;
            i = atomicAdd(&counters[at], 1);
            if (i < length(at)) return at * per + i;
        }
    };
    struct Tile { int row0, n_rows, f0, e, rt; };
    auto tile_of = [&](int task) {
        Tile t;
        const int q = task / nts, te = tile_expert[q], e = te & 1023;
        const int start = offs[e], cnt = offs[e + 1] - start;
        const int m = (cnt + MOE_PRODUCT_ROWS - 1) / MOE_PRODUCT_ROWS, rpt = ((cnt + m - 1) / m + 31) & ~31;
        const int local = task - (q - (te >> 10)) * nts, mt = local % m;
        t.f0 = local / m * FEATURES;
        t.row0 = start + mt * rpt;
        t.n_rows = min(rpt, cnt - mt * rpt);                              // (never empty: rpt <= MOE_PRODUCT_ROWS)
        t.e = e;
        t.rt = max((t.n_rows + 31) / 32, 3);
        t.row0 = __builtin_amdgcn_readfirstlane(t.row0);
        t.n_rows = __builtin_amdgcn_readfirstlane(t.n_rows);
        t.f0 = __builtin_amdgcn_readfirstlane(t.f0);
        t.e = __builtin_amdgcn_readfirstlane(t.e);
        t.rt = __builtin_amdgcn_readfirstlane(t.rt);
        return t;
    };
    auto bring_list = [&](const Tile& t, int to) {                        // a wavefront its 64 of 256
        bring4(rows + t.row0 + min((int)threadIdx.x, t.n_rows - 1), lds_byte(list[to]) + wave * 256);
    };
    if (threadIdx.x == 0) taken = take(atomicAdd(&counters[home], 1));
    __syncthreads();
    int task = __builtin_amdgcn_readfirstlane(taken);
    if (task < 0) return;
    Tile now = tile_of(task), next = now;
    bool more = false, stored = false;
    int at = 0;                                                           // the list of this tile
    bring_list(now, 0);
    landed<0>();
    unsigned ao[MOST], bo[CT];
    const char* const xa0 = (const char*)in;
    const char* xa = xa0;
    const char* wa0;
    const char* wa;
    int ra_rows = now.rt;                                                 // groups of 32 rows of the tile that is fetched
    auto aim_a = [&](const Tile& t, int from) {
        int lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));                                    // (worked out again for every tile: no registers held)
        const int chunk = (lane & 7) ^ (lane >> 3);
#pragma unroll
        for (int i = 0; i < MOST; ++i) {
            const int pair = list[from][min((i * 4 + wave) * 8 + (lane >> 3), t.n_rows - 1)];
            ao[i] = (KIND == MOE_DOWN || !by_top ? (unsigned)pair : __umulhi((unsigned)pair, by_top)) * (unsigned)(ldi * 2) + chunk * 16;
        }
        ra_rows = t.rt;
    };
    auto aim_b = [&](const Tile& t) {
        int lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));
        const int chunk = (lane & 7) ^ (lane >> 3);
        wa0 = (const char*)(w + (long)t.e * (KIND == MOE_GATED ? 2 : 1) * N * K);
#pragma unroll
        for (int i = 0; i < CT; ++i) {
            const int row = (i * 4 + wave) * 8 + (lane >> 3);
            int n;
            if (KIND == MOE_GATED) n = min(t.f0 + (row >> 5) * 16 + (row & 15), N - 1) + (row & 16 ? N : 0);
            else n = min(t.f0 + row, N - 1);
            bo[i] = (unsigned)n * (unsigned)(K * 2) + chunk * 16;
        }
    };
    int fa = 0, fb = 0, sa = 0, sb = 0;                                   // what is fetched next: piece, stage
    auto fetch_a = [&](int i) { bring16_at(xa, ao[i], base + (sa * AS + (i * 4 + wave) * 64) * 16); };
    auto fetch_b = [&](int i) { stream16_at(wa, bo[i], base + (B0 + sb * BS + (i * 4 + wave) * 64) * 16); };
    // behind a tile's last piece the next tile's first (behind the last tile's: its own, which nothing reads)
    auto next_a = [&]() {
        sa = sa + 1 == SA ? 0 : sa + 1;
        xa += 128;
        if (++fa == pieces) {
            fa = 0;
            xa = xa0;
            if (more) aim_a(next, at ^ 1);
        }
    };
    auto next_b = [&]() {
        sb = sb + 1 == SB ? 0 : sb + 1;
        wa += 128;
        if (++fb == pieces) {
            fb = 0;
            if (more) aim_b(next);
            wa = wa0;
        }
    };
    aim_a(now, 0);
    aim_b(now);
    wa = wa0;
    auto all_a = [&]() {
#pragma unroll
        for (int j = 0; j < MOST; ++j)
            if (j < ra_rows) fetch_a(j);
        next_a();
    };
    auto all_b = [&]() {
#pragma unroll
        for (int j = 0; j < CT; ++j) fetch_b(j);
        next_b();
    };
    all_b();
    all_a();
    all_b();
    all_a();
    all_b();
    landed<CT>();
    const int sw0 = r * 8 + (g ^ (r & 7)), sw1 = r * 8 + ((4 + g) ^ (r & 7));
    int ra = 0, rb = 0;                                                   // the stages of the piece that is multiplied
    auto run = [&](auto groups) {
        constexpr int RT = decltype(groups)::value;
        rfloatx4_t acc[RT][CT];
        rbf16x8_t a[2][RT], b[2][CT];
        auto read_one = [&](int s, int i, const ru32x4_t* as, const ru32x4_t* bs) {      // a0 b0 .. b7 a1 ..
            const int sw = s ? sw1 : sw0;
            if (i == 0) a[s][0] = *(const rbf16x8_t*)&as[wm * (RT * 128) + sw];
            else if (i <= CT) b[s][i - 1] = *(const rbf16x8_t*)&bs[wn * (CT * 128) + (i - 1) * 128 + sw];
            else a[s][i - CT] = *(const rbf16x8_t*)&as[wm * (RT * 128) + (i - CT) * 128 + sw];
        };
        constexpr int READS = RT + CT, MM = RT * CT, STEPS = MM / 2;
        static_assert(READS <= STEPS, "");
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
            __builtin_amdgcn_s_waitcnt(0xC07F);                           // lgkmcnt(0)
        };
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
#pragma unroll
        for (int x = 0; x < RT; ++x)
#pragma unroll
            for (int y = 0; y < CT; ++y) acc[x][y] = rfloatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int x = 0; x < RT; ++x)
#pragma unroll
            for (int y = 0; y < CT; ++y) in_place(acc[x][y]);
#pragma unroll
        for (int i = 0; i < READS; ++i) read_one(0, i, lds + ra * AS, lds + B0 + rb * BS);
        __builtin_amdgcn_s_waitcnt(0xC07F);
        asm volatile("s_nop 7" ::: "memory");
        auto piece = [&]() {
            half(I0(), lds + ra * AS, lds + B0 + rb * BS);
            if (stored) {                                                 // all but the weights of the piece after the next and the last tile's results
                stored = false;
                landed<CT + STORES>();
            } else {
                landed<CT>();
            }
            __builtin_amdgcn_s_waitcnt(0xC07F);
            ra = ra + 1 == SA ? 0 : ra + 1;
            rb = rb + 1 == SB ? 0 : rb + 1;
            if (ra_rows > RT) {                                           // the next tile has more rows (before the weights: landed() counts those)
#pragma unroll
                for (int j = RT; j < MOST; ++j)
                    if (j < ra_rows) fetch_a(j);
            }
            half(I1(), lds + ra * AS, lds + B0 + rb * BS);
            next_a();
            next_b();
        };
        int asked = 0;
        if (threadIdx.x == 0) asked = atomicAdd(&counters[home], 1);
        int end = 2;
        asm volatile("" : "+s"(end));
        for (int p = 0;;) {
#pragma unroll 1
            for (; p < end; ++p) piece();
            if (end == pieces) break;
            end = pieces;
            if (threadIdx.x == 0) taken = take(asked);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            task = __builtin_amdgcn_readfirstlane(taken);
            more = task >= 0;
            if (more) {
                next = tile_of(task);
                bring_list(next, at ^ 1);
            }
        }
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");                // the matrix instructions' results are there
        const int n0 = now.f0 + wn * 16 * CT / (KIND == MOE_GATED ? 2 : 1);
        int er = wm * 16 * RT + r, ec = n0 + (g & 1) * 16 + (g >> 1) * 8;
        asm volatile("" : "+v"(er), "+v"(ec));
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(out, 0, (int)((unsigned)out_rows * (unsigned)N * 2u), 0x00020000);
        auto finish = [&](auto ACT) {                                     // (the nonlinearity known: no branches between the results)
            constexpr int act = decltype(ACT)::value;
#pragma unroll
            for (int x = 0; x < RT; ++x) {
                const bool ok = er + x * 16 < now.n_rows;
                const unsigned line = (unsigned)list[at][er + x * 16] * (unsigned)N;
#pragma unroll
                for (int y = 0; y < CT; y += KIND == MOE_GATED ? 4 : 2) {
                    unsigned d[2][2];
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int i = 0; i < 2; ++i) {
                            float v[2];
#pragma unroll
                            for (int j = 0; j < 2; ++j) {
                                if (KIND == MOE_GATED) {
                                    float gt = sum_of(acc[x][y + 2 * h][2 * i + j]), up = sum_of(acc[x][y + 2 * h + 1][2 * i + j]);
                                    gate_prepare(gt, up, act, act_limit);
                                    v[j] = gate_act(gt, act) * up;
                                } else {
                                    v[j] = sum_of(acc[x][y + h][2 * i + j]);
                                    if (KIND == MOE_PLAIN) v[j] = plain_act(v[j], act);
                                }
                            }
                            d[h][i] = bf16_pair(v[0], v[1]);
                        }
                    const cpmcu_u32x2_t p0 = __builtin_amdgcn_permlane16_swap(d[0][0], d[1][0], false, false);
                    const cpmcu_u32x2_t p1 = __builtin_amdgcn_permlane16_swap(d[0][1], d[1][1], false, false);
                    const int col = ec + y * (KIND == MOE_GATED ? 8 : 16);
                    // (N % 8 == 0: the whole chunk.  Beyond the buffer's end nothing is written, and every wavefront counts the same stores)
                    __builtin_amdgcn_raw_buffer_store_b128(ru32x4_t{p0.x, p1.x, p0.y, p1.y}, rsrc, ok && col < N ? (line + (unsigned)col) * 2u : 0xFFFFF000u, 0, KIND == MOE_DOWN ? 0 : 2);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        if (KIND == MOE_DOWN || act == CPMCU_ACT_SILU) finish(std::integral_constant<int, CPMCU_ACT_SILU>());
        else if (act == CPMCU_ACT_GELU_TANH) finish(std::integral_constant<int, CPMCU_ACT_GELU_TANH>());
        else finish(std::integral_constant<int, KIND == MOE_PLAIN ? CPMCU_ACT_RELU_SQUARED : CPMCU_ACT_CLAMPED_SWISH>());
    };
    for (;;) {
        if (now.rt == 3) run(std::integral_constant<int, 3>());
        else if (now.rt == 4) run(std::integral_constant<int, 4>());
        else if (now.rt == 5) run(std::integral_constant<int, 5>());
        else if (now.rt == 6) run(std::integral_constant<int, 6>());
        else run(std::integral_constant<int, 7>());
        if (!more) break;
        stored = true;
        now = next;
        at ^= 1;
    }
    landed<0>();
}

bool moe_product_takes(int K, int N, bool gated, long in_rows, long ldi, long pairs, int top) {
    return pairs * top < (1L << 32) && K % 64 == 0 && K >= 512 && N % 8 == 0 && in_rows * ldi < (1L << 31) && (long)N * (gated ? 2 : 1) * K < (1L << 31) &&
           pairs * N < (1L << 31) - 4096;
}

const char* moe_product(int kind, const bf16_t* in, long ldi, const bf16_t* w, const int* rows, const int* offs, const int* tile_expert,
                        const int* n_tiles, int* counters, bf16_t* out, long pairs, int K, int N, int top, long most_tiles, int act, float act_limit,
                        hipStream_t stream) {
    const int features = kind == MOE_GATED ? 128 : 256;
    const long blocks = (most_tiles * ((N + features - 1) / features) + 7) / 8 * 8;
    CPMCU_REQUIRE(blocks < (1L << 31) - 4096, "moe_product: %ld tiles", blocks);
    // pair / top as the upper half of pair * by_top (exact: pair * top < 2^32, below); top = 1: none
    const unsigned by_top = top == 1 ? 0u : (unsigned)(((1UL << 32) + top - 1) / top);
    CPMCU_REQUIRE(pairs * top < (1L << 32), "moe_product: %ld pairs of %d a token", pairs, top);
    const unsigned grid = (unsigned)(blocks < 256 ? blocks : 256);
    auto* const kernel = kind == MOE_GATED ? moe_product_kernel<MOE_GATED> : kind == MOE_PLAIN ? moe_product_kernel<MOE_PLAIN> : moe_product_kernel<MOE_DOWN>;
    kernel<<<grid, 256, 0, stream>>>(in, (int)ldi, w, rows, offs, tile_expert, n_tiles, counters, out, (int)pairs, K, N, by_top, act, act_limit);
    CPMCU_LAUNCH_CHECK("moe_product");
    return nullptr;
}
