// Products of routed experts that have many rows each (moe_product.hip).
#pragma once
#include "common.h"

#define MOE_PRODUCT_ROWS 224                   // rows of a tile at most
#define MOE_PRODUCT_COUNTERS 16                // ints that moe_group_kernel clears: 8 of the first product, 8 of the second
enum { MOE_GATED = 0, MOE_PLAIN = 1, MOE_DOWN = 2 };

// whether the kernel takes rows of K columns and N features at all (widths and sizes; addresses are the caller's)
bool moe_product_takes(int K, int N, bool gated, long in_rows, long ldi, long pairs, int top);
const char* moe_product(int kind, const bf16_t* in, long ldi, const bf16_t* w, const int* rows, const int* offs, const int* tile_expert,
                        const int* n_tiles, int* counters, bf16_t* out, long pairs, int K, int N, int top, long most_tiles, int act, float act_limit,
                        hipStream_t stream);
