// What the kernels of large products share: operands straight into LDS, matrix instructions with their sums in place, results as bf16.
#pragma once
#include "lds_direct.h"

typedef __bf16 rbf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 rbf16x2_t __attribute__((ext_vector_type(2)));
typedef float rfloatx4_t __attribute__((ext_vector_type(4)));
typedef float rfloatx2_t __attribute__((ext_vector_type(2)));
typedef unsigned ru32x4_t __attribute__((ext_vector_type(4)));

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"                      // m0 on the clobber list
__device__ inline void bring16_at(const void* base, unsigned off, unsigned to) {      // as bring16, `off` bytes behind a uniform address
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(off), "s"(base) : "memory", "m0");
}
__device__ inline void stream16_at(const void* base, unsigned off, unsigned to) {    // the same past the caches
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(to), "v"(off), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop
__device__ inline void multiply_into(rfloatx4_t& c, rbf16x8_t a, rbf16x8_t b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
// An accumulator is written up to here: blocks of asm keep their order, and what one takes as an operand stands before it.  (The compiler keeps
// no distances for instructions inside asm: zeros belong in front of the wait that stands in front of the first matrix instruction.)
__device__ inline void in_place(rfloatx4_t& c) { asm volatile("" : "+a"(c)); }
__device__ inline float sum_of(float c) {
    float v;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(c));
    return v;
}
__device__ inline unsigned bf16_pair(float a, float b) {             // to the nearest, ties to even
    return __builtin_bit_cast(unsigned, __builtin_convertvector(rfloatx2_t{a, b}, rbf16x2_t));
}
