// Loads from memory straight to LDS, and the waits for them.
#pragma once
#include "common.h"

// 64 lanes' 16 bytes, one behind the other from byte `to` of LDS on (the wavefront's; the lanes' addresses are free).  Nothing
// waits for them but landed(): the compiler does not count loads of an asm block (those of the builtin it does, and makes
// every LDS read behind them wait for all).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"                      // m0 on the clobber list
__device__ inline void bring16(const void* from, unsigned to) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(to), "v"(from) : "memory", "m0");
}
__device__ inline void stream16(const void* from, unsigned to) {      // the same past the caches
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(to), "v"(from) : "memory", "m0");
}
__device__ inline void bring4(const void* from, unsigned to) {        // 4 bytes a lane
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(to), "v"(from) : "memory", "m0");
}
#pragma clang diagnostic pop
__device__ inline unsigned lds_byte(const void* p) {                  // where a shared variable lies
    return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}
// all but this wavefront's last N loads have landed and what it read from and wrote to LDS is done; then the workgroup meets
template <int N>
__device__ inline void landed() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"i"(N) : "memory");
    __builtin_amdgcn_sched_barrier(0);
}
