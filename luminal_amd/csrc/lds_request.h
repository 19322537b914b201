// Requests from memory straight into LDS, counted and waited for by the kernel itself: what the kernels that stage their tiles
// through several buffers share.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lhip {

// 64 lanes x 16 (4) bytes from base + the lane's offset to consecutive LDS from `lds` on.  Inline assembly, because the compiler
// would otherwise wait for the newest of them ahead of every LDS read.  (m0 is a reserved register: the compiler keeps nothing in it
// from one statement to another.)
template <int BYTES>
__device__ __forceinline__ void lds_request(const void *base, uint32_t voff, uint32_t lds) {
    static_assert(BYTES == 16 || BYTES == 4, "a lane's share");
    if constexpr (BYTES == 16)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(base) : "memory");
    else
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(voff), "s"(base) : "memory");
}
// Until at most N of this wave's loads are under way.
template <int N>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}
// A barrier that waits for nothing by itself, and that no access of the source crosses.
__device__ __forceinline__ void bare_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

}  // namespace lhip
