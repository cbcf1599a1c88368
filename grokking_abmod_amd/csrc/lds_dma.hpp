// Loads from global memory straight into LDS, and the waits of a pipeline that
// keeps some in flight.
#pragma once

#include <hip/hip_runtime.h>

namespace meshgpt::kern {

typedef __attribute__((address_space(3))) float lds_f32;

// LDS[base + 16 * lane .. +16) = g[0..4) for every lane of the wave; base is
// wave-uniform.  Earlier LDS reads complete first; m0 is preserved.
__device__ __forceinline__ void dma16(const void *g, void *base) {
    const uint32_t m = __builtin_amdgcn_readfirstlane(uint32_t(size_t((lds_f32 *)base)));
    uint32_t save;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %1\n\t"
        "s_waitcnt lgkmcnt(0)\n\t"
        "global_load_lds_dwordx4 %2, off\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(save)
        : "s"(m), "v"(g)
        : "memory");
}

// All but the wave's N latest loads have landed.
template <int N>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// A workgroup barrier that waits for LDS operations only (in-flight global
// loads, such as the next tile's, keep flying).
__device__ __forceinline__ void barrier_lds() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

}  // namespace meshgpt::kern
