// Transfers from memory straight to LDS, and the small helpers around them.
#pragma once

#include "common.hpp"

namespace lmx {

// The value as one the compiler cannot see through: what is derived from it
// inside the key loop is computed there, not hoisted into registers that the
// loop does not have (spilled addresses would be reloaded through the same
// counter as the transfers, and wait for them).
template <typename T>
__device__ __forceinline__ void opaque(T& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ const char* uniform_ptr(const char* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<const char*>(((uint64_t)hi << 32) | lo);
}

// Sixteen bytes a lane from memory to LDS: lane l's land at lds + 16 l.
// Written out so that the compiler, which cannot tell a transfer's stage from
// the one being read, puts no wait for it before every LDS read; wait_dma
// waits before the barrier that publishes the tile.  base is wave-uniform.
__device__ __forceinline__ void dma16(const char* base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :: "v"(off), "s"(uniform_ptr(base)), "s"(__builtin_amdgcn_readfirstlane(lds))
                 : "memory", "m0");
}
// The same from an address of the lane's own.
__device__ __forceinline__ void dma16_lane(const void* p, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" :: "v"(p), "s"(__builtin_amdgcn_readfirstlane(lds))
                 : "memory", "m0");
}
// All but the newest N transfers have landed.
template <int N>
__device__ __forceinline__ void wait_dma() {
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

}  // namespace lmx
