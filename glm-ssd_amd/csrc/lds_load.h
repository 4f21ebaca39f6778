// Loads from global memory straight to LDS, waited for by hand on the vector-memory counter.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef uint32_t u4 __attribute__((ext_vector_type(4)));

// a wave-uniform pointer whose 64-bit arithmetic ran on the vector unit, back in scalar registers
// (a buffer resource or scalar base kept in VGPRs costs a readfirstlane loop per load)
__device__ __forceinline__ const uint8_t *uniform_ptr(const uint8_t *p) {
    const uint64_t v = (uint64_t)p;
    return (const uint8_t *)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32)) << 32) |
                             (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v));
}
// 16 bytes per lane from rsrc + voff + soff to LDS address lds + 16 lane, in flight on the vector-memory
// counter. Written as an asm statement because the compiler waits for every outstanding load of this
// kind before any LDS read; the waits are placed by hand (wait_vm) instead. No register is written but
// M0, which the compiler only holds between a write of its own and the instruction that needs it.
__device__ __forceinline__ void dma16(uint32_t lds, uint32_t voff, uint32_t soff, u4 rsrc) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voff), "s"(rsrc), "s"(__builtin_amdgcn_readfirstlane(soff)) : "memory");
}
// the words of a raw buffer resource over `bytes` bytes from a wave-uniform base (as BufferAt makes it)
__device__ __forceinline__ u4 rsrc_words(const uint8_t *base, uint32_t bytes) {
    const uint64_t b = (uint64_t)base;
    return u4{(uint32_t)b, (uint32_t)(b >> 32) & 0xffffu, bytes, 0x00020000u};
}
template <int N>
__device__ __forceinline__ void wait_vm() {   // until at most N vector-memory operations are outstanding
    static_assert(N < 64, "vmcnt");
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}
