// Loads that the kernel waits for itself (gfx950).  A 16-byte load into registers and the LDS reads of the same compute unit
// return their data over one path: 8 KB per wave of loads and 56 table reads take 64 and 55 ns apart and 118 together, with
// the loads going to LDS 66 (256 workgroups of eight waves).  The kernels that read LDS most of the time therefore have
// their activations brought into LDS directly.  The compiler, seeing such loads, would wait for all of them at every use of a
// loaded register and at every LDS store: here they are instructions it does not look into, so every wait is written out.
// For the compiler a register that such a load fills holds its value at once, and is free from its last use on.  So every
// destination is passed ("+v") through a wait that covers its load, on EVERY path from there, also where nothing uses what was
// loaded (tests/test_async_loads.py follows the assembly).
#pragma once
#include "epilogue.hpp"

namespace tuna {

// A buffer descriptor of `bytes` bytes from `base` on (uniform): loads beyond it give zeros, in registers and in LDS.
__device__ __forceinline__ u32x4 buffer_at(const void *base, size_t bytes)
{
    const uint64_t p = (uint64_t)(uintptr_t)base;
    const uint32_t n = (uint32_t)(bytes < 0xffffffffu ? bytes : 0xffffffffu);
    return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)p), (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(p >> 32)) & 0xffffu,
                 (uint32_t)__builtin_amdgcn_readfirstlane((int)n), 0x00020000u};
}
// 16 bytes a lane into LDS, lane l's at lds + 16 l.
__device__ __forceinline__ void load_to_lds(const u32x4 &rsrc, uint32_t offset, uint32_t uniform, uint32_t lds)
{
    // (the address in M0 is an operand: the compiler writes that register itself and knows when it has changed)
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(offset), "s"(rsrc), "s"(uniform), "{m0}"(lds));
}
__device__ __forceinline__ void load_async(u32x4 &dst, const u32x4 &rsrc, uint32_t offset, uint32_t uniform)
{
    asm volatile("buffer_load_dwordx4 %0, %1, %2, %3 offen" : "=v"(dst) : "v"(offset), "s"(rsrc), "s"(uniform));
}
__device__ __forceinline__ void load_async(u32x2 &dst, const u32x4 &rsrc, uint32_t offset, uint32_t uniform)
{
    asm volatile("buffer_load_dwordx2 %0, %1, %2, %3 offen" : "=v"(dst) : "v"(offset), "s"(rsrc), "s"(uniform));
}
__device__ __forceinline__ void load_async(uint32_t &dst, const u32x4 &rsrc, uint32_t offset, uint32_t uniform)
{
    asm volatile("buffer_load_dword %0, %1, %2, %3 offen" : "=v"(dst) : "v"(offset), "s"(rsrc), "s"(uniform));
}
// At most N of the wave's vector memory operations are pending: those before the last N have arrived.
template <int N>
__device__ __forceinline__ void wait_loads()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

}  // namespace tuna
