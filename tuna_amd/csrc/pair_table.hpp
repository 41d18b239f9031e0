// The decode table of the streaming kernels and their kin (kLutBytes in tuna_internal.h), made by all threads of a workgroup.
#pragma once
#include "epilogue.hpp"

namespace tuna {

// Entries of four banks, 16 bytes each, go to `store(entry, value)`; piece p belongs to byte p >> 4.  code_lane: code[lane & 15].  The high
// code of a piece is one for a whole wave and comes from a lane as a scalar, the low one is a thread's own for all its pieces where
// the workgroup has a multiple of 256 threads: seven instructions a piece, where gathering both across lanes took eighteen - 0.7 -> 0.3
// us of a launch's start with eight waves, which issue them two to a SIMD.
template <int THREADS, class Store>
__device__ __forceinline__ void build_pair_table(int tid, float code_lane, const Store &store)
{
    constexpr int kPieces = kLutBytes / 16;
    const int code_bits = (int)(uint32_t)__builtin_bit_cast(uint16_t, (f16)code_lane);
    if constexpr (THREADS % 256 == 0 && kPieces % THREADS == 0) {
        const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(((tid >> 4) & 15) << 2, code_bits) << 16;
        const int high = __builtin_amdgcn_readfirstlane(tid >> 8);
#pragma unroll
        for (int i = 0; i < kPieces / THREADS; ++i) {
            const uint32_t v = lo | (uint32_t)__builtin_amdgcn_readlane(code_bits, high + i * (THREADS / 256));
            store(tid + i * THREADS, u32x4{v, v, v, v});
        }
    } else {
#pragma unroll 4
        for (int p = tid; p < kPieces; p += THREADS) {
            const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(((p >> 4) & 15) << 2, code_bits) << 16;
            const uint32_t v = lo | (uint32_t)__builtin_amdgcn_readlane(code_bits, __builtin_amdgcn_readfirstlane(p >> 8));
            store(p, u32x4{v, v, v, v});
        }
    }
}
// The same for a number of threads known at run time, a multiple of 64.
template <class Store>
__device__ __forceinline__ void build_pair_table(int tid, int threads, float code_lane, const Store &store)
{
    constexpr int kPieces = kLutBytes / 16;
    const int code_bits = (int)(uint32_t)__builtin_bit_cast(uint16_t, (f16)code_lane);
    if (threads % 256 == 0) {
        const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(((tid >> 4) & 15) << 2, code_bits) << 16;
        int high = __builtin_amdgcn_readfirstlane(tid >> 8);
#pragma unroll 4
        for (int p = tid; p < kPieces; p += threads, high += threads >> 8) {
            const uint32_t v = lo | (uint32_t)__builtin_amdgcn_readlane(code_bits, high);
            store(p, u32x4{v, v, v, v});
        }
    } else {
#pragma unroll 4
        for (int p = tid; p < kPieces; p += threads) {
            const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(((p >> 4) & 15) << 2, code_bits) << 16;
            const uint32_t v = lo | (uint32_t)__builtin_amdgcn_readlane(code_bits, __builtin_amdgcn_readfirstlane(p >> 8));
            store(p, u32x4{v, v, v, v});
        }
    }
}
template <int THREADS>
__device__ __forceinline__ void build_pair_table(unsigned char *lut, int tid, float code_lane)
{
    build_pair_table<THREADS>(tid, code_lane, [&](int p, const u32x4 &v) { reinterpret_cast<u32x4 *>(lut)[p] = v; });
}

}  // namespace tuna
