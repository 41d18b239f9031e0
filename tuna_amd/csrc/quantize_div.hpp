// The quantizer's division by a block maximum (dequant_kernel.hip) and nothing else: shared with the
// self-test kernel of the diagnostic build (bench_kernels.hip), which runs it on every pair of fp16 values.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace tuna {

// fp32(w) / a, correctly rounded, for the quotients this kernel forms: w an fp16 value, a the
// largest |fp16| of its block, so |w| <= a and both are normal binary32 numbers (or w is zero).
// y is the reciprocal of a refined once from v_rcp_f32 (computed once per block); the quotient is one
// multiply and one fused correction step.  No denormal-mode switches, no scaling: the ranges rule
// out what the general division sequence guards against.  Equality with the IEEE division is
// checked for every pair (w, a) of fp16 values with |w| <= a in tests/test_gpu_parity.py.
__device__ __forceinline__ float refined_rcp(float a)
{
    const float y = __builtin_amdgcn_rcpf(a);
    return __builtin_fmaf(__builtin_fmaf(-a, y, 1.0f), y, y);
}

// (float)h * y and w - q * a with the fp16 operand read in place (no conversion instruction).
template <int HI>
__device__ __forceinline__ float mix_mul(uint32_t pair, float y)
{
    float q;
    if constexpr (HI) asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(q) : "v"(pair), "v"(y));
    else asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(q) : "v"(pair), "v"(y));
    return q;
}
template <int HI>
__device__ __forceinline__ float mix_residual(float q, float a, uint32_t pair)
{
    float r;
    if constexpr (HI) asm("v_fma_mix_f32 %0, -%1, %2, %3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(r) : "v"(q), "v"(a), "v"(pair));
    else asm("v_fma_mix_f32 %0, -%1, %2, %3 op_sel:[0,0,0] op_sel_hi:[0,0,1]" : "=v"(r) : "v"(q), "v"(a), "v"(pair));
    return r;
}

template <int HI>  // w = the low or high half of `pair`
__device__ __forceinline__ float div_by_block_max(uint32_t pair, float a, float y)
{
    const float q = mix_mul<HI>(pair, y);
    return __builtin_fmaf(mix_residual<HI>(q, a, pair), y, q);
}

}  // namespace tuna
