// Device-side types and the fused output epilogues shared by the GEMM kernels.
#pragma once
#include "tuna_internal.h"

namespace tuna {

typedef _Float16 f16;
typedef f16 f16x2 __attribute__((ext_vector_type(2)));
typedef f16 f16x4 __attribute__((ext_vector_type(4)));
typedef f16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) uint32_t lds_u32;

// Final store of 4 consecutive output features (columns col .. col+3 of a row of `out` that is
// ld long) of one token, with the fused epilogues:
//   TUNA_EPILOGUE_NONE      out = fp16(v)
//   TUNA_EPILOGUE_RESIDUAL  out = fp16(v + residual), residual fp16 with the layout of out
//   TUNA_EPILOGUE_SILU_MUL  weight rows interleaved (2i: gate_i, 2i+1: up_i): the four values are
//                           (g0, u0, g1, u1) and out, ld/2 long, gets fp16(silu(g) * u) for both
__device__ __forceinline__ float silu_mul(float g, float u) { return g / (1.0f + __expf(-g)) * u; }

__device__ __forceinline__ void store_features4(f16 *out, const f16 *residual, int epilogue, size_t tok, int ld, int col,
                                                float v0, float v1, float v2, float v3)
{
    if (epilogue == TUNA_EPILOGUE_SILU_MUL) {
        const f16x2 h = {(f16)silu_mul(v0, v1), (f16)silu_mul(v2, v3)};
        *reinterpret_cast<f16x2 *>(out + tok * (size_t)(ld >> 1) + (col >> 1)) = h;
        return;
    }
    const size_t at = tok * (size_t)ld + col;
    if (epilogue == TUNA_EPILOGUE_RESIDUAL) {
        const f16x4 r = *reinterpret_cast<const f16x4 *>(residual + at);
        v0 += (float)r[0], v1 += (float)r[1], v2 += (float)r[2], v3 += (float)r[3];
    }
    *reinterpret_cast<f16x4 *>(out + at) = f16x4{(f16)v0, (f16)v1, (f16)v2, (f16)v3};
}

// The same for 8 consecutive output features (col a multiple of 8, ld a multiple of 8: 16-byte stores of `out`).
__device__ __forceinline__ void store_features8(f16 *out, const f16 *residual, int epilogue, size_t tok, int ld, int col,
                                                const f32x4 lo, const f32x4 hi)
{
    float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    if (epilogue == TUNA_EPILOGUE_SILU_MUL) {
        f16x4 h;
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i] = (f16)silu_mul(v[2 * i], v[2 * i + 1]);
        *reinterpret_cast<f16x4 *>(out + tok * (size_t)(ld >> 1) + (col >> 1)) = h;
        return;
    }
    const size_t at = tok * (size_t)ld + col;
    if (epilogue == TUNA_EPILOGUE_RESIDUAL) {  // (the residual is aligned to 8 bytes only)
        const f16x4 r0 = *reinterpret_cast<const f16x4 *>(residual + at), r1 = *reinterpret_cast<const f16x4 *>(residual + at + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += (float)r0[i], v[4 + i] += (float)r1[i];
    }
    f16x8 h;
#pragma unroll
    for (int i = 0; i < 8; ++i) h[i] = (f16)v[i];
    *reinterpret_cast<f16x8 *>(out + at) = h;
}

}  // namespace tuna
