// What the kernels whose lanes hold one packed dword per 16-row tile (gemm_tall.hip, gemm_broad.hip) have in common: how they group
// those tiles into loads, and a tile's end - the exchange between parts of k and the output.
#pragma once
#include "epilogue.hpp"
#include "pair_table.hpp"

namespace tuna {

// Pieces of a lane's weights of a k-step's half: row tiles of 16 in loads of four, two and one dwords.
template <int RT>
struct Pieces {
    static constexpr int fours = RT / 4, twos = (RT & 2) / 2, ones = RT & 1, count = fours + twos + ones;
    static constexpr int width(int p) { return p < fours ? 4 : p < fours + twos ? 2 : 1; }
    static constexpr int first(int p) { return p <= fours ? 4 * p : p <= fours + twos ? 4 * fours + 2 * (p - fours) : RT - 1; }  // row tile
    static constexpr int of(int r) { return r < 4 * fours ? r / 4 : r < 4 * fours + 2 * twos ? fours : count - 1; }
    // the same of the piece that row tile r, known at run time, is in
    static __device__ __forceinline__ int width_at(int r) { return r < 4 * fours ? 4 : r < 4 * fours + 2 * twos ? 2 : 1; }
    static __device__ __forceinline__ int first_at(int r) { return r < 4 * fours ? r & ~3 : r < 4 * fours + 2 * twos ? 4 * fours : RT - 1; }
};

// Sums of a tile between its parts of k: each part's go to its slot of the workspace, and the last workgroup to arrive adds all of
// them in k order.  Wave w holds the sums of row tiles w, w + WAVES .. of TILES; PB parts' loads are issued before the first is
// awaited.  Whether this workgroup is that last one.
template <int WAVES, int TILES, int NT, int PB>
__device__ __forceinline__ bool add_parts(f32x4 (&sum)[(TILES + WAVES - 1) / WAVES][NT], float *ws, unsigned *counter, size_t item, int part, int split,
                                          int tid, int wave, volatile unsigned *ticket)
{
    constexpr int TW = (TILES + WAVES - 1) / WAVES;
    constexpr size_t SLOT = (size_t)TILES * NT * 1024;
    auto slot = [&](int p) {
        return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<unsigned char *>(ws) + (item * split + p) * SLOT, 0, (int)SLOT, 0x00020000);
    };
    const int at = (wave * NT * 64 + (tid & 63)) * 16;
    const auto dst = slot(part);
#pragma unroll
    for (int w = 0; w < TW; ++w)
        if (wave + w * WAVES < TILES) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, sum[w][t]), dst, at, (w * WAVES * NT + t) * 1024, 16);
        }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the sums have left this CU
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __syncthreads();
    if (tid == 0) *ticket = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    // (one value for the wave: a branch that could differ between lanes makes the slots below look as if they did)
    if (__builtin_amdgcn_readfirstlane((int)*ticket) != split - 1) return false;
    if (tid == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int w = 0; w < TW; ++w) {
        if (wave + w * WAVES >= TILES) continue;
#pragma unroll
        for (int t = 0; t < NT; ++t) sum[w][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int p = 0; p < split; p += PB) {
            f32x4 v[PB][NT];
#pragma unroll
            for (int b = 0; b < PB; ++b) {
                const auto src = slot(min(p + b, split - 1));
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    v[b][t] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(src, at, (w * WAVES * NT + t) * 1024, 16));
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int b = 0; b < PB; ++b)
                if (p + b < split) {
#pragma unroll
                    for (int t = 0; t < NT; ++t) sum[w][t] += v[b][t];
                }
        }
    }
    return true;
}

// A tile's sums to its outputs, through LDS into rows of eight consecutive features.  RT row tiles to a row group.
template <int WAVES, int TILES, int NT, int RT>
__device__ __forceinline__ void store_tile(const f32x4 (&sum)[(TILES + WAVES - 1) / WAVES][NT], float *ob, int tid, int wave, void *out, const void *residual,
                                           int epilogue, int row_base, int m, int tok_base, int tokens)
{
    using P = Pieces<RT>;
    constexpr int PITCH = 16 * TILES + 4;
    const int i16 = tid & 15, g = (tid & 63) >> 4;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < (TILES + WAVES - 1) / WAVES; ++w) {
        const int r = wave + w * WAVES, group = TILES > RT && r >= RT ? 1 : 0, r16 = r - group * RT;
        if (r < TILES) {
            const int width = P::width_at(r16), first = P::first_at(r16);
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) ob[(16 * t + i16) * PITCH + 16 * (group * RT + first) + width * (4 * g + v) + r16 - first] = sum[w][t][v];
        }
    }
    __syncthreads();
    for (int c = tid; c < 16 * NT * 2 * TILES; c += 64 * WAVES) {
        const int tok = c / (2 * TILES), r8 = c - tok * (2 * TILES), row = row_base + 8 * r8;
        if (tok < tokens && row + 8 <= m) {
            const float *src = ob + tok * PITCH + 8 * r8;
            store_features8(reinterpret_cast<f16 *>(out), reinterpret_cast<const f16 *>(residual), epilogue, (size_t)(tok_base + tok), m, row,
                            *reinterpret_cast<const f32x4 *>(src), *reinterpret_cast<const f32x4 *>(src + 4));
        }
    }
}

}  // namespace tuna
