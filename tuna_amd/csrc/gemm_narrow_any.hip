// Instantiations and launcher of the narrow-row kernel's variants for any m and k (gemm_narrow.hpp).
//
// Buffer loads that return zeros beyond the operands take the place of the aligned variants' plain loads: 16-row tiles with
// 16 waves along k for the smallest launches, 32- and 64-row tiles with 4 or 8 waves beyond, rings of 2 .. 8, passes of 1, 2
// or 4 token tiles.  What bounds them: at one token the launch and two memory round trips (1192 x 2000 3.0 us, an empty
// launch 1.7; the general kernel 9.1), then the workgroup's own chain of ring turns: 8576 x 9856 at 5 tokens 14.8 us (31.0),
// where 134 workgroups leave half of the compute units idle and the LDS of the others is busy 59 % of the cycles.
#include "gemm_narrow.hpp"

namespace tuna {

typedef void (*NarrowKernelFn)(const uint8_t *, const void *, const float *, const float *, int, int, int, int, void *, int,
                               const void *, int, int, int);
// (fn[2], fn[3]: with a scale per block of a row)
#define BLKV(LW, WK, U, TT, P) gemm_narrow_kernel<LW, WK, U, P, TT, true, 16 * LW, true>
#define ANY1(LW, WK, U) {16 * LW, WK, U, 1, {gemm_narrow_kernel<LW, WK, U, 0, 1, false, 16 * LW, true>, gemm_narrow_kernel<LW, WK, U, 1, 1, false, 16 * LW, true>, BLKV(LW, WK, U, 1, 0), BLKV(LW, WK, U, 1, 1)}}
#define ANYT(LW, WK, U, TT) {16 * LW, WK, U, TT, {gemm_narrow_kernel<LW, WK, U, 1, TT, false, 16 * LW, true>, gemm_narrow_kernel<LW, WK, U, 1, TT, false, 16 * LW, true>, BLKV(LW, WK, U, TT, 1), BLKV(LW, WK, U, TT, 1)}}
static const struct {
    int rows, wk, u, tt;
    NarrowKernelFn fn[4];  // B fragments loaded per lane (up to 4 tokens) / contiguously and permuted
} kAny[] = {
    ANY1(1, 16, 4), ANY1(1, 16, 2), ANY1(2, 8, 4), ANY1(2, 8, 8), ANY1(4, 4, 4), ANY1(4, 8, 4),
    ANYT(2, 8, 2, 2), ANYT(2, 8, 4, 2), ANYT(4, 8, 2, 2), ANYT(2, 8, 2, 4), ANYT(4, 4, 2, 4),
};
#undef ANY1
#undef ANYT
#undef BLKV
static constexpr int kNumAny = sizeof(kAny) / sizeof(kAny[0]);
static OptInFlag g_any_attr_done[16][kNumAny][4];

static int find_any(int rows, int wk, int u, int tt)
{
    for (int i = 0; i < kNumAny; ++i)
        if (kAny[i].rows == rows && kAny[i].wk == wk && kAny[i].u == u && kAny[i].tt == tt) return i;
    return -1;
}

bool narrow_any_variant_exists(int rows, int waves_k, int prefetch, int token_tiles)
{
    return find_any(rows, waves_k, prefetch, token_tiles) >= 0;
}

// blk_shift >= 0: a scale per 64 << blk_shift weights of a row; the workgroup's scales are kept in LDS where they fit.
hipError_t launch_gemm_narrow_any(const NarrowArgs &args, int blk_shift, int rows, int waves_k, int prefetch, int token_tiles, int dev,
                                  hipStream_t stream)
{
    const int vi = find_any(rows, waves_k, prefetch, token_tiles), fi = (args.n > 4 ? 1 : 0) + (blk_shift >= 0 ? 2 : 0);
    if (vi < 0 || dev < 0 || dev >= 16) return hipErrorInvalidConfiguration;
    const NarrowKernelFn fn = kAny[vi].fn[fi];
    const hipError_t e = ensure_lds_opt_in(g_any_attr_done[dev][vi][fi], reinterpret_cast<const void *>(fn));
    if (e != hipSuccess) return e;
    size_t lds = (size_t)kLutBytes + (size_t)waves_k * (rows / 16) * token_tiles * 1024;
    const int nblk = blk_shift >= 0 ? args.k >> (6 + blk_shift) : 1;
    const size_t scale_bytes = (size_t)rows * (nblk + 1) * 4;
    const int slds = blk_shift >= 0 && lds + scale_bytes <= (size_t)kLdsLimit;
    if (slds) lds += scale_bytes;
    const dim3 grid((unsigned)((args.m + rows - 1) / rows), (unsigned)((args.n + 16 * token_tiles - 1) / (16 * token_tiles)), 1);
    hipLaunchKernelGGL(fn, grid, dim3(waves_k * 64), lds, stream, args.q, args.x, args.code, args.absmax, args.k, args.n, args.n_it,
                       args.m, args.out, args.epilogue, args.residual, blk_shift >= 0 ? blk_shift : 0, nblk, slds);
    return hipGetLastError();
}

}  // namespace tuna
