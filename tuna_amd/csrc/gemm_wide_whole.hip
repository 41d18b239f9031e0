// Many-token tiles that no workgroups share: 256 weight rows x 16 NT tokens each, the steps and the decode of gemm_wide.hpp.  For a dense
// GEMM a kernel for every number of token tiles, without the bookkeeping of gemm_wide.hip: the arguments arrive in scalar registers
// and a tile's end is short; one for groups.
#include "gemm_wide.hpp"

namespace tuna {

namespace {
// One tile, from its first token on.
template <int NT, bool KTAIL, bool BLK>
__device__ __forceinline__ void wide_whole_tile(const WideTile &w, const float *code, unsigned char *smem, int tok0, void *out, int epilogue, const void *residual)
{
    constexpr int kTiles = (NT + 3) / 4 * 4;  // (outputs are stored four token tiles at a time)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i16 = lane & 15, g = lane >> 4;
    f32x4 acc[4][kTiles];
    wide_steps<NT, KTAIL, BLK>(acc, w, smem, code, true, 0, w.steps_total, tid);
    __syncthreads();  // every wave is done with the stages
    unsigned char *const xs = smem + kLutBytes;
    if (epilogue == TUNA_EPILOGUE_NONE) {
        // [token of 64][8 pieces of eight rows, XOR-swizzled with the token]
        unsigned char *const mine = xs + wave * 8192;
        const int r8 = lane & 7, tk = lane >> 3, row = w.row_base + wave * 64 + 8 * r8;
        f16 *outp = reinterpret_cast<f16 *>(out) + (size_t)(tok0 + tk) * (size_t)w.m + row;
        int left = row + 8 <= w.m ? w.tokens - tk : 0;
#pragma unroll
        for (int b = 0; b < kTiles; b += 4) {
#pragma unroll
            for (int i = 0; i < 16; ++i) asm volatile("" : "+a"(acc[i & 3][b + (i >> 2)]));  // (read here, not ahead of it)
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            f16x8 y;
#pragma unroll
                            for (int i = 0; i < 8; ++i) y[i] = (f16)acc[i & 3][b + t][2 * h + (i >> 2)];
                            *reinterpret_cast<f16x8 *>(mine + (16 * t + i16) * 128 + (((2 * g + h) ^ (i16 & 7)) << 4)) = y;
                        }
            f16x8 y[8];  // tokens tk + 8 h, rows `row` .. + 7
#pragma unroll
            for (int h = 0; h < 8; ++h) y[h] = *reinterpret_cast<const f16x8 *>(mine + (8 * h + tk) * 128 + ((r8 ^ tk) << 4));
#pragma unroll
            for (int h = 0; h < 8; ++h)
                if (8 * h < left) *reinterpret_cast<f16x8 *>(outp + (size_t)(8 * h) * (size_t)w.m) = y[h];
            outp += (size_t)64 * (size_t)w.m, left -= 64;
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
        unsigned char *const mine = xs + wave * 16384;
        WideOut o = wide_out(lane, out, residual, epilogue, w.m, tok0, w.tokens, w.row_base + wave * 64);
#pragma unroll
        for (int b = 0; b < kTiles; b += 4) {
#pragma unroll
            for (int i = 0; i < 16; ++i) asm volatile("" : "+a"(acc[i & 3][b + (i >> 2)]));  // (read here, not ahead of it)
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                            *wide_piece(mine, lane, t, v) = f32x4{acc[0][b + t][v], acc[1][b + t][v], acc[2][b + t][v], acc[3][b + t][v]};
            __builtin_amdgcn_sched_barrier(0);
            wide_store(o, mine, lane);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}
// Consecutive tiles - the token tiles of a few row tiles - to an XCD, as in gemm_wide.hip.
__device__ __forceinline__ int wide_place()
{
    const int grid = (int)gridDim.x, xcd = (int)blockIdx.x & 7;
    return xcd * (grid >> 3) + min(xcd, grid & 7) + ((int)blockIdx.x >> 3);
}

template <int NT, bool KTAIL, bool BLK>
__global__ __launch_bounds__(kWideThreads, 1) void gemm_wide_whole_kernel(const uint8_t *a_q, const void *a_x, const float *a_code, const float *a_absmax,
                                                                          int a_m, int a_n, int a_k, int a_width, int a_tok_tiles, void *a_out, int a_epilogue,
                                                                          const void *a_residual, int a_blk_shift)
{
    extern __shared__ __align__(16) unsigned char smem[];  // the byte-pair table at LDS address 0, three stages of activations
    const int tile = wide_place(), row_tile = tile / a_tok_tiles, tok0 = (tile - row_tile * a_tok_tiles) * a_width;
    WideTile w;
    w.q = a_q;
    w.x = reinterpret_cast<const unsigned char *>(a_x) + (size_t)tok0 * (size_t)a_k * 2;
    w.absmax = a_absmax;
    w.m = a_m, w.k = a_k, w.row_base = row_tile * kWideRows;
    w.tokens = min(a_n - tok0, a_width);
    w.steps_total = (a_k + 63) >> 6, w.blk_shift = a_blk_shift;
    wide_whole_tile<NT, KTAIL, BLK>(w, a_code, smem, tok0, a_out, a_epilogue, a_residual);
}

// The tiles of several groups, one matrix and its tokens each.  What a tile's group needs is looked up at once: lane e reads group e's
// numbers (in the order of WideArgs: a chain of scalar loads otherwise).
template <bool KTAIL>
__global__ __launch_bounds__(kWideThreads, 1) void gemm_wide_groups_kernel(const uint8_t *a_q, const void *a_x, const float *a_code, const float *a_absmax,
                                                                           void *a_out, int a_m, int a_k, const WideGroups a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    // (the widest tiles come first: they go to the XCDs in turn, 32 at a time, so that each has its part of every width)
    const int grid = (int)gridDim.x, xcd = (int)blockIdx.x & 7, local = (int)blockIdx.x >> 3, full = grid >> 8, rest = grid & 255;
    const int lane = threadIdx.x & 63, tile = local < 32 * full ? (local >> 5) * 256 + xcd * 32 + (local & 31)
                                                                 : 256 * full + xcd * (rest >> 3) + min(xcd, rest & 7) + local - 32 * full;
    const int tile_end = a.tile_end[lane], begin = a.tok_begin[lane], count = a.tok_count[lane], tiles = a.tok_tiles[lane], wid = a.width[lane],
              matrix = a.id[lane], tok_tiles16 = a.nt[lane];
    const int group = __builtin_popcountll(__ballot(tile_end <= tile));
    auto of = [&](int v) { return __builtin_amdgcn_readlane(v, group); };
    const int index = tile - (group > 0 ? __builtin_amdgcn_readlane(tile_end, group - 1) : 0), per_row = of(tiles), width = of(wid), id = of(matrix), nt = of(tok_tiles16);
    const int row_tile = index / per_row, first = (index - row_tile * per_row) * width, tok0 = of(begin) + first;
    WideTile w;
    w.q = a_q + (size_t)id * (size_t)(a_m >> 3) * (size_t)(a_k >> 3) * 32;
    w.x = reinterpret_cast<const unsigned char *>(a_x) + (size_t)tok0 * (size_t)a_k * 2;
    w.absmax = a_absmax + (size_t)id * (size_t)a_m;
    w.m = a_m, w.k = a_k, w.row_base = row_tile * kWideRows;
    w.tokens = min(of(count) - first, width);
    w.steps_total = (a_k + 63) >> 6, w.blk_shift = 0;
    if (nt == 16) wide_whole_tile<16, KTAIL, false>(w, a_code, smem, tok0, a_out, TUNA_EPILOGUE_NONE, nullptr);
    else if (nt == 15) wide_whole_tile<15, KTAIL, false>(w, a_code, smem, tok0, a_out, TUNA_EPILOGUE_NONE, nullptr);
    else if (nt == 14) wide_whole_tile<14, KTAIL, false>(w, a_code, smem, tok0, a_out, TUNA_EPILOGUE_NONE, nullptr);
    else if (nt == 13) wide_whole_tile<13, KTAIL, false>(w, a_code, smem, tok0, a_out, TUNA_EPILOGUE_NONE, nullptr);
    else if (nt == 12) wide_whole_tile<12, KTAIL, false>(w, a_code, smem, tok0, a_out, TUNA_EPILOGUE_NONE, nullptr);
    else if (nt == 11) wide_whole_tile<11, KTAIL, false>(w, a_code, smem, tok0, a_out, TUNA_EPILOGUE_NONE, nullptr);
    else if (nt == 10) wide_whole_tile<10, KTAIL, false>(w, a_code, smem, tok0, a_out, TUNA_EPILOGUE_NONE, nullptr);
    else if (nt == 9) wide_whole_tile<9, KTAIL, false>(w, a_code, smem, tok0, a_out, TUNA_EPILOGUE_NONE, nullptr);
    else wide_whole_tile<8, KTAIL, false>(w, a_code, smem, tok0, a_out, TUNA_EPILOGUE_NONE, nullptr);
}

template <int NT>
hipError_t launch(const WideArgs &a, bool scale_blocks, hipStream_t stream)
{
    static OptInFlag done[16][3];
    const bool ktail = a.k % 64 != 0;
    if (scale_blocks && ktail) return hipErrorInvalidConfiguration;
    const auto fn = scale_blocks ? gemm_wide_whole_kernel<NT, false, true> : ktail ? gemm_wide_whole_kernel<NT, true, false> : gemm_wide_whole_kernel<NT, false, false>;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 16) return hipErrorInvalidDevice;
    if ((e = ensure_lds_opt_in(done[dev][scale_blocks ? 2 : ktail], reinterpret_cast<const void *>(fn))) != hipSuccess) return e;
    hipLaunchKernelGGL(fn, dim3((unsigned)a.tiles), dim3(kWideThreads), wide_lds_bytes(), stream, a.q, a.x, a.code, a.absmax, a.m, a.g.tok_count[0], a.k,
                       a.g.width[0], a.g.tok_tiles[0], a.out, a.epilogue, a.residual, a.blk_shift);
    return hipGetLastError();
}
}  // namespace

hipError_t launch_gemm_wide_whole(const WideArgs &a, bool scale_blocks, hipStream_t stream)
{
    if (a.n_groups > 1) {
        static OptInFlag done[16][2];
        const bool ktail = a.k % 64 != 0;
        const auto fn = ktail ? gemm_wide_groups_kernel<true> : gemm_wide_groups_kernel<false>;
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        if (dev < 0 || dev >= 16) return hipErrorInvalidDevice;
        if ((e = ensure_lds_opt_in(done[dev][ktail], reinterpret_cast<const void *>(fn))) != hipSuccess) return e;
        hipLaunchKernelGGL(fn, dim3((unsigned)a.tiles), dim3(kWideThreads), wide_lds_bytes(), stream, a.q, a.x, a.code, a.absmax, a.out, a.m, a.k, a.g);
        return hipGetLastError();
    }
    switch (a.g.nt[0]) {
    case 8: return launch<8>(a, scale_blocks, stream);
    case 9: return launch<9>(a, scale_blocks, stream);
    case 10: return launch<10>(a, scale_blocks, stream);
    case 11: return launch<11>(a, scale_blocks, stream);
    case 12: return launch<12>(a, scale_blocks, stream);
    case 13: return launch<13>(a, scale_blocks, stream);
    case 14: return launch<14>(a, scale_blocks, stream);
    case 15: return launch<15>(a, scale_blocks, stream);
    default: return launch<16>(a, scale_blocks, stream);
    }
}

}  // namespace tuna
