// Packed 4-bit weights -> fp16 [m, k] row-major, for gfx950.
//
// Replaces dequantize_4bit / dequantize_wrapper (kernel.cu:3158-3253).  The op is a
// pure stream (k*m/2 bytes in, 2*k*m bytes out), so the design is about HBM
// transactions only:
//   * a wave reads 1 KB of one block row with one global_load_dwordx4 per lane
//     (lane l: block column kb0 + l/2, rows 4*(l%2) .. +3), nontemporal;
//   * a dword is one weight row x 8 consecutive k, i.e. 16 bytes of output; lanes of
//     equal parity write 512 contiguous bytes per output row, nontemporal.  No LDS
//     transpose is needed (the reference needs one because its lanes own single bytes,
//     kernel.cu:3218-3240);
//   * decode: 16-entry fp32 (or fp16) table in LDS - all lanes hit 16 dwords in 16
//     distinct banks, equal addresses broadcast, so it is conflict free - then
//     fp32 multiply + round (TUNA_DECODE_DEQUANT, kernel.cu:3222-3228) or an fp16
//     multiply (TUNA_DECODE_GEMM, kernel.cu:2178-2192).
#include "tuna_internal.h"
#include "quantize_div.hpp"

#include <type_traits>

namespace tuna {

typedef _Float16 f16;
typedef f16 f16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kDqUnroll = 4;  // 1 KB chunks per wave

// BLK: one scale per `bs` consecutive weights of a row, absmax [m, k/bs] (the layout the reference's
// quantizer writes for block_size < k, test.py:15-17); otherwise one scale per row.
template <int DEC, bool BLK>
__global__ __launch_bounds__(256) void dequant_kernel(const uint8_t *__restrict__ q,
                                                      const float *__restrict__ absmax,
                                                      const float *__restrict__ code,
                                                      f16 *__restrict__ out, int m, int k, int bs)
{
    __shared__ float cf[16];
    __shared__ f16 ch[16];
    const int tid = threadIdx.x;
    if (tid < 16) {
        cf[tid] = code[tid];
        ch[tid] = (f16)code[tid];
    }
    __syncthreads();
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int kb_total = k >> 3;
    const int mb = blockIdx.y * 4 + wave;
    if (mb >= (m >> 3)) return;
    const int half = lane & 1;
    const int kb_lane = blockIdx.x * (32 * kDqUnroll) + (lane >> 1);
    const int nblk = BLK ? k / bs : 1;

    float s32[4];
    f16 s16[4];
    if constexpr (!BLK) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            s32[j] = absmax[mb * 8 + half * 4 + j];
            s16[j] = (f16)s32[j];
        }
    }
    const uint8_t *src = q + ((size_t)mb * kb_total) * 32 + half * 16;
    u32x4 w[kDqUnroll];
#pragma unroll
    for (int u = 0; u < kDqUnroll; ++u) {
        const int kb = kb_lane + u * 32;
        if (kb < kb_total) w[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(src + (size_t)kb * 32));
    }
#pragma unroll
    for (int u = 0; u < kDqUnroll; ++u) {
        const int kb = kb_lane + u * 32;
        if (kb >= kb_total) continue;
        if constexpr (BLK) {
            const int blk = (kb * 8) / bs;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                s32[j] = absmax[(size_t)(mb * 8 + half * 4 + j) * nblk + blk];
                s16[j] = (f16)s32[j];
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t d = w[u][j];
            f16x8 r;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                // column e of the row sits at bit 8*(e/2) + 4*(1 - e%2)  (test.py:58-65)
                const uint32_t nib = (d >> (8 * (e >> 1) + 4 * (1 - (e & 1)))) & 15u;
                if constexpr (DEC == TUNA_DECODE_DEQUANT) r[e] = (f16)(cf[nib] * s32[j]);
                else r[e] = ch[nib] * s16[j];
            }
            f16 *dst = out + (size_t)(mb * 8 + half * 4 + j) * k + (size_t)kb * 8;
            __builtin_nontemporal_store(r, reinterpret_cast<f16x8 *>(dst));
        }
    }
}

hipError_t launch_dequant(const uint8_t *q, const float *absmax, const float *code, void *out,
                          int m, int k, int bs, int decode, hipStream_t stream)
{
    const int kb_total = k >> 3;
    dim3 grid((kb_total + 32 * kDqUnroll - 1) / (32 * kDqUnroll), ((m >> 3) + 3) / 4, 1);
    f16 *o = reinterpret_cast<f16 *>(out);
    if (bs == k) {
        if (decode == TUNA_DECODE_DEQUANT)
            hipLaunchKernelGGL((dequant_kernel<TUNA_DECODE_DEQUANT, false>), grid, dim3(256), 0, stream, q, absmax, code, o, m, k, bs);
        else
            hipLaunchKernelGGL((dequant_kernel<TUNA_DECODE_GEMM, false>), grid, dim3(256), 0, stream, q, absmax, code, o, m, k, bs);
    } else {
        if (decode == TUNA_DECODE_DEQUANT)
            hipLaunchKernelGGL((dequant_kernel<TUNA_DECODE_DEQUANT, true>), grid, dim3(256), 0, stream, q, absmax, code, o, m, k, bs);
        else
            hipLaunchKernelGGL((dequant_kernel<TUNA_DECODE_GEMM, true>), grid, dim3(256), 0, stream, q, absmax, code, o, m, k, bs);
    }
    return hipGetLastError();
}

// fp16 weights [m, k] -> packed 4-bit codes + absmax: the device form of the reference harness's
// quantize_blockwise_dynamic_4bit (test.py:7-68).  Same arithmetic: absmax = max |w| over a block of
// `bs` consecutive weights of a row as fp32 (bs == k: one scale per row, what the kernels of the
// reference run); normalized = fp32(w) / absmax with an fp32 division (test.py:41, fp16 / fp32
// promotes to fp32); index = argmin_j |normalized - code[j]| in fp32, first index on ties
// (torch.argmin, test.py:50-53); nibble packing of test.py:55-65.  A block of zeros gets index 0: the
// reference divides by zero there, every candidate distance is NaN, and torch.argmin over an all-NaN
// column returns index 0.
//
// A wave works on 8 weight rows x 256 columns (a "quad": four 16-byte loads per lane, each 128 contiguous bytes of
// every row).  The eight lanes of a row are neighbours, so the maximum over a block of up to 64 weights is three DPP
// steps and one over 128 or 256 the maximum over the lane's own registers; with one scale per row the workgroup's eight
// waves share a block row and exchange their maxima through LDS (one barrier; the row's weights stay in registers up to
// k = 16384, beyond that a second pass reads them again).  A lane's four dwords (one row each, 8 consecutive k) are
// turned against the lanes of the other rows with permlane swaps: it then holds 4 rows of one block column, 16 bytes of
// the packed layout, and the wave stores 1 KB contiguous.  Neither the weights nor the records pass through LDS, so that
// blocked quantization has no barrier at all.
// For a codebook that is sorted with gaps wide enough that fp32 rounding cannot reorder distances, the
// nearest entry is found from the 15 decision boundaries between neighbouring entries (each the smallest fp32 value
// the argmin gives to the upper entry, found by bisection with the argmin's own arithmetic once per wave) - the
// argmin's result, since |nv - c| is monotonic in c on either side of nv; any other codebook takes the 16 comparisons.
// The division by the block maximum is a multiply by its refined reciprocal and one fused correction.
//
// What bounds it: at 14336 x 4096 with blocks of 64 (151 MB of traffic) the vector ALUs, busy 90 % of the launch at 1.80 GHz
// with sixteen instructions a weight: 62.5 -> 32.3 us against the version that passed block rows through LDS, with one scale
// per row 53.1 -> 32.1; 8192 x 28672 in blocks of 64 224 -> 114 us (5.3 TB/s), 4096 x 14336 per row 56 -> 35; 3 us before the
// first table is complete.
// Nearest entry of a sorted codebook: bnd[i] (i = 0..14) is the smallest binary32 value that the
// argmin assigns to entry i + 1 rather than entry i, so the index is the number of boundaries <= nv:
// a 4-step binary search, as a tree of selects over the 15 values (uniform, held in registers).
__device__ __forceinline__ uint32_t nearest_sorted(float nv, const float (&b)[16])
{
    const bool b3 = nv >= b[7];
    const float t2 = b3 ? b[11] : b[3];
    const float u3 = b3 ? b[13] : b[5], v3 = b3 ? b[9] : b[1];
    const float p4 = b3 ? b[14] : b[6], q4 = b3 ? b[12] : b[4], r4 = b3 ? b[10] : b[2], s4 = b3 ? b[8] : b[0];
    const bool b2 = nv >= t2;
    const float t3 = b2 ? u3 : v3;
    const float x4 = b2 ? p4 : r4, y4 = b2 ? q4 : s4;
    const bool b1 = nv >= t3;
    const float t4 = b1 ? x4 : y4;
    const bool b0 = nv >= t4;
    return (b3 ? 8u : 0u) + (b2 ? 4u : 0u) + (b1 ? 2u : 0u) + (b0 ? 1u : 0u);  // a NaN nv ends at 0 like the argmin
}

// The same count of boundaries <= nv without the search: the quotients lie in [-1, 1], cut into 64 buckets
// of 1/32; when no two boundaries share a bucket, a bucket knows how many boundaries lie below it and the one
// boundary (if any) inside it, and the index is that count plus one comparison.  The bucket is monotonic in
// nv (a fused multiply-add, a truncation), so every value of a lower bucket is below the boundary
// of a higher one and vice versa: the result is the binary search's for every nv, NaN included (bucket 0, the
// comparison false, index 0).  One LDS table of {boundary, count} pairs in the lane-private layout of the
// GEMM's decode table (entry e of lane l at (e << 9) | (l << 3): one 8-byte read, no bank conflicts whatever
// the data).
constexpr int kQuantBuckets = 65;
constexpr int kQuantTabBytes = kQuantBuckets * 512;  // per bucket and lane: fp32 boundary (+inf if none), boundaries below it
typedef __attribute__((address_space(3))) unsigned char lds_u8;
typedef uint32_t quant_u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) quant_u32x2 lds_pair;

// (nv * 16384 + 16384) / 2^24 plus a half: the fp32 pattern's low bits are nv * 16384 + 16384 as an integer, its multiples
// of 512 the bucket - which is the entry's offset.  Clamped to [0, 1] (an output modifier of the fused multiply-add, no
// instruction of its own): a NaN becomes 0 whatever its payload - which an fp16 weight's NaN carries through the division
// and which would otherwise show in those bits - and so goes to bucket 0, as infinities do.
__device__ __forceinline__ uint32_t bucket_bits(float nv)
{
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_fmed3f(__builtin_fmaf(nv, 0x1p-10f, 0.5f + 0x1p-10f), 0.0f, 1.0f)) & 0xfe00u;
}

__device__ __forceinline__ quant_u32x2 bucket_entry(float nv, uint32_t tab_lane)
{
    return *reinterpret_cast<const lds_pair *>((uintptr_t)(bucket_bits(nv) | tab_lane));
}

__device__ __forceinline__ uint32_t nearest_any(float nv, const float (&c)[16])
{
    float bd = fabsf(__fsub_rn(nv, c[0]));
    uint32_t best = 0;
#pragma unroll
    for (int i = 1; i < 16; ++i) {
        const float dd = fabsf(__fsub_rn(nv, c[i]));
        if (dd < bd) {
            bd = dd;
            best = i;
        }
    }
    return best;
}

// Smallest binary32 v in [lo, hi] for which the argmin prefers hi: |v - hi| < |v - lo| in fp32
// arithmetic (ties keep the lower index).  The predicate is monotonic in v (both rounded differences
// are), so a bisection over the bit patterns finds it; lo < hi finite, and it holds at v = hi.  Two probes
// 64 patterns either side of the rounded midpoint come first: the boundary lies between them unless the
// midpoint is tiny against the gap, and the bisection then takes 7 steps instead of 31.
__device__ inline float decision_boundary(float lo, float hi)
{
    auto key = [](float f) {  // order-preserving map of finite floats to integers (both zeros -> 0)
        const int32_t i = __builtin_bit_cast(int32_t, f);
        return i < 0 ? -(i & 0x7fffffff) : i;
    };
    auto unkey = [](int32_t k) {
        const uint32_t i = k < 0 ? (uint32_t)(-k) | 0x80000000u : (uint32_t)k;
        return __builtin_bit_cast(float, i);
    };
    auto prefers_hi = [&](int32_t kv) {
        const float v = unkey(kv);
        return fabsf(__fsub_rn(v, hi)) < fabsf(__fsub_rn(v, lo));
    };
    int32_t a = key(lo), b = key(hi);  // predicate false at a (distance 0 to lo), true at b; b - a < 2^32
    const int32_t mid0 = key(0.5f * lo + 0.5f * hi);
#pragma unroll
    for (int side = -1; side <= 1; side += 2) {
        const int64_t want = (int64_t)mid0 + side * 64;
        if (want > (int64_t)a && want < (int64_t)b) {
            const int32_t p = (int32_t)want;
            if (prefers_hi(p)) b = p;
            else a = p;
        }
    }
    while ((uint32_t)b - (uint32_t)a > 1u) {
        const int32_t mid = (int32_t)((uint32_t)a + (((uint32_t)b - (uint32_t)a) >> 1));
        if (prefers_hi(mid)) b = mid;
        else a = mid;
    }
    return unkey(b);
}

// max(acc, |t|) over eight fp16 values, two at a time: the magnitudes are the bit patterns with the sign
// cleared, packed maxima never round, and the conversion to fp32 at the end is exact - the maximum the
// reference forms in fp32, at one instruction per weight.  (NaN is skipped by either form of the maximum.)
typedef f16 quant_f16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ quant_f16x2 pk_absmax8(quant_f16x2 acc, f16x8 t)
{
    const u32x4 b = __builtin_bit_cast(u32x4, t) & 0x7fff7fffu;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t pair = b[i];  // (a bit_cast of the vector element itself reads element 0)
        acc = __builtin_elementwise_max(acc, __builtin_bit_cast(quant_f16x2, pair));
    }
    return acc;
}
__device__ __forceinline__ float pk_absmax_value(quant_f16x2 acc) { return fmaxf((float)acc[0], (float)acc[1]); }

// The packed dword of 8 consecutive weights of a row.  MODE 0: bucket table; 1: binary search over the boundaries
// (c); 2: the 16 comparisons with the codebook (c).  A block of zeros (y is NaN) gets index 0 throughout.
template <int MODE>
__device__ __forceinline__ uint32_t quant_dword(f16x8 t, float amax, uint32_t tab_lane, const float (&c)[16])
{
    const float y = refined_rcp(amax);
    const u32x4 w = __builtin_bit_cast(u32x4, t);
    uint32_t d = 0;
#pragma unroll
    for (int p = 3; p >= 0; --p) {  // byte p: columns 2p (high nibble) and 2p + 1
        const uint32_t pair = w[p];
        const float n0 = div_by_block_max<0>(pair, amax, y), n1 = div_by_block_max<1>(pair, amax, y);
        if constexpr (MODE == 0) {
            const quant_u32x2 e0 = bucket_entry(n0, tab_lane), e1 = bucket_entry(n1, tab_lane);
            const uint32_t b0 = e0[0], b1 = e1[0];
            d = (d << 4) + e0[1] + (n0 >= __builtin_bit_cast(float, b0) ? 1u : 0u);
            d = (d << 4) + e1[1] + (n1 >= __builtin_bit_cast(float, b1) ? 1u : 0u);
        } else if constexpr (MODE == 1) {
            d = (d << 4) | nearest_sorted(n0, c);
            d = (d << 4) | nearest_sorted(n1, c);
        } else {
            d = (d << 4) | nearest_any(n0, c);
            d = (d << 4) | nearest_any(n1, c);
        }
    }
    return d;
}

template <int CTRL>
__device__ __forceinline__ float dpp_max(float v)
{
    const int i = __builtin_bit_cast(int, v);
    return fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(i, i, CTRL, 0xf, 0xf, true)));
}
constexpr int kDppXor1 = 0xb1, kDppXor2 = 0x4e, kDppHalfMirror = 0x141;  // (the last: lane i of 8 <-> 7 - i)

// Exchanges register index bits with lane bits 5 and 4: d[i] of lane (b5, b4) <-> d[2 b5 + b4] of lane (i1, i0).
__device__ __forceinline__ void turn4(uint32_t (&d)[4])
{
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const auto r = __builtin_amdgcn_permlane32_swap(d[i], d[i + 2], false, false);
        d[i] = r[0];
        d[i + 2] = r[1];
    }
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
        const auto r = __builtin_amdgcn_permlane16_swap(d[i], d[i + 1], false, false);
        d[i] = r[0];
        d[i + 1] = r[1];
    }
}

constexpr int kQuadCols = 256;  // columns of a quad

// NQ == 0: blocks of up to 256 weights (bs a power of two), the waves walk the quads; NQ > 0: one scale per row, NQ quads
// per wave in registers (k <= 256 NQ WAVES); NQ < 0: one scale per row, two passes.
template <int NQ, int WAVES>
__global__ __launch_bounds__(WAVES * 64, NQ >= 2 ? 4 : 6)
void quantize_kernel(const f16 *__restrict__ w, const float *__restrict__ code, uint32_t *__restrict__ q32,
                     float *__restrict__ absmax, int m, int k, int bs)
{
    // the bucket table from LDS address 0 on (nothing here is statically allocated: an entry's offset is or-ed to the
    // lane's address), then the waves' maxima
    extern __shared__ __align__(16) unsigned char qtab[];
    float (*wave_max)[WAVES][8] = reinterpret_cast<float (*)[WAVES][8]>(qtab + kQuantTabBytes);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 7;  // column group of the load
    const int r8 = ((lane >> 4) & 3) | ((lane >> 1) & 4);  // weight row of the load: lane bits 5, 4 -> row bits 1, 0
    const int kb_total = k >> 3;
    const int quads = (k + kQuadCols - 1) / kQuadCols;  // of a block row
    const int rows8 = m >> 3;

    auto load_quad = [&](f16x8 (&v)[4], int mb, int g) {
        const f16 *src = w + (size_t)(mb * 8 + r8) * k + g * kQuadCols + j * 8;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
            if (g * kQuadCols + i * 64 + j * 8 < k) v[i] = __builtin_nontemporal_load(reinterpret_cast<const f16x8 *>(src + i * 64));
        }
    };
    // the first weights are on their way while the table is built
    constexpr int NV = NQ > 0 ? NQ : 1;
    f16x8 v[NV][4];
    const int n_waves = (int)gridDim.x * WAVES;
    int item = NQ == 0 ? (int)blockIdx.x * WAVES + wave : (int)blockIdx.x;  // quad, or block row
    const int items = NQ == 0 ? rows8 * quads : rows8;
    if constexpr (NQ == 0) {
        if (item < items) load_quad(v[0], item / quads, item % quads);
    } else if constexpr (NQ > 0) {
#pragma unroll
        for (int n = 0; n < NQ; ++n) load_quad(v[n], item, wave + n * WAVES);
    }

    // lane i of every wave: codebook entry i, the boundary above it
    const float mine = code[lane & 15];
    const float next = __shfl_down(mine, 1, 64);
    auto lane_value = [](float x, int i) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), i)); };
    // sorted, and every gap far above the rounding of a difference (|nv| <= 1, so a difference is
    // at most 1 + max|c| and its rounding error below 2^-23 of that)
    const float cmax = fmaxf(fabsf(lane_value(mine, 0)), fabsf(lane_value(mine, 15)));
    const float thr = (1.0f + cmax) * 9.5367431640625e-7f;  // 2^-20
    const bool fast = (__ballot(next - mine >= thr) & 0x7fffu) == 0x7fffu && cmax < 3.0e38f;
    float bnd = 0.f;
    bool tabled = false;
    if (fast) {
        if (lane < 15) bnd = decision_boundary(mine, next);
        // the bucket table, if every boundary is finite and has a bucket of its own
        const int bucket = (int)bucket_bits(bnd);
        const int below = __shfl_up(bucket, 1, 64);
        const bool ok = fabsf(bnd) < 3.0e38f && (lane == 0 || bucket > below);
        tabled = (__ballot(ok) & 0x7fffu) == 0x7fffu;
        // (outside [-1, 1] no quotient lies, and the patterns would wrap)
        tabled = tabled && (__ballot(fabsf(bnd) <= 1.0f) & 0x7fffu) == 0x7fffu;
        if (tabled) {
            for (int e = wave; e < kQuantBuckets; e += WAVES) {
                const uint64_t at = __ballot(bucket == (e << 9)) & 0x7fffu, under = __ballot(bucket < (e << 9)) & 0x7fffu;
                const float b = at ? lane_value(bnd, __builtin_ctzll(at | 0x8000u)) : __builtin_inff();
                const quant_u32x2 pair = {__builtin_bit_cast(uint32_t, b), (uint32_t)__builtin_popcountll(under)};
                *reinterpret_cast<quant_u32x2 *>(qtab + (e << 9) + (lane << 3)) = pair;
            }
        }
    }
    __syncthreads();
    const uint32_t tab_lane = (uint32_t)(uintptr_t)(lds_u8 *)qtab + ((uint32_t)lane << 3);

    // The nearest-entry rule is a compile-time choice (the loops share nothing but their registers: the table path must
    // not carry the 15 boundaries of the search).
    auto run = [&](auto mode_tag) {
        constexpr int MODE = decltype(mode_tag)::value;
        float c[16];  // MODE 1: the boundaries; MODE 2: the codebook
#pragma unroll
        for (int i = 0; i < 16; ++i) c[i] = MODE == 1 ? lane_value(bnd, i) : MODE == 2 ? lane_value(mine, i) : 0.f;
        auto pack_quad = [&](const f16x8 (&t)[4], const float (&am)[4], int mb, int g) {
            uint32_t d[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                d[i] = quant_dword<MODE>(t[i], am[i], tab_lane, c);
                __builtin_amdgcn_sched_barrier(0);  // (all four at once would not fit in the registers)
            }
            turn4(d);  // now rows 4 * (lane bit 3) + 0 .. 3 of block column 8 * (lane bits 5, 4) + j of the quad
            const int kb = g * (kQuadCols / 8) + (lane >> 4) * 8 + j;
            if (kb < kb_total)
                *reinterpret_cast<u32x4 *>(q32 + ((size_t)mb * kb_total + kb) * 8 + ((lane >> 3) & 1) * 4) = u32x4{d[0], d[1], d[2], d[3]};
        };
        const quant_f16x2 zero2 = quant_f16x2{(f16)0.f, (f16)0.f};
        if constexpr (NQ == 0) {
            const int lanes_blk = bs >> 3;  // 16-byte groups that share a scale: 1, 2, 4 .. 32
            const int nblk = k / bs;
            for (; item < items; item += n_waves) {
                const int mb = item / quads, g = item % quads;
                f16x8 vn[4];
                const int after = item + n_waves;
                if (after < items) load_quad(vn, after / quads, after % quads);
                float am[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) am[i] = pk_absmax_value(pk_absmax8(zero2, v[0][i]));
                if (lanes_blk > 1) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) am[i] = dpp_max<kDppXor1>(am[i]);
                }
                if (lanes_blk > 2) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) am[i] = dpp_max<kDppXor2>(am[i]);
                }
                if (lanes_blk > 4) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) am[i] = dpp_max<kDppHalfMirror>(am[i]);
                }
                if (lanes_blk > 8) {
                    am[0] = am[1] = fmaxf(am[0], am[1]);
                    am[2] = am[3] = fmaxf(am[2], am[3]);
                }
                if (lanes_blk > 16) am[0] = am[1] = am[2] = am[3] = fmaxf(am[0], am[2]);
                float *scales = absmax + (size_t)(mb * 8 + r8) * nblk;
                if (lanes_blk == 8) {  // lane i of the row's eight stores the i-th of the four scales
                    const float s = j & 2 ? (j & 1 ? am[3] : am[2]) : (j & 1 ? am[1] : am[0]);
                    if (j < 4 && g * 4 + j < nblk) scales[g * 4 + j] = s;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int kb = g * (kQuadCols / 8) + i * 8 + j;
                        if (kb < kb_total && (kb & (lanes_blk - 1)) == 0) scales[kb / lanes_blk] = am[i];
                    }
                }
                pack_quad(v[0], am, mb, g);
#pragma unroll
                for (int i = 0; i < 4; ++i) v[0][i] = vn[i];
            }
        } else {
            constexpr bool AHEAD = NQ > 0 && NQ <= 2;  // registers for two block rows
            int flip = 0;
            for (; item < items; item += (int)gridDim.x) {
                f16x8 vn[AHEAD ? NQ : 1][4];
                if constexpr (AHEAD) {
                    if (item + (int)gridDim.x < items) {
#pragma unroll
                        for (int n = 0; n < NQ; ++n) load_quad(vn[n], item + (int)gridDim.x, wave + n * WAVES);
                    }
                }
                quant_f16x2 pm = zero2;
                if constexpr (NQ < 0) {
                    for (int g = wave; g < quads; g += WAVES) {
                        load_quad(v[0], item, g);
#pragma unroll
                        for (int i = 0; i < 4; ++i) pm = pk_absmax8(pm, v[0][i]);
                    }
                }
#pragma unroll
                for (int n = 0; n < NQ; ++n)
#pragma unroll
                    for (int i = 0; i < 4; ++i) pm = pk_absmax8(pm, v[n][i]);
                float row_max = dpp_max<kDppHalfMirror>(dpp_max<kDppXor2>(dpp_max<kDppXor1>(pk_absmax_value(pm))));
                if (j == 0) wave_max[flip][wave][r8] = row_max;
                __syncthreads();  // (two buffers: a wave writes one only after every wave passed the barrier in between)
#pragma unroll
                for (int o = 0; o < WAVES; ++o) row_max = fmaxf(row_max, wave_max[flip][o][r8]);
                flip ^= 1;
                if (wave == 0 && j == 0) absmax[item * 8 + r8] = row_max;
                const float am[4] = {row_max, row_max, row_max, row_max};
#pragma unroll
                for (int n = 0; n < NQ; ++n) {
                    if (wave + n * WAVES < quads) pack_quad(v[n], am, item, wave + n * WAVES);
                    if constexpr (AHEAD) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) v[n][i] = vn[n][i];
                    } else if (item + (int)gridDim.x < items) {
                        load_quad(v[n], item + (int)gridDim.x, wave + n * WAVES);
                    }
                }
                if constexpr (NQ < 0) {
                    for (int g = wave; g < quads; g += WAVES) {
                        load_quad(v[0], item, g);
                        pack_quad(v[0], am, item, g);
                    }
                }
            }
        }
    };
    if (tabled) run(std::integral_constant<int, 0>{});
    else if (fast) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 2>{});
}

hipError_t launch_quantize(const void *w, const float *code, void *q, float *absmax, int m, int k, int bs, hipStream_t stream)
{
    const f16 *wp = static_cast<const f16 *>(w);
    uint32_t *qp = static_cast<uint32_t *>(q);
    // as many workgroups as fit beside their tables and registers, which then walk the quads or block rows: the
    // tables are built once per workgroup
    int dev = 0, cus = 0;
    hipError_t e = device_cus(&dev, &cus);
    if (e != hipSuccess) return e;
    const int rows8 = m / 8;
    const bool blocked = bs <= kQuadCols && (bs & (bs - 1)) == 0;
    const int waves = blocked || k <= 8192 ? 8 : 16;
    const int work = blocked ? (int)(((int64_t)rows8 * ((k + kQuadCols - 1) / kQuadCols) + waves - 1) / waves) : rows8;
    const int per_cu = blocked || k <= 2048 ? 3 : k <= 8192 ? 2 : 1;
    const dim3 grid((unsigned)(work < per_cu * cus ? work : per_cu * cus)), block((unsigned)waves * 64);
    const size_t lds = (size_t)kQuantTabBytes + 2 * waves * 8 * sizeof(float);
    if (blocked) hipLaunchKernelGGL((quantize_kernel<0, 8>), grid, block, lds, stream, wp, code, qp, absmax, m, k, bs);
    else if (k <= 2048) hipLaunchKernelGGL((quantize_kernel<1, 8>), grid, block, lds, stream, wp, code, qp, absmax, m, k, bs);
    else if (k <= 4096) hipLaunchKernelGGL((quantize_kernel<2, 8>), grid, block, lds, stream, wp, code, qp, absmax, m, k, bs);
    else if (k <= 8192) hipLaunchKernelGGL((quantize_kernel<4, 8>), grid, block, lds, stream, wp, code, qp, absmax, m, k, bs);
    else if (k <= 16384) hipLaunchKernelGGL((quantize_kernel<4, 16>), grid, block, lds, stream, wp, code, qp, absmax, m, k, bs);
    else hipLaunchKernelGGL((quantize_kernel<-1, 16>), grid, block, lds, stream, wp, code, qp, absmax, m, k, bs);
    return hipGetLastError();
}

}  // namespace tuna
