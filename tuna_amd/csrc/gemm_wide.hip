// FP16-activation x 4-bit-codebook-weight GEMM for MANY tokens, 256 weight rows x 256 tokens per workgroup, one wave per
// SIMD (4 waves of 512 registers), every wave decoding the weights it multiplies straight into the MFMA's registers.
//
//   * A wave owns 64 rows x all 256 tokens of the tile: 4 x 16 tiles of v_mfma_f32_16x16x32_f16, whose 256 accumulator
//     registers sit in the AGPR half of the register file.  A 16-byte load of the packed layout is four rows x 8 k of a
//     lane, one dword of it - eight byte pairs through the decode table, scaled - IS a lane's weight operand of one
//     MFMA: no weight tile in LDS, and every weight is decoded once per 256 tokens.
//   * Only the activations go through LDS, in a ring of three k-steps of [token][64 k] (128-byte rows, 16-byte slots
//     XOR-swizzled with token & 7: no bank conflicts), 32 KB each beside the decode table's 64 KB.  They are loaded into LDS
//     directly (lds_dma.hpp): through registers they took the path that LDS reads return their data over.
//   * The work of a k-step is spread evenly between its 128 MFMAs: per token tile (4 MFMAs) one fragment read, one table
//     read, one address, one scaling; the loads behind the step's one barrier.
//
// What bounds it: in the loop the matrix pipes, busy 75 % of the cycles at the 1.68 GHz that the power limit leaves (with the
// activations loaded into registers and stored to LDS 68 % at 1.72 GHz); around it the start and end of a tile, 12 us by
// wide_time's fit, which nothing overlaps - one workgroup per compute unit - and compute units without a tile in the last round.
// The power limit alone explains less: torch's fp16 product of the first two shapes takes 187 and 367 us on the card of these
// figures.  8192 x 8192 at 2048 tokens 241 -> 224 us, 28672 x 4096 at 2000 tokens 403 -> 381, 4096 x 14336 at 2000 200 -> 190,
// 6144 x 4096 at 2000 101 -> 93, 8192 x 8200 at 4096 468 -> 420 (one card, launch loop).
//
// Tiles of 1 .. 128 tokens (the last of a group) run the same steps with half the token tiles.  How tiles become
// workgroups is plan_gemm_wide's choice.  KTAIL: k is any multiple of 8 - the slots of the last k-step beyond k load
// the last slot inside k (no access leaves a row), and their activations are zeros.  BLK: one scale per block
// of a row.  Decode and rounding are those of the other kernels (bit-identical to kernel.cu:2178-2192); an unshared
// tile's sums are the same products in the same order as the 16 x 16 x 32 variants of gemm_tiled.hip.
#include "lds_dma.hpp"

namespace tuna {

constexpr int kWideThreads = 256;
constexpr int kWideRows = 256, kWideTokens = 256;
constexpr int kWideStage = kWideTokens * 128;  // a k-step of 64 of the token tile

// One token tile of a row tile's k range [s0, s1) (in k-steps of 64), accumulated onto acc.  NT token tiles of 16.
struct WideTile {
    const uint8_t *q;      // the group's weights
    const unsigned char *x;  // first activation row of the token tile
    const float *absmax;   // the group's scales
    int m, k;              // rows of the group, reduction length
    int row_base;          // first row of the tile in the group
    int tokens;            // tokens of the tile (1 .. 16 NT)
    int steps_total, blk_shift;
};

template <int NT, bool KTAIL, bool BLK>
__device__ __forceinline__ void wide_steps(f32x4 (&acc)[4][16], const WideTile &w, unsigned char *xs, int s0, int s1)
{
    constexpr int XP = NT / 2;  // 16-byte pieces of a step's activations a thread stages
    constexpr int FB = 8;       // token fragments on their way (the ring: 2 NT tiles of a step divide into it)
    constexpr int LPT = 16 / NT; // table reads per token tile and half
    constexpr int T_NEXT = 13 / LPT; // the token tile from which on the table reads of a half are the one after next's
    static_assert(NT == 16 || NT == 8, "token tiles");
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i16 = lane & 15, g = lane >> 4;
    const uint32_t lane4 = (uint32_t)lane << 2;
    const int kb_total = w.k >> 3;

    // weights: lane (i16, g) loads 16 bytes = rows 4 i16 .. + 3 of the wave's 64, block column 4 h + g of half h of a
    // step (rows beyond the matrix are clamped: their products are never stored)
    const int row_w = w.row_base + wave * 64;
    const uint32_t a_off = tile_weight_lane(tid, ((w.m - w.row_base) >> 3) - 1, kb_total);
    // activations: piece i of a thread is token tid / 8 + 32 i (tokens beyond the tile's read its last), the 8-k slot that
    // belongs at place tid % 8 of that token's row of the stage
    const int x_slot = (tid & 7) ^ ((tid >> 3) & 7);
    uint32_t x_off[XP];
#pragma unroll
    for (int i = 0; i < XP; ++i) x_off[i] = ((uint32_t)min((tid >> 3) + 32 * i, w.tokens - 1) * (uint32_t)w.k + (uint32_t)x_slot * 8u) * 2u;
    const uint32_t xs_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)xs + (uint32_t)wave * 1024u;
    // KTAIL: slots of the last step beyond k load the last slot inside k, and their activations are requested out of range:
    // zeros
    const int slot_last = ((w.k >> 3) - 1) & 7;
    const uint32_t x_beyond = KTAIL && x_slot > slot_last ? 0x7fffffffu : 0u;
    const uint32_t a_back0 = KTAIL ? (uint32_t)wide_weight_back(tid, 0, slot_last) : 0u;
    const uint32_t a_back1 = KTAIL ? (uint32_t)wide_weight_back(tid, 1, slot_last) : 0u;

    const u32x4 q_rsrc = buffer_at(w.q + (size_t)(w.row_base >> 3) * kb_total * 32, (size_t)(w.m - w.row_base) * (size_t)(w.k >> 1));
    const u32x4 x_rsrc = buffer_at(w.x, (size_t)w.tokens * (size_t)w.k * 2);

    // scales of rows 4 i16 + j: one per row, or (BLK) one per block of 64 << blk_shift weights, which travel through the
    // register sets with the weights (a step lies inside one block)
    const int nblk = BLK ? w.k >> (6 + w.blk_shift) : 1;
    const float *s_base = w.absmax + (size_t)w.row_base * (size_t)nblk;
    const u32x4 s_rsrc = buffer_at(s_base, (size_t)(w.m - w.row_base) * (size_t)nblk * 4);
    uint32_t s_off[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) s_off[j] = (uint32_t)(min(row_w + 4 * i16 + j, w.m - 1) - w.row_base) * (uint32_t)nblk * 4u;
    uint32_t sq[BLK ? 2 : 1][4];
    f16x2 sc[4];
#define WIDE_SCALES(set)                                                                                      \
    _Pragma("unroll") for (int j = 0; j < 4; ++j)                                                             \
    {                                                                                                         \
        const f16 h_ = (f16)__builtin_bit_cast(float, sq[set][j]);                                            \
        sc[j] = f16x2{h_, h_};                                                                                \
    }

    u32x4 wq[2][2];   // [set][half]: packed weights of two k-steps
    const int s_last = w.steps_total - 1;
    // Requests, in an order that the waits count on: for a step the weights and scales (WL operations), then the activations
    // (XP), then the next step's weights ...  A step of a small tile is shorter than a scale's way from memory: there the scales
    // (SL) are requested as soon as their registers are free, half a step and more ahead of the weights (44160 x 13824 at 92 tokens
    // with blocks of 64 227.0 -> 221.7 us, 28672 x 4096 at 100 71.6 -> 70.6; no gain with large tiles, nor from activations requested a step earlier).
    constexpr bool EARLY = BLK && NT == 8;
    constexpr int WL = BLK ? 6 : 2, SL = EARLY ? 4 : 0;
#define WIDE_LOAD_W(set, s)                                                                                   \
    {                                                                                                         \
        const int s_ = min((s), s_last);                                                                      \
        const bool t_ = KTAIL && s_ == s_last;                                                                \
        load_async(wq[set][0], q_rsrc, t_ ? a_off - a_back0 : a_off, (uint32_t)wide_weight_uniform(s_, 0, t_, slot_last)); \
        load_async(wq[set][1], q_rsrc, t_ ? a_off - a_back1 : a_off, (uint32_t)wide_weight_uniform(s_, 1, t_, slot_last)); \
        if (BLK && !EARLY) WIDE_LOAD_S(set, s)                                                                \
    }
#define WIDE_LOAD_S(set, s)                                                                                   \
    _Pragma("unroll") for (int j = 0; j < 4; ++j) load_async(sq[set][j], s_rsrc, s_off[j], (uint32_t)min((s) >> w.blk_shift, nblk - 1) * 4u);
#define WIDE_LOAD_X(i, off, s)                                                                                \
    {                                                                                                         \
        const int s_ = min((s), s_last);                                                                      \
        load_to_lds(x_rsrc, KTAIL && s_ == s_last ? x_off[i] | x_beyond : x_off[i], (uint32_t)s_ * 128u, xs_lds + (off) + (i) * 4096u); \
    }
    // A step's weights (and scales) have arrived: at most N operations behind them are pending.
#define WIDE_ARRIVED(set, N)                                                                                  \
    asm volatile("s_waitcnt vmcnt(%2)" : "+v"(wq[set][0]), "+v"(wq[set][1]) : "n"(N));                       \
    if (BLK) asm volatile("" : "+v"(sq[set][0]), "+v"(sq[set][1]), "+v"(sq[set][2]), "+v"(sq[set][3]));

    f16x8 fa[2][4];  // decoded weights of a half: rows 4 i16 + j
    f16x8 fb[FB];
    uint32_t lt[4];  // table reads on their way
    const int swz = (g ^ (i16 & 7)) << 4;
    const unsigned char *x_frag0 = xs + i16 * 128 + swz, *x_frag1 = xs + i16 * 128 + (64 ^ swz);
#define WIDE_READ_B(slot, half, off, t) \
    fb[slot] = *reinterpret_cast<const f16x8 *>(((half) ? x_frag1 : x_frag0) + (off) + (t) * 2048);
    // table read of byte pair l (dword l / 4, byte l % 4) of a half, and its scaling (bit-identical to kernel.cu:2178-2192)
#define WIDE_LUT(l, set, half)                                                                                \
    lt[(l) & 3] = *reinterpret_cast<const lds_u32 *>(                                                         \
        (uintptr_t)__builtin_amdgcn_perm(wq[set][half][(l) >> 2], lane4, 0x0c0c0400u + 0x100u * ((l) & 3)));
#define WIDE_SCALE(l, ab)                                                                                     \
    {                                                                                                         \
        const f16x2 h_ = __builtin_bit_cast(f16x2, lt[(l) & 3]) * sc[(l) >> 2];                               \
        fa[ab][(l) >> 2][2 * ((l) & 3)] = h_[0];                                                              \
        fa[ab][(l) >> 2][2 * ((l) & 3) + 1] = h_[1];                                                          \
    }
    // (inline assembly with the accumulator pinned to the AGPR half of the register file: left to itself the register
    // allocator spreads 64 four-register accumulators over both halves and spills in the loop; an accumulator is next
    // touched 63 MFMAs later, a decoded weight is written at least four MFMAs before it is read)
#define WIDE_MFMA(ab, j, t, slot) \
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc[j][t]) : "v"(fa[ab][j]), "v"(fb[slot]));

    // Half `h` of k-step `step` (iteration `it` of the loop unrolled by two): per token tile t four MFMAs with the
    // decoded weights fa[h] and token fragment t, and between them: the fragment FB - 1 tiles on; the scaling of a byte
    // pair of the next half into fa[h ^ 1] and the table read of the pair three on.
    // Stages cur, nxt, nx2 hold steps step .. step + 2.  The barrier of a step comes where the first fragment of the
    // next step is requested: every wave has waited for its pieces of that step.  Behind it the pieces of step + 2 are
    // requested, into the stage of step - 1: its last fragments were used by every wave before that barrier.
#define WIDE_HALF(it, step, h)                                                                                \
    {                                                                                                         \
        constexpr int dset_ = (h) == 0 ? (it) : (it) ^ 1, dh_ = (h) ^ 1;                                      \
        _Pragma("unroll") for (int t = 0; t < NT; ++t)                                                        \
        {                                                                                                     \
            const int base_ = (h) * NT + t;                                                                   \
            WIDE_MFMA(h, 0, t, base_ % FB)                                                                    \
            if ((h) == 0 && t == T_NEXT) { WIDE_ARRIVED((it) ^ 1, XP + SL) } /* the table reads reach the next step */ \
            if ((h) == 1 && t == NT - FB + 1) {                                                               \
                wait_loads<WL>(); /* this wave's pieces of the next step are in LDS */                        \
                __builtin_amdgcn_s_barrier();                                                                 \
                asm volatile("" ::: "memory");                                                                \
            }                                                                                                 \
            {                                                                                                 \
                const int nt_ = base_ + FB - 1;                                                               \
                WIDE_READ_B(nt_ % FB, (nt_ / NT) & 1, nt_ >= 2 * NT ? nxt : cur, nt_ % NT)                    \
            }                                                                                                 \
            __builtin_amdgcn_sched_barrier(0);                                                                \
            WIDE_MFMA(h, 1, t, base_ % FB)                                                                    \
            if (BLK && (h) == 1 && t == 0) {                                                                  \
                WIDE_SCALES((it) ^ 1)                                                                         \
                if (EARLY) WIDE_LOAD_S((it) ^ 1, (step) + 3)                                                  \
            }                                                                                                 \
            _Pragma("unroll") for (int l = t * LPT; l < (t + 1) * LPT; ++l) {                                 \
                WIDE_SCALE(l, dh_)                                                                            \
                if (l + 3 < 16) WIDE_LUT(l + 3, dset_, dh_)                                                   \
                else WIDE_LUT(l + 3 - 16, (it) ^ 1, h)                                                        \
            }                                                                                                 \
            __builtin_amdgcn_sched_barrier(0);                                                                \
            WIDE_MFMA(h, 2, t, base_ % FB)                                                                    \
            if ((h) == 1 && t > NT - FB + 1 && (t - (NT - FB + 2)) * 2 < XP) {                                \
                WIDE_LOAD_X((t - (NT - FB + 2)) * 2, (uint32_t)nx2, (step) + 2)                               \
                WIDE_LOAD_X((t - (NT - FB + 2)) * 2 + 1, (uint32_t)nx2, (step) + 2)                           \
            }                                                                                                 \
            __builtin_amdgcn_sched_barrier(0);                                                                \
            WIDE_MFMA(h, 3, t, base_ % FB)                                                                    \
            if (t == NT - 1) {                                                                                \
                if ((h) == 0) WIDE_LOAD_W(dset_, (step) + 2)                                                  \
                if ((h) == 1) {                                                                               \
                    const int c_ = cur;                                                                       \
                    cur = nxt, nxt = nx2, nx2 = c_;                                                           \
                }                                                                                             \
            }                                                                                                 \
            __builtin_amdgcn_sched_barrier(0);                                                                \
        }                                                                                                     \
    }
    int cur = 0, nxt = kWideStage, nx2 = 2 * kWideStage;
    if (!BLK) {
#pragma unroll
        for (int j = 0; j < 4; ++j) load_async(sq[0][j], s_rsrc, s_off[j], 0u);
    }
    if (EARLY) WIDE_LOAD_S(0, s0)
    WIDE_LOAD_W(0, s0)
    __syncthreads();  // decode table complete; the previous tile's work area has been read
#pragma unroll
    for (int i = 0; i < XP; ++i) WIDE_LOAD_X(i, 0u, s0)
    if (EARLY) WIDE_LOAD_S(EARLY ? 1 : 0, s0 + 1)
    WIDE_LOAD_W(1, s0 + 1)
#pragma unroll
    for (int i = 0; i < XP; ++i) WIDE_LOAD_X(i, (uint32_t)kWideStage, s0 + 1)
    WIDE_ARRIVED(0, XP + WL)
    if (!BLK) asm volatile("" : "+v"(sq[0][0]), "+v"(sq[0][1]), "+v"(sq[0][2]), "+v"(sq[0][3]));
    WIDE_SCALES(0)
    if (EARLY) WIDE_LOAD_S(0, s0 + 2)
#pragma unroll
    for (int l = 0; l < 16; ++l) {
        WIDE_LUT(l, 0, 0)
        WIDE_SCALE(l, 0)
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < FB - 1; ++t) WIDE_READ_B(t, 0, 0, t)
#pragma unroll
    for (int l = 0; l < 3; ++l) WIDE_LUT(l, 0, 1)

    int s = s0;
    for (; s + 1 < s1; s += 2) {
        WIDE_HALF(0, s, 0)
        WIDE_HALF(0, s, 1)
        WIDE_HALF(1, s + 1, 0)
        WIDE_HALF(1, s + 1, 1)
    }
    if (s < s1) {
        WIDE_HALF(0, s, 0)
        WIDE_HALF(0, s, 1)
    }
    // The requests beyond the last step have arrived: their LDS and registers are free.  Every set passes through this wait,
    // used or not: a register that the compiler takes for free while its load is on its way would be overwritten under whatever
    // it holds by then (the scales of a segment's last step came to lie on a token fragment).
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(wq[0][0]), "+v"(wq[0][1]), "+v"(wq[1][0]), "+v"(wq[1][1])::"memory");
    if (BLK) {
#pragma unroll
        for (int i = 0; i < 2; ++i) asm volatile("" : "+v"(sq[BLK ? i : 0][0]), "+v"(sq[BLK ? i : 0][1]), "+v"(sq[BLK ? i : 0][2]), "+v"(sq[BLK ? i : 0][3]));
    }
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // the last MFMAs have written their accumulators
    // (pinned once more: no copy of an accumulator moves up between the MFMAs, whose latency the compiler does not know)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int t = 0; t < NT; ++t) asm volatile("" : "+a"(acc[j][t]));
#undef WIDE_HALF
#undef WIDE_MFMA
#undef WIDE_SCALE
#undef WIDE_LUT
#undef WIDE_READ_B
#undef WIDE_ARRIVED
#undef WIDE_LOAD_X
#undef WIDE_LOAD_S
#undef WIDE_LOAD_W
#undef WIDE_SCALES
}

// Position in the k-steps of the shared tiles laid end to end: tile (counted from `whole`) and step.  A step of a large
// tile weighs kCostLarge, one of a small tile kCostSmall (half the MFMAs, the same decode).
constexpr int kCostLarge = 5, kCostSmall = 3;
struct WidePos {
    int tile, step;
};
__device__ __forceinline__ bool before(const WidePos &a, const WidePos &b) { return a.tile < b.tile || (a.tile == b.tile && a.step < b.step); }
__device__ __forceinline__ WidePos wide_share_begin(const WideArgs &a, int share)
{
    const unsigned large = (unsigned)(a.large - a.whole), span = (unsigned)a.steps_total;
    const unsigned w_large = large * span * kCostLarge;
    const unsigned total = w_large + (unsigned)a.small * span * kCostSmall;
    unsigned p = (unsigned)((unsigned long long)total * (unsigned)share / (unsigned)a.n_shares);
    if (p < w_large) {
        p /= kCostLarge;
        return WidePos{(int)(p / span), (int)(p % span)};
    }
    p = (p - w_large) / kCostSmall;
    return WidePos{(int)(large + p / span), (int)(p % span)};
}

template <bool KTAIL, bool BLK>
__global__ __launch_bounds__(kWideThreads, 1) void gemm_wide_kernel(const WideArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char *lut = smem;  // byte-pair table at LDS address 0
    unsigned char *xs = smem + kLutBytes;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i16 = lane & 15, g = lane >> 4;

    // decode table (as in the streaming kernels)
    {
        const int code_bits = (int)(uint32_t)__builtin_bit_cast(uint16_t, (f16)a.code[lane & 15]);
#pragma unroll 4
        for (int p = tid; p < kLutBytes / 16; p += kWideThreads) {
            const int e = p >> 4;
            const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute((e >> 4) << 2, code_bits);
            const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute((e & 15) << 2, code_bits);
            const uint32_t v = hi | (lo << 16);
            reinterpret_cast<u32x4 *>(lut)[p] = u32x4{v, v, v, v};
        }
    }

    // Workgroups are dealt to the 8 XCDs in turn (workgroup L sits on XCD L % 8): an XCD takes consecutive tiles - the
    // token tiles of a few row tiles, which share the weights through its L2 - or consecutive shares.
    const int grid = (int)gridDim.x, xcd = (int)blockIdx.x & 7;
    const int place = xcd * (grid >> 3) + min(xcd, grid & 7) + ((int)blockIdx.x >> 3);

    int tile = place, s0 = 0, s1 = a.steps_total;  // the segment at hand
    WidePos at{0, 0}, end{0, 0};
    bool shared = a.whole <= place;
    if (a.n_shares) end = wide_share_begin(a, place + 1);
    if (shared) {
        if (!a.n_shares) return;
        at = wide_share_begin(a, place);
    }
    const WidePos begin = a.n_shares ? wide_share_begin(a, place) : at;
    for (;;) {
        if (shared) {
            if (!before(at, end)) return;
            tile = a.whole + at.tile;
            s0 = at.step;
            s1 = end.tile == at.tile ? end.step : a.steps_total;
        }
        // the tile's group, rows and tokens
        int group = 0, row_tile, tok_tile, index = tile;
        if (tile < a.large) {
            for (;; ++group) {
                const int per_row = (a.tok_count[group] + 127) >> 8, here = per_row * a.row_tiles;
                if (index < here) {
                    row_tile = index / per_row, tok_tile = index % per_row;
                    break;
                }
                index -= here;
            }
        } else {
            index -= a.large;
            for (;; ++group) {
                const int n = a.tok_count[group];
                const int here = (n & 255) >= 1 && (n & 255) <= 128 ? a.row_tiles : 0;
                if (index < here) {
                    row_tile = index, tok_tile = n >> 8;
                    break;
                }
                index -= here;
            }
        }
        const int tok0 = a.tok_begin[group] + tok_tile * kWideTokens, id = a.id[group];
        WideTile w;
        w.q = a.q + (size_t)id * (size_t)(a.m >> 3) * (size_t)(a.k >> 3) * 32;
        w.x = reinterpret_cast<const unsigned char *>(a.x) + (size_t)tok0 * (size_t)a.k * 2;
        w.absmax = a.absmax + (size_t)id * (size_t)a.m * (size_t)(BLK ? a.k >> (6 + a.blk_shift) : 1);
        w.m = a.m, w.k = a.k, w.row_base = row_tile * kWideRows;
        w.tokens = min(a.tok_count[group] - tok_tile * kWideTokens, kWideTokens);
        w.steps_total = a.steps_total, w.blk_shift = a.blk_shift;
        const bool large = w.tokens > 128;

        // accumulators: [j][t] element v of lane (i16, g) is weight row 16 g + 4 v + j of the wave's 64, token 16 t + i16
        f32x4 acc[4][16];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < 16; ++t) acc[j][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (large) wide_steps<16, KTAIL, BLK>(acc, w, xs, s0, s1);
        else wide_steps<8, KTAIL, BLK>(acc, w, xs, s0, s1);

        // ---- sums to outputs ----------------------------------------------------------------------------------
        // Straight-line code for 64 accumulators and every way a tile can end is 60 KB that each workgroup fetches once,
        // at 30 us a pass.  So the accumulators of four token tiles at a time go through LDS, where a loop can index
        // them (each lane reads back what it wrote), and one rolled piece of code does the rest.
        f16 *outp = reinterpret_cast<f16 *>(a.out);
        const f16 *resp = reinterpret_cast<const f16 *>(a.residual);
        const int row = w.row_base + wave * 64 + 16 * g;
        const uint32_t lane_off = (uint32_t)(wave * 64 * 64 + lane) * 16u;  // of the partial sums: [wave][t][j][lane] of 16 bytes
        int c_lo = 0, c_hi = -1;  // contributors whose partial sums are read
        bool own = true, store = true;
        int my_slot = 0, lo = place, lo_slot = 0;
        // (cache policy 16: sc1, past the XCD's L2 - writer and reader may sit on different XCDs)
        auto slot = [&](int share) {
            const int which = share == place ? my_slot : share == lo ? lo_slot : 0;
            return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<unsigned char *>(a.ws) + (size_t)(a.slots * share + which) * kWideSlot, 0,
                                                     (int)kWideSlot, 0x00020000);
        };
        __syncthreads();  // every wave is done with the stages
        if (s0 != 0 || s1 != a.steps_total) {
            // A shared tile: its contributors are shares lo .. hi in k order, each with a slot for its partial sums (the
            // second of a share's two where the share began in an earlier tile).  The last to arrive adds all of them
            // from memory in that order, so the sums do not depend on who that is.  With two contributors, the usual
            // number, it adds the other's to its own registers (the same sum), and one that finds the other arrived
            // does not write its own at all.
            const WidePos first{at.tile, 0}, past{at.tile + 1, 0};
            int hi = place;
            while (before(first, wide_share_begin(a, lo))) --lo;
            while (before(wide_share_begin(a, hi + 1), past)) ++hi;
            lo_slot = before(wide_share_begin(a, lo), first) ? 1 : 0;
            my_slot = before(begin, first) ? 1 : 0;
            const unsigned others = (unsigned)(hi - lo);
            unsigned *counter = a.counters + at.tile;
            volatile unsigned *ticket = reinterpret_cast<volatile unsigned *>(xs);
            if (tid == 0) *ticket = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            store = others == 1 && *ticket == 1;
            if (!store) {
                const auto mine = slot(place);
#pragma unroll
                for (int t = 0; t < 16; ++t)
                    if (t < 8 || large) {
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[j][t]), mine, (int)lane_off, (4 * t + j) * 1024, 16);
                    }
                __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the partial sums have left this CU
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
                __syncthreads();
                if (tid == 0) *ticket = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __syncthreads();
                store = *ticket == others;
            }
            if (store && tid == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            own = others == 1;
            c_lo = lo, c_hi = hi;
            if (own) c_lo = c_hi = lo == place ? hi : lo;
            __syncthreads();  // the ticket has been read: its LDS is free
        }
        if (store) {
            f32x4 *const mine = reinterpret_cast<f32x4 *>(xs) + wave * (16 * 64) + lane;  // [t][j][lane]
#pragma unroll 1
            for (int tb = 0; tb < (large ? 16 : 8); tb += 4) {
                f32x4 sum[4][4];
                if (own) {
#pragma unroll
                    for (int b = 0; b < 16; b += 4)
                        if (tb == b) {
#pragma unroll
                            for (int t = 0; t < 4; ++t)
#pragma unroll
                                for (int j = 0; j < 4; ++j) mine[(4 * t + j) * 64] = acc[j][b + t];
                        }
                }
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int j = 0; j < 4; ++j) sum[t][j] = own ? mine[(4 * t + j) * 64] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
                for (int c = c_lo; c <= c_hi; ++c) {
                    // (all loads issued before the first is awaited: the pass is a chain of memory round trips)
                    const auto src = slot(c);
                    f32x4 v[4][4];
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            v[t][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(src, (int)lane_off, (4 * (tb + t) + j) * 1024, 16));
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int j = 0; j < 4; ++j) sum[t][j] += v[t][j];
                }
                // a lane's sixteen rows of a token are consecutive: two 16-byte stores
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int tl = 16 * (tb + t) + i16;
                    const size_t tok = (size_t)(tok0 + tl);
                    if (tl < w.tokens && row + 8 <= a.m)
                        store_features8(outp, resp, a.epilogue, tok, a.m, row, f32x4{sum[t][0][0], sum[t][1][0], sum[t][2][0], sum[t][3][0]},
                                        f32x4{sum[t][0][1], sum[t][1][1], sum[t][2][1], sum[t][3][1]});
                    if (tl < w.tokens && row + 16 <= a.m)
                        store_features8(outp, resp, a.epilogue, tok, a.m, row + 8, f32x4{sum[t][0][2], sum[t][1][2], sum[t][2][2], sum[t][3][2]},
                                        f32x4{sum[t][0][3], sum[t][1][3], sum[t][2][3], sum[t][3][3]});
                }
            }
        }
        if (shared) {
            at = WidePos{at.tile + 1, 0};
        } else {
            tile += grid;
            if (tile >= a.whole) {
                if (!a.n_shares) return;
                shared = true;
                at = begin;
            }
        }
    }
}

size_t wide_lds_bytes() { return (size_t)kLutBytes + 3 * (size_t)kWideStage; }

void count_wide_tiles(const WideArgs &a, long long *large, long long *small)
{
    const long long row_tiles = ceil_div_i(a.m, kWideRows);
    *large = *small = 0;
    for (int e = 0; e < a.n_groups; ++e) {
        const int n = a.tok_count[e];
        *large += ((n + 127) >> 8) * row_tiles;
        *small += (n & 255) >= 1 && (n & 255) <= 128 ? row_tiles : 0;
    }
}

bool plan_gemm_wide(int split, int cus, WidePlan *plan)
{
    WideArgs &a = plan->args;
    a.steps_total = ceil_div_i(a.k, 64);
    a.row_tiles = ceil_div_i(a.m, kWideRows);
    a.n_shares = 0;
    long long large, small;
    count_wide_tiles(a, &large, &small);
    const long long tiles = large + small, weight = (large * kCostLarge + small * kCostSmall) * a.steps_total;
    if (tiles < 1 || tiles > 0x7fffffff || weight > 0x7fffffff) return false;
    a.large = (int)large, a.small = (int)small;
    a.whole = (int)tiles;
    if (split > 1) {
        a.whole = 0;
        a.n_shares = (int)(tiles * split);
    } else if (split == 0) {
        // as many rounds of whole large tiles as leave between a quarter and one and a quarter of a tile's work per
        // compute unit; that is shared
        const double per_cu = (double)weight / ((double)kCostLarge * a.steps_total * cus);
        long long rounds = (long long)(per_cu - 0.25);
        if (rounds > large / cus) rounds = large / cus;
        a.whole = (int)(rounds * cus);
        a.n_shares = tiles > a.whole ? cus : 0;
        // (at most eight shares to a tile, of at least eight steps)
        const long long rest = weight - (long long)a.whole * kCostLarge * a.steps_total;
        if (!rounds && a.n_shares > 8 * tiles) a.n_shares = (int)(8 * tiles);
        if (!rounds && a.n_shares > rest / (8 * kCostLarge)) a.n_shares = (int)(rest / (8 * kCostLarge)) + 1;
    }
    // (a share is at least a step of a large tile, so that every share between a tile's first and last has a part of it)
    if (a.n_shares > weight / kCostLarge) a.n_shares = (int)(weight / kCostLarge) > 0 ? (int)(weight / kCostLarge) : 1;
    plan->grid = (unsigned)(a.n_shares ? a.n_shares : tiles);
    const long long divided = tiles - a.whole;
    const bool alike = a.whole == a.large || !a.small;  // the divided tiles are of one kind: shares are equal parts of them
    a.slots = !a.n_shares || (alike && divided % a.n_shares == 0) ? 0 : alike && a.n_shares % divided == 0 ? 1 : 2;
    plan->ws_bytes = (size_t)a.n_shares * a.slots * kWideSlot;
    plan->n_counters = a.slots ? (size_t)divided : 0;
    return true;
}

hipError_t launch_gemm_wide(const WidePlan &plan, bool scale_blocks, hipStream_t stream)
{
    static OptInFlag done[16][3];
    const bool ktail = plan.args.k % 64 != 0;
    if (scale_blocks && ktail) return hipErrorInvalidConfiguration;
    const auto fn = scale_blocks ? gemm_wide_kernel<false, true> : ktail ? gemm_wide_kernel<true, false> : gemm_wide_kernel<false, false>;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 16) return hipErrorInvalidDevice;
    if ((e = ensure_lds_opt_in(done[dev][scale_blocks ? 2 : ktail], reinterpret_cast<const void *>(fn))) != hipSuccess) return e;
    hipLaunchKernelGGL(fn, dim3(plan.grid), dim3(kWideThreads), wide_lds_bytes(), stream, plan.args);
    return hipGetLastError();
}

}  // namespace tuna
