// What the kernels with 256-row many-token tiles share (gemm_wide.hip, gemm_wide_whole.hip): a tile's k-steps, and its outputs.  256
// weight rows x 16 NT tokens (NT 8 .. 16) per workgroup, one wave per SIMD (4 waves of 512 registers), every wave decoding the
// weights it multiplies straight into the MFMA's registers.
//
//   * A wave owns 64 rows x all tokens of the tile: 4 x NT tiles of v_mfma_f32_16x16x32_f16, whose up to 256 accumulator
//     registers sit in the AGPR half of the register file.  A 16-byte load of the packed layout is four rows x 8 k of a
//     lane, one dword of it - eight byte pairs through the decode table, scaled - IS a lane's weight operand of one
//     MFMA: no weight tile in LDS, and every weight is decoded once per token tile.
//   * Only the activations go through LDS, in a ring of three k-steps of [token][64 k] (128-byte rows, 16-byte slots
//     XOR-swizzled with token & 7: no bank conflicts), 32 KB each beside the decode table's 64 KB.  They are loaded into LDS
//     directly (lds_dma.hpp): through registers they took the path that LDS reads return their data over.
//   * The work of a k-step is spread evenly between its 8 NT MFMAs: per token tile (4 MFMAs) one fragment read, one or two table
//     reads, addresses and scalings; the loads behind the step's one barrier.
//
// What bounds it: the power limit.  With all compute units at work a step of 256 tokens takes 1.4 us, with half of them 1.08 (0.85 at 2.4 GHz
// would be the matrix pipes alone, which are busy for 75 per cent of the cycles over 128 steps, 68 over 64, 52 with tiles of 128 tokens), and
// what is left out of it saves what it draws: table reads 10 per cent, the way of the activations into LDS 9, their fragments 5.  torch's fp16
// product, which decodes nothing, takes as long on the same card (8192 x 8192 at 2048 tokens 182 us, here 190; at 2000 tokens 28672 x 4096 347
// and 350, 4096 x 14336 190 and 185, 6144 x 4096 82 and 81, 4096 x 4096 60 and 62).  So what pays is no work for
// tokens that are not there: NT for every number of token tiles (of 8 and 16 only, 4096 x 14336 at 777 tokens with blocks of 128 took
// 119 us in the smaller tiles that were picked then and takes 93; 4096 x 4096 at 2000 tokens 74 -> 62, 6144 x 4096 88 -> 81.5).  A step decodes as
// much whatever NT is: 0.36 us of it, beside 0.04 to 0.065 per token tile.  Around the loop (stamps at 4096 x 4096 x 4096): 3.2 us to the
// first step (4.9 with the table made before the first loads) and 3.1 for the outputs (6.9 as 16-byte pieces of 64 rows, a lane its own).
//
// KTAIL: k is any multiple of 8 - the slots of the last k-step beyond k load the last slot inside k (no access leaves a row), and their
// activations are zeros.  BLK: one scale per block of a row.  Decode and rounding are those of the other kernels (bit-identical to
// kernel.cu:2178-2192); an unshared tile's sums are the same products in the same order as the 16 x 16 x 32 variants of gemm_tiled.hip.
#pragma once
#include "lds_dma.hpp"
#include "row_pieces.hpp"

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

// (first: the workgroup's first segment, which makes the decode table; smem: it, and the three stages behind it)
template <int NT, bool KTAIL, bool BLK>
__device__ __forceinline__ void wide_steps(f32x4 (&acc)[4][(NT + 3) / 4 * 4], const WideTile &w, unsigned char *smem, const float *code, bool first, int s0, int s1, int tid)
{
    unsigned char *const xs = smem + kLutBytes;
    constexpr int XP = (NT + 1) / 2;  // 16-byte pieces of a step's activations a thread stages (32 tokens each)
    // token fragments on their way: a ring that the 4 NT of two steps make whole turns of
    constexpr int FB = NT % 2 == 0 ? 8 : NT == 15 ? 10 : NT;
    constexpr int T_NEXT = (14 * NT + 15) / 16 - 1;  // the token tile from which on the table reads of a half are the one after next's
    static_assert(4 * NT % FB == 0 && NT >= FB && NT <= 16, "token tiles");
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

    // scales of rows 4 i16 + j: one per row, or (BLK) one per block of 64 << blk_shift weights (a step lies inside one block).  Those
    // come two blocks at a time, for the steps s and s + 1 of an iteration: lane (i16, g) loads row 4 i16 + g's, rounds them, and the
    // lanes of a column exchange theirs.  (Four loads a step, of each lane's own rows: four times as many lines.  A step took 0.23 us
    // longer than with one scale per row, now 0.10: 8.5 per cent of 1245 random launches.)
    const int nblk = BLK ? w.k >> (6 + w.blk_shift) : 1;
    const float *s_base = w.absmax + (size_t)w.row_base * (size_t)nblk;
    const u32x4 s_rsrc = buffer_at(s_base, (size_t)(w.m - w.row_base) * (size_t)nblk * 4);
    uint32_t s_off[BLK ? 1 : 4];
#pragma unroll
    for (int j = 0; j < (BLK ? 1 : 4); ++j) s_off[j] = (uint32_t)(min(row_w + 4 * i16 + (BLK ? g : j), w.m - 1) - w.row_base) * (uint32_t)nblk * 4u;
    uint32_t sq[4];
    u32x2 sb;      // (BLK: blocks b and b + 1, b of step s and at most the last but one)
    f16x2 sc[4];   // (BLK: of the steps s and s + 1, else twice the same)
#define WIDE_BLOCK(s) min((s) >> w.blk_shift, nblk - 1)
#define WIDE_LOAD_S(s) load_async(sb, s_rsrc, s_off[0] + (uint32_t)min(WIDE_BLOCK(s), nblk - 2) * 4u, 0u);
#define WIDE_SCALES(s)                                                                                        \
    if (BLK) {                                                                                                \
        asm volatile("" : "+v"(sb));                                                                          \
        const int b_ = WIDE_BLOCK(s), c_ = WIDE_BLOCK((s) + 1), first_ = min(b_, nblk - 2);                   \
        const f16x2 p_ = {(f16)__builtin_bit_cast(float, b_ > first_ ? sb[1] : sb[0]),                        \
                          (f16)__builtin_bit_cast(float, c_ > first_ ? sb[1] : sb[0])};                       \
        const uint32_t v_ = __builtin_bit_cast(uint32_t, p_);                                                 \
        const auto h_ = __builtin_amdgcn_permlane32_swap(v_, v_, false, false);                               \
        const auto l0_ = __builtin_amdgcn_permlane16_swap(h_[0], h_[0], false, false);                        \
        const auto l1_ = __builtin_amdgcn_permlane16_swap(h_[1], h_[1], false, false);                        \
        sc[0] = __builtin_bit_cast(f16x2, (uint32_t)l0_[0]), sc[1] = __builtin_bit_cast(f16x2, (uint32_t)l0_[1]);                 \
        sc[2] = __builtin_bit_cast(f16x2, (uint32_t)l1_[0]), sc[3] = __builtin_bit_cast(f16x2, (uint32_t)l1_[1]);                 \
    } else {                                                                                                  \
        _Pragma("unroll") for (int j = 0; j < 4; ++j)                                                         \
        {                                                                                                     \
            const f16 h_ = (f16)__builtin_bit_cast(float, sq[j]);                                             \
            sc[j] = f16x2{h_, h_};                                                                            \
        }                                                                                                     \
    }

    u32x4 wq[2][2];   // [set][half]: packed weights of two k-steps
    const int s_last = w.steps_total - 1;
    // Requests, in an order that the waits count on: for a step the weights (WL operations), then the activations (XP), then the next
    // step's weights ...; with scale blocks, ahead of the activations of every other step (it 1), the scales of the next two.
    constexpr int WL = 2, SL = BLK ? 1 : 0;
#define WIDE_LOAD_W(set, s)                                                                                   \
    {                                                                                                         \
        const int s_ = min((s), s_last);                                                                      \
        const bool t_ = KTAIL && s_ == s_last;                                                                \
        load_async(wq[set][0], q_rsrc, t_ ? a_off - a_back0 : a_off, (uint32_t)wide_weight_uniform(s_, 0, t_, slot_last)); \
        load_async(wq[set][1], q_rsrc, t_ ? a_off - a_back1 : a_off, (uint32_t)wide_weight_uniform(s_, 1, t_, slot_last)); \
    }
#define WIDE_LOAD_X(i, off, s)                                                                                \
    {                                                                                                         \
        const int s_ = min((s), s_last);                                                                      \
        load_to_lds(x_rsrc, KTAIL && s_ == s_last ? x_off[i] | x_beyond : x_off[i], (uint32_t)s_ * 128u, xs_lds + (off) + (i) * 4096u); \
    }
    // A step's weights have arrived: at most N operations behind them are pending.
#define WIDE_ARRIVED(set, N)                                                                                  \
    asm volatile("s_waitcnt vmcnt(%2)" : "+v"(wq[set][0]), "+v"(wq[set][1]) : "n"(N));

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
#define WIDE_SCALE(l, ab, it)                                                                                 \
    {                                                                                                         \
        const f16x2 s_ = sc[(l) >> 2], h_ = __builtin_bit_cast(f16x2, lt[(l) & 3]) * f16x2{s_[BLK ? (it) : 0], s_[BLK ? (it) : 0]}; \
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
            const int base_ = (h) * NT + t, ring_ = (it) * 2 * NT + base_; /* of the step, of the two steps */  \
            WIDE_MFMA(h, 0, t, ring_ % FB)                                                                    \
            if ((h) == 0 && t == T_NEXT) { WIDE_ARRIVED((it) ^ 1, XP + ((it) == 0 ? SL : 0)) } /* the table reads reach the next step */ \
            if ((h) == 1 && t == NT - FB + 1) {                                                               \
                wait_loads<WL + ((it) == 1 ? SL : 0)>(); /* this wave's pieces of the next step are in LDS */                        \
                __builtin_amdgcn_s_barrier();                                                                 \
                asm volatile("" ::: "memory");                                                                \
            }                                                                                                 \
            {                                                                                                 \
                const int nt_ = base_ + FB - 1;                                                               \
                WIDE_READ_B((ring_ + FB - 1) % FB, (nt_ / NT) & 1, nt_ >= 2 * NT ? nxt : cur, nt_ % NT)       \
            }                                                                                                 \
            __builtin_amdgcn_sched_barrier(0);                                                                \
            WIDE_MFMA(h, 1, t, ring_ % FB)                                                                    \
            if (BLK && (it) == 1 && (h) == 1 && t == 0) {                                                     \
                WIDE_SCALES((step) + 1) /* (they came ahead of the weights of the step at hand) */             \
                WIDE_LOAD_S((step) + 3)                                                                       \
            }                                                                                                 \
            _Pragma("unroll") for (int l = 16 * t / NT; l < 16 * (t + 1) / NT; ++l) {                         \
                WIDE_SCALE(l, dh_, dset_)                                                                     \
                if (l + 3 < 16) WIDE_LUT(l + 3, dset_, dh_)                                                   \
                else WIDE_LUT(l + 3 - 16, (it) ^ 1, h)                                                        \
            }                                                                                                 \
            __builtin_amdgcn_sched_barrier(0);                                                                \
            WIDE_MFMA(h, 2, t, ring_ % FB)                                                                    \
            if ((h) == 1 && t > NT - FB + 1 && (t - (NT - FB + 2)) * 2 < XP) {                                \
                WIDE_LOAD_X((t - (NT - FB + 2)) * 2, (uint32_t)nx2, (step) + 2)                               \
                if ((t - (NT - FB + 2)) * 2 + 1 < XP)                                                         \
                    WIDE_LOAD_X((t - (NT - FB + 2)) * 2 + 1, (uint32_t)nx2, (step) + 2)                       \
            }                                                                                                 \
            __builtin_amdgcn_sched_barrier(0);                                                                \
            WIDE_MFMA(h, 3, t, ring_ % FB)                                                                    \
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
    // Everything that two steps need is requested before the decode table is made: its codes in front.
    uint32_t code_bits;
    load_async(code_bits, buffer_at(code, 64), (uint32_t)i16 * 4u, 0u);
    if (BLK) {
        WIDE_LOAD_S(s0)
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) load_async(sq[j], s_rsrc, s_off[j], 0u);
    }
    WIDE_LOAD_W(0, s0)
    if (!first) {  // the previous segment's work area has been read (its outputs may still be on their way)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
    }
#pragma unroll
    for (int i = 0; i < XP; ++i) WIDE_LOAD_X(i, 0u, s0)
    WIDE_LOAD_W(1, s0 + 1)
#pragma unroll
    for (int i = 0; i < XP; ++i) WIDE_LOAD_X(i, (uint32_t)kWideStage, s0 + 1)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int t = 0; t < (NT + 3) / 4 * 4; ++t) {
            acc[j][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            asm volatile("" : "+a"(acc[j][t]));
        }
    asm volatile("s_waitcnt vmcnt(%1)" : "+v"(code_bits) : "n"(2 * XP + 2 * WL + (BLK ? 1 : 4)));
    if (first) build_pair_table<kWideThreads>(smem, tid, __builtin_bit_cast(float, code_bits));
    WIDE_ARRIVED(0, XP + WL)
    if (!BLK) asm volatile("" : "+v"(sq[0]), "+v"(sq[1]), "+v"(sq[2]), "+v"(sq[3]));
    WIDE_SCALES(s0)
    if (BLK) WIDE_LOAD_S(s0 + 2)
    __syncthreads();  // the table, and the activations of the first step
#pragma unroll
    for (int l = 0; l < 16; ++l) {
        WIDE_LUT(l, 0, 0)
        WIDE_SCALE(l, 0, 0)
    }
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
    if (BLK) asm volatile("" : "+v"(sb));
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
#undef WIDE_BLOCK
}

// Outputs of four token tiles of a wave.  A lane's sums of a token tile are four pieces [v] of four consecutive rows: 16 g + 4 v ..
// + 3 of the wave's 64, of token 16 t + i16.  They go through the wave's 16 KB of LDS - [token of 64][16 pieces, XOR-swizzled with the
// token], no bank conflicts either way - and come back as rows of outputs: eight lanes hold 64 consecutive rows of a token.  (Each lane
// storing its own, 64 pieces of 16 bytes an instruction, a tile of 256 tokens took 6.9 us to end; now 5.2, 3.1 through fp16 pieces.)
__device__ __forceinline__ f32x4 *wide_piece(unsigned char *mine, int lane, int t, int v)
{
    const int i16 = lane & 15, g = lane >> 4;
    return reinterpret_cast<f32x4 *>(mine + (16 * t + i16) * 256 + (((4 * g + v) ^ i16) << 4));
}
struct WideOut {
    f16 *out;             // of the lane's first token and rows
    const f16 *residual;
    int epilogue, ld;     // ld: outputs of a token
    int tokens;           // of the tile from the lane's first one on; 0 where the lane's rows are beyond the matrix
};
// (tok: the tile's first token; row: the wave's first row)
__device__ __forceinline__ WideOut wide_out(int lane, void *out, const void *residual, int epilogue, int m, int tok, int tokens, int row)
{
    const int r = row + 8 * (lane & 7), tk = lane >> 3, ld = epilogue == TUNA_EPILOGUE_SILU_MUL ? m >> 1 : m;
    WideOut o;
    o.out = reinterpret_cast<f16 *>(out) + (size_t)(tok + tk) * (size_t)ld + (epilogue == TUNA_EPILOGUE_SILU_MUL ? r >> 1 : r);
    o.residual = reinterpret_cast<const f16 *>(residual) + (size_t)(tok + tk) * (size_t)ld + r;
    o.epilogue = epilogue, o.ld = ld;
    o.tokens = r + 8 <= m ? tokens - tk : 0;
    return o;
}
__device__ __forceinline__ void wide_store(WideOut &w, const unsigned char *mine, int lane)
{
    const int r8 = lane & 7, tk = lane >> 3;
    const size_t step = (size_t)8 * (size_t)w.ld;
    f32x4 o[8][2];  // tokens tk + 8 h, eight rows
#pragma unroll
    for (int h = 0; h < 8; ++h)
#pragma unroll
        for (int e = 0; e < 2; ++e)
            o[h][e] = *reinterpret_cast<const f32x4 *>(mine + (8 * h + tk) * 256 + (((2 * r8 + e) ^ (8 * (h & 1) + tk)) << 4));
    if (w.epilogue == TUNA_EPILOGUE_SILU_MUL) {
#pragma unroll
        for (int h = 0; h < 8; ++h) {
            f16x4 y;
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = (f16)silu_mul(o[h][i >> 1][2 * (i & 1)], o[h][i >> 1][2 * (i & 1) + 1]);
            if (8 * h < w.tokens) *reinterpret_cast<f16x4 *>(w.out + h * step) = y;
        }
    } else {
        if (w.epilogue == TUNA_EPILOGUE_RESIDUAL) {  // (the residual is aligned to 8 bytes only)
            f16x4 r[8][2];
#pragma unroll
            for (int h = 0; h < 8; ++h)
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    r[h][e] = 8 * h < w.tokens ? *reinterpret_cast<const f16x4 *>(w.residual + h * step + 4 * e) : f16x4{0, 0, 0, 0};
#pragma unroll
            for (int h = 0; h < 8; ++h)
#pragma unroll
                for (int i = 0; i < 8; ++i) o[h][i >> 2][i & 3] += (float)r[h][i >> 2][i & 3];
        }
#pragma unroll
        for (int h = 0; h < 8; ++h) {
            f16x8 y;
#pragma unroll
            for (int i = 0; i < 8; ++i) y[i] = (f16)o[h][i >> 2][i & 3];
            if (8 * h < w.tokens) *reinterpret_cast<f16x8 *>(w.out + h * step) = y;
        }
    }
    w.out += 8 * step, w.residual += 8 * step, w.tokens -= 64;
}

}  // namespace tuna
