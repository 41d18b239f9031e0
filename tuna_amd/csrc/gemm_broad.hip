// Fused FP16 x 4-bit-codebook GEMM from 49 tokens on, where an MFMA tile of 16 tokens no longer waits for its weights but a
// token tile of 128 or 256 leaves compute units idle or takes k in many parts: a workgroup is 32 RT rows (RT 2 .. 8) x 64, 80 or
// 96 tokens in one of `split` parts of k.
//
// Eight waves, two along the rows and four along k: the waves of a row group divide a unit of four k-steps, so a weight is
// decoded once per token tile, straight into the MFMA's operand, and the waves of a k group share its activations.  These
// come into LDS directly (lds_dma.hpp), a unit ahead in the other of two buffers, and the loop has one barrier per unit, at its
// middle: every wave has read this unit's activations there and has its pieces of the next one's.  Weights are on their way two
// units ahead in registers, table reads two turns (a turn: a row tile's products of 32 k).  The k groups' sums meet in LDS in
// their order, over the table, and parts of k in the workspace, added by the last to arrive in k order.  Units are walked from a
// hash of the tile on, as in gemm_tall.hip.
//
// What bounds it: no single unit.  A unit takes 0.13 us per row tile of a wave (two turns: table reads, scaling; the matrix
// instructions hide under them) and 0.09 .. 0.14 per token tile (its way into LDS and out of it, twice).  Of 31 us for 28672 x
// 4096 at 80 tokens, 24 are left without the loads, 27 with either kind.  No gain, and not kept: table reads three and four turns
// ahead, the matrix instructions dealt out between the decode of byte pairs, the barrier two turns before a unit's end.
//
// Against the launches that were chosen before, in us on one card: 28672 x 4096 at 80 tokens 44 -> 29, at 128 43 -> 37; 8192 x 8192
// at 96 29 -> 24, at 160 47 -> 30, at 256 52 -> 43; 4096 x 14336 at 192 45 -> 32; 5120 x 13824 at 160 45 -> 34; 11008 x 2048 at 192
// 27 -> 17; 57344 x 8192 at 64 88 -> 73.  Groups: one launch over all row tiles and token tiles of all groups, eight experts of
// 14336 x 4096 on 512 tokens 147 -> 98.  Scales in blocks of 128: 4096 x 14336 at 777 tokens 126 -> 115, 5120 x 5120 at 594
// 55 -> 42.  The floor of the first, its weights at the rate of a large copy: 12.
#include "lds_dma.hpp"
#include "row_pieces.hpp"
#include <type_traits>

namespace tuna {

namespace {
constexpr int kRowGroups = 2, kStepGroups = 4;  // the waves: two along the rows, four along k
constexpr int kWaves = kRowGroups * kStepGroups, kThreads = 64 * kWaves;

constexpr size_t x_bytes(int nt) { return (size_t)2 * kStepGroups * nt * 2048; }  // two units' activations
// In the end, over the table and the activations: the waves' sums, as many token tiles at a time as fit, then the outputs.
constexpr int red_tiles(int rt, int nt)
{
    const int fit = (kLdsLimit - 16) / (kWaves * rt * 1024);
    return fit < nt ? fit : nt;
}
constexpr size_t end_bytes(int rt, int nt)
{
    const size_t red = (size_t)kWaves * rt * red_tiles(rt, nt) * 1024, out = (size_t)16 * nt * (kRowGroups * 16 * rt + 4) * 4;
    return red > out ? red : out;
}
// Scales in blocks of 64 << blk_shift weights lie behind the activations, two bytes each and a lane's of a block together: [block][row
// group][16 lanes][scale_dwords].  Where they fit all those of a tile's part of k (SCALES_PART), else a unit's, four, two or one
// a row, in the other of two slots (SCALES_UNIT: 0.2 us more a unit).
enum { SCALES_ROW, SCALES_PART, SCALES_UNIT };
constexpr int scale_dwords(int rt) { return rt <= 2 ? 1 : rt <= 4 ? 2 : 4; }
constexpr int scale_block(int rt) { return kRowGroups * 64 * scale_dwords(rt); }
constexpr size_t loop_bytes(int rt, int nt, int blocks) { return kLutBytes + x_bytes(nt) + (size_t)blocks * scale_block(rt); }
constexpr size_t lds_bytes(int rt, int nt, int blocks)
{
    const size_t loop = loop_bytes(rt, nt, blocks), end = end_bytes(rt, nt) + 16;
    return loop > end ? loop : end;
}

// (GROUPS: BroadGroups, or nothing for one matrix)
template <int RT, int NT, int BLK, class GROUPS>
__global__ __launch_bounds__(kThreads, 2) void gemm_broad_kernel(const uint8_t *a_q, const void *a_x, const float *a_code, const float *a_absmax,
                                                                     int a_k, int a_n, int a_m, int a_part_steps, void *a_out, int a_epilogue,
                                                                     const void *a_residual, float *a_ws, unsigned *a_counters, int a_blk_shift, int a_ticket, const GROUPS groups)
{
    constexpr bool GRP = !std::is_empty<GROUPS>::value;
    using P = Pieces<RT>;
    constexpr int NS = 2;      // units whose weights are on their way
    constexpr int T = 2 * RT;  // turns of a step: a row tile of a half each
    constexpr int ROWS = kRowGroups * 16 * RT, STAGE = kStepGroups * NT * 2048;  // activations of a unit
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), rg = wave & (kRowGroups - 1), kg = wave / kRowGroups;
    const int i16 = lane & 15, g = lane >> 4;
    const uint32_t lane4 = (uint32_t)lane << 2;
    const int kb_total = a_k >> 3, steps_total = (a_k + 63) >> 6;

    unsigned char *const work = smem + kLutBytes;
    volatile unsigned *const ticket = reinterpret_cast<volatile unsigned *>(smem + a_ticket);
    const float code_lane = a_code[lane & 15];

    // weights, per lane and piece: rows LW i16 .. + LW - 1 of the piece's, block column g of a half
    uint32_t w_off[P::count];
#pragma unroll
    for (int p = 0; p < P::count; ++p) {
        const int row = 16 * (rg * RT + P::first(p)) + P::width(p) * i16;
        w_off[p] = ((uint32_t)(row >> 3) * (uint32_t)kb_total + (uint32_t)g) * 32u + (uint32_t)(row & 7) * 4u;
    }
    // the slots of the last step beyond k read the last slot inside it (and their activations are zeros)
    const int slot_last = (kb_total - 1) & 7, s_tail = (a_k & 63) ? steps_total - 1 : -1;
    const uint32_t back0 = (uint32_t)max(0, g - slot_last) * 32u, back1 = (uint32_t)max(0, 4 + g - slot_last) * 32u;
    // activations: piece i of a wave is tokens 8 (rg NT + i) .. + 7, lane l's sixteen bytes slot (l ^ l / 8) % 8 of token l / 8: a
    // piece lands in LDS in lane order, [token][8 slots], slot s of token t at s ^ (t % 8)
    const uint32_t x_lane = ((uint32_t)(rg * NT * 8 + (lane >> 3)) * (uint32_t)a_k + (uint32_t)((lane ^ (lane >> 3)) & 7) * 8u) * 2u;
    const int x_k_left = a_k - ((lane ^ (lane >> 3)) & 7) * 8;
    const uint32_t x_lds = (uint32_t)(kLutBytes + kg * (NT * 2048) + rg * (NT * 1024));
    const int swz = (g ^ (i16 & 7)) << 4;
    const unsigned char *const x_frag0 = smem + kLutBytes + kg * (NT * 2048) + i16 * 128 + swz, *const x_frag1 = x_frag0 - swz + (64 ^ swz);

    const int part = (int)blockIdx.y, split = (int)gridDim.y;
    int tile = (int)blockIdx.x, tok_base = (int)blockIdx.z * (16 * NT), tokens = min(16 * NT, a_n - tok_base), group = 0;
    if constexpr (GRP) {
        // the group whose items are the last to begin at or in front of this one; a row tile's token tiles are neighbours
        const bool begun = lane < groups.n && groups.item[lane] <= tile;
        const int at = __builtin_popcountll(__ballot(begun)) - 1, count = groups.tok_count[at], tok_tiles = (count + 16 * NT - 1) / (16 * NT);
        const int local = tile - groups.item[at];
        tile = local / tok_tiles;
        const int first = (local - tile * tok_tiles) * (16 * NT);
        tok_base = groups.tok_begin[at] + first;
        tokens = min(16 * NT, count - first);
        group = groups.id[at];
    }
    const int row_base = tile * ROWS;  // (of the group's rows)
    const size_t first_row = (size_t)group * (size_t)a_m + (size_t)row_base;
    const int s0 = part * a_part_steps, s1 = min(s0 + a_part_steps, steps_total);
    const size_t rows_left = (size_t)(a_m - row_base);
    const __amdgpu_buffer_rsrc_t q_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(a_q) + first_row * (size_t)(a_k >> 1), 0,
        (int)(uint32_t)min(rows_left * (size_t)(a_k >> 1), (size_t)0xffffffffu), 0x00020000);
    const u32x4 x_rsrc = buffer_at(reinterpret_cast<const f16 *>(a_x) + (size_t)tok_base * (size_t)a_k, (size_t)tokens * (size_t)a_k * 2);
    const int nblk = BLK ? a_k >> (6 + a_blk_shift) : 1;
    const __amdgpu_buffer_rsrc_t s_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a_absmax) + first_row * (size_t)nblk, 0, (int)(uint32_t)min(rows_left * (size_t)nblk * 4, (size_t)0xffffffffu), 0x00020000);

    f32x4 acc[RT][NT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    // units of four steps, one per k group; the part's, from one that depends on the tile on and around (workgroups that
    // walk k in step ask the same memory channels)
    const int units = (s1 - s0 + kStepGroups - 1) / kStepGroups;
    const int u_first = (int)(((((unsigned)blockIdx.x * 2654435761u) >> 16) * (unsigned)units) >> 16);
    int u_w = u_first, u_x = u_first;
    auto next = [&](int u) { return u + 1 < units ? u + 1 : 0; };

    uint32_t wq[NS][2][RT];
#define BROAD_LOAD_W(set, h)                                                                                   \
    {                                                                                                         \
        const int s_ = min(s0 + u_w * kStepGroups + kg, steps_total - 1);                                     \
        const uint32_t at_ = (uint32_t)s_ * 256u + (h) * 128u - (s_ == s_tail ? ((h) ? back1 : back0) : 0u);  \
        _Pragma("unroll") for (int p = 0; p < P::count; ++p)                                                  \
        {                                                                                                     \
            const int o_ = (int)(w_off[p] + at_), r_ = P::first(p);                                           \
            if (P::width(p) == 4) {                                                                           \
                const u32x4 v_ = __builtin_amdgcn_raw_buffer_load_b128(q_rsrc, o_, 0, 2);                     \
                _Pragma("unroll") for (int j = 0; j < 4; ++j) wq[set][h][r_ + j] = v_[j];                     \
            } else if (P::width(p) == 2) {                                                                    \
                const u32x2 v_ = __builtin_amdgcn_raw_buffer_load_b64(q_rsrc, o_, 0, 2);                      \
                _Pragma("unroll") for (int j = 0; j < 2; ++j) wq[set][h][r_ + j] = v_[j];                     \
            } else {                                                                                          \
                wq[set][h][r_] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(q_rsrc, o_, 0, 2);            \
            }                                                                                                 \
        }                                                                                                     \
        if (h) u_w = next(u_w);                                                                               \
    }
    // (steps beyond k, and in the last part those of a unit that the part doesn't have: out of range, zeros)
#define BROAD_LOAD_X(off)                                                                                     \
    {                                                                                                         \
        const int s_ = s0 + u_x * kStepGroups + kg;                                                           \
        const uint32_t l_ = s_ * 64 < x_k_left ? x_lane : 0x7fffffffu;                                        \
        _Pragma("unroll") for (int i = 0; i < NT; ++i)                                                        \
            load_to_lds(x_rsrc, l_ + (uint32_t)i * 16u * (uint32_t)a_k, (uint32_t)min(s_, steps_total - 1) * 128u, x_lds + (uint32_t)(off) + i * 1024u); \
        asm volatile("" ::: "memory");                                                                        \
        u_x = next(u_x);                                                                                      \
    }
    BROAD_LOAD_X(0)
    BROAD_LOAD_W(0, 0)
    float sc32[RT];
    if constexpr (!BLK) {
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int p = P::of(r);
            sc32[r] = __builtin_bit_cast(float, (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(
                                                    s_rsrc, (16 * (rg * RT + P::first(p)) + P::width(p) * i16 + r - P::first(p)) * 4, 0, 0));
        }
    }
    BROAD_LOAD_W(0, 1)
    f16x2 sc[BLK ? 2 : 1][(RT + 1) / 2];  // of the step at hand and of the next one
    f16x8 fa[2], fb[2][NT];
    uint32_t lt[2][4];  // table reads of a turn and of the next one
    // (turn tau of step u: row tile tau % RT of half tau / RT; u and tau may run over into the next step)
#define BROAD_LUT(u, tau)                                                                                      \
    {                                                                                                         \
        const int u_ = ((u) + (tau) / T) % NS, h_ = (tau) % T / RT, r_ = (tau) % RT, l_ = ((u) * T + (tau)) % 2; \
        _Pragma("unroll") for (int b = 0; b < 4; ++b) lt[l_][b] = *reinterpret_cast<const lds_u32 *>(         \
            (uintptr_t)__builtin_amdgcn_perm(wq[u_][h_][r_], lane4, 0x0c0c0400u + 0x100u * b));               \
        if (r_ == RT - 1) BROAD_LOAD_W(u_, h_) /* the half's registers are free */                             \
    }
#define BROAD_SCALE(u, tau)                                                                                    \
    {                                                                                                         \
        const int r_ = (tau) % RT, l_ = ((u) * T + (tau)) % 2, f_ = (tau) & 1; /* (as for BROAD_LUT) */       \
        _Pragma("unroll") for (int b = 0; b < 4; ++b)                                                         \
        {                                                                                                     \
            f16x2 v_;                                                                                         \
            if (r_ & 1) asm volatile("v_pk_mul_f16 %0, %1, %2 op_sel:[0,1] op_sel_hi:[1,1]" : "=v"(v_) : "v"(lt[l_][b]), "v"(sc[BLK ? ((u) + (tau) / T) % NS : 0][r_ / 2])); \
            else asm volatile("v_pk_mul_f16 %0, %1, %2 op_sel:[0,0] op_sel_hi:[1,0]" : "=v"(v_) : "v"(lt[l_][b]), "v"(sc[BLK ? ((u) + (tau) / T) % NS : 0][r_ / 2])); \
            fa[f_][2 * b] = v_[0];                                                                            \
            fa[f_][2 * b + 1] = v_[1];                                                                        \
        }                                                                                                     \
    }
#define BROAD_READ_B(h, off, t) fb[h][t] = *reinterpret_cast<const f16x8 *>(((h) ? x_frag1 : x_frag0) + (off) + (t) * 2048);
/* A turn: the products of its row tile, the scaling of the next one, the table reads of the one after it.  The unit's only
   barrier stands at its middle: every wave has read this unit's activations and has the next unit's of its own in
   LDS (all loads but the weights requested since are done), so the ones of the unit after that may be requested over this unit's,
   and the next unit's first half is read. */
#define BROAD_STEP(u)                                                                                         \
    _Pragma("unroll") for (int tau = 0; tau < T; ++tau)                                                       \
    {                                                                                                         \
        _Pragma("unroll") for (int t = 0; t < NT; ++t) acc[tau % RT][t] =                                     \
            __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[tau & 1], fb[tau / RT][t], acc[tau % RT][t], 0, 0, 0);  \
        BROAD_SCALE(u, tau + 1)                                                                               \
        _Pragma("unroll") for (int t = 0; t < NT; ++t) if (tau == t * (RT - 1) / NT) BROAD_READ_B(1, ((u) & 1) * STAGE, t) \
        if (BLK == SCALES_UNIT && tau == RT - 1) BROAD_STORE_SCALES(((u) + 1) & 1)                                           \
        if (tau == RT) {                                                                                      \
            __builtin_amdgcn_sched_barrier(0);                                                                \
            __builtin_amdgcn_s_waitcnt(0x0070 | (2 * P::count)); /* (for the compiler to know, and lgkmcnt(0)) */ \
            wait_loads<2 * P::count>();                                                                       \
            __builtin_amdgcn_s_barrier();                                                                     \
            asm volatile("" ::: "memory");                                                                    \
            BROAD_LOAD_X(((u) & 1) * STAGE)                                                                   \
            if (BLK) {                                                                                        \
                if (BLK == SCALES_UNIT) BROAD_LOAD_SCALES()                                                                           \
                BROAD_READ_SCALES(((u) + 1) & 1)                                                              \
            }                                                                                                 \
        }                                                                                                     \
        _Pragma("unroll") for (int t = 0; t < NT; ++t) if (tau == RT + t * (RT - 1) / NT) BROAD_READ_B(0, (((u) + 1) & 1) * STAGE, t) \
        BROAD_LUT(u, tau + 2)                                                                                 \
        __builtin_amdgcn_sched_barrier(0);                                                                    \
    }
    const int b0 = BLK == SCALES_PART ? s0 >> a_blk_shift : 0;
    // SCALES_UNIT: a row a lane, 64 rows a wave; requested behind the barrier for the unit after the next, stored in front of
    // the next one, read behind that.
    constexpr int SD = scale_dwords(RT);
    unsigned char *const scales = smem + kLutBytes + 2 * STAGE;
    const lds_u32 *const sc_lane = reinterpret_cast<const lds_u32 *>(
        (uintptr_t)(uint32_t)(kLutBytes + 2 * STAGE + (((BLK == SCALES_UNIT ? kg >> a_blk_shift : 0) * kRowGroups + rg) * 16 + i16) * (SD * 4)));
    const int sc_row = wave * 64 + lane;
    int sc_dst = 0, u_sc = u_first;
    if constexpr (BLK == SCALES_UNIT) {
        const int group_ = sc_row / (16 * RT), r16 = (sc_row >> 4) - group_ * RT;
        const int width = P::width_at(r16), first = P::first_at(r16);
        const int in = sc_row - 16 * (group_ * RT + first);
        sc_dst = (group_ * 16 + in / width) * (SD * 4) + (first + in % width) * 2;
    }
    u32x4 sv = {0u, 0u, 0u, 0u};
#define BROAD_LOAD_SCALES()                                                                                   \
    {                                                                                                         \
        if (wave * 64 < ROWS) {                                                                               \
            const int at_ = (sc_row * nblk + ((s0 + u_sc * kStepGroups) >> a_blk_shift)) * 4;                 \
            if (a_blk_shift == 0) {                                                                           \
                sv = __builtin_amdgcn_raw_buffer_load_b128(s_rsrc, at_, 0, 0);                                \
            } else if (a_blk_shift == 1) {                                                                    \
                const u32x2 v_ = __builtin_amdgcn_raw_buffer_load_b64(s_rsrc, at_, 0, 0);                     \
                sv[0] = v_[0], sv[1] = v_[1];                                                                 \
            } else {                                                                                          \
                sv[0] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(s_rsrc, at_, 0, 0);                    \
            }                                                                                                 \
        }                                                                                                     \
        u_sc = next(u_sc);                                                                                    \
    }
#define BROAD_STORE_SCALES(slot)                                                                              \
    if (wave * 64 < ROWS && sc_row < ROWS) {                                                                  \
        _Pragma("unroll") for (int e = 0; e < kStepGroups; ++e) {                                             \
            const uint32_t bits_ = sv[e]; /* (a copy: a bit cast of a vector's element would take the first) */ \
            if (e << a_blk_shift < kStepGroups)                                                               \
                *reinterpret_cast<f16 *>(scales + (slot) * (kStepGroups * scale_block(RT)) + e * (kRowGroups * 64 * SD) + sc_dst) = (f16)__builtin_bit_cast(float, bits_); \
        }                                                                                                     \
    }
#define BROAD_READ_SCALES(slot)                                                                               \
    {                                                                                                         \
        const lds_u32 *from_ = sc_lane + (slot) * (kStepGroups * scale_block(RT) / 4);                        \
        if (BLK == SCALES_PART) {                                                                             \
            from_ = sc_lane + ((min(s0 + u_sc * kStepGroups + kg, s1 - 1) >> a_blk_shift) - b0) * (scale_block(RT) / 4); \
            u_sc = next(u_sc);                                                                                \
        }                                                                                                     \
        _Pragma("unroll") for (int j = 0; j < (RT + 1) / 2; ++j) sc[BLK ? (slot) : 0][j] = __builtin_bit_cast(f16x2, from_[j]); \
    }
    if constexpr (BLK == SCALES_UNIT) {
        BROAD_LOAD_SCALES()
        BROAD_STORE_SCALES(0)
    }
    if constexpr (BLK == SCALES_PART) {
        // Four blocks of a row a lane, 64 rows a wave: the LDS banks of a store are those of 16 lanes and two or four pairs of
        // row tiles.  (The last four of a row where four from here on would go beyond it: what is in front of the part or
        // behind it isn't stored.)
        const int nb = ((s1 - 1) >> a_blk_shift) + 1 - b0, quads = (nb + 3) >> 2;
        constexpr int RG = (ROWS + 63) / 64, PIECES = 4;  // groups of 64 rows; loads on their way
        for (int j0 = wave; j0 < RG * quads; j0 += kWaves * PIECES) {
            u32x4 v[PIECES];
#pragma unroll
            for (int i = 0; i < PIECES; ++i) {
                const int j = min(j0 + kWaves * i, RG * quads - 1), c = min(b0 + 4 * (j / RG), nblk - 4);
                v[i] = __builtin_amdgcn_raw_buffer_load_b128(s_rsrc, ((64 * (j % RG) + lane) * nblk + c) * 4, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < PIECES; ++i) {
                const int j = min(j0 + kWaves * i, RG * quads - 1), c = min(b0 + 4 * (j / RG), nblk - 4) - b0;
                const int row = 64 * (j % RG) + lane, rows_of = row / (16 * RT), r16 = (row >> 4) - rows_of * RT;
                const int width = P::width_at(r16), first = P::first_at(r16);
                const int in = row - 16 * (rows_of * RT + first), lane16 = in / width, r = first + in % width;
                if (row < ROWS)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t bits = v[i][e];  // (a copy: a bit cast of a vector's element would take the first)
                        if (c + e >= 0 && c + e < nb)
                            *reinterpret_cast<f16 *>(scales + (((c + e) * kRowGroups + rows_of) * 16 + lane16) * (SD * 4) + r * 2) = (f16)__builtin_bit_cast(float, bits);
                    }
            }
        }
    }
    build_pair_table<kThreads>(smem, tid, code_lane);
    BROAD_LOAD_W(1, 0)
    wait_loads<P::count>();
    __builtin_amdgcn_s_waitcnt(0x0F70 | P::count);
    __syncthreads();
    BROAD_LOAD_X(STAGE)
    if constexpr (BLK == SCALES_UNIT) BROAD_LOAD_SCALES()
    BROAD_LOAD_W(1, 1)  // (behind the activations, as in the loop: its count of loads is exact)
    if constexpr (BLK) {
        BROAD_READ_SCALES(0)
    } else {
#pragma unroll
        for (int r = 0; r < RT; ++r) sc[0][r / 2][r & 1] = (f16)sc32[r];
    }
    BROAD_LUT(0, 0)
    BROAD_SCALE(0, 0)
    BROAD_LUT(0, 1)
#pragma unroll
    for (int t = 0; t < NT; ++t) BROAD_READ_B(0, 0, t)
    // Two units a turn and the odd one behind them: the compiler counts the loads on their way for the worst way into an
    // instruction, and with a branch around the second unit the first one's weights waited for the activations that had been
    // requested half a unit ago.  4096 x 11008 at 96 tokens 23.6 -> 20.6 us, 11008 x 4096 21.1 -> 19.7, with blocks of 64 4096 x
    // 4096 at 80 14.0 -> 13.1.  Not where the two units, one block of instructions then, spill.
    if constexpr (RT * NT <= (BLK ? 28 : 30)) {
        for (int pairs = units >> 1; pairs > 0; --pairs) {
            BROAD_STEP(0)
            BROAD_STEP(1)
        }
        if (units & 1) {
            BROAD_STEP(0)
        }
    } else {
        int left = units;
        do {
            BROAD_STEP(0)
            if (left > 1) {
                BROAD_STEP(1)
            } else {
                __builtin_amdgcn_s_waitcnt(0x0070);  // (one wait here, where the two paths' would differ)
            }
            left -= 2;
        } while (left > 0);
    }
    wait_loads<0>();  // (no activations on their way to where the sums go)
#undef BROAD_STEP
#undef BROAD_READ_SCALES
#undef BROAD_STORE_SCALES
#undef BROAD_LOAD_SCALES
#undef BROAD_READ_B
#undef BROAD_SCALE
#undef BROAD_LUT
#undef BROAD_LOAD_X
#undef BROAD_LOAD_W

    // ---- the sums of the k groups, added in their order: wave w ends with row tile w (of both row groups') ------
    constexpr int TILES = kRowGroups * RT, TW = (TILES + kWaves - 1) / kWaves;  // row tiles; of a wave: w and w + 8
    f32x4 sum[TW][NT];
    f32x4 *const red = reinterpret_cast<f32x4 *>(smem);
    constexpr int TP = red_tiles(RT, NT);  // token tiles a pass
#pragma unroll
    for (int t0 = 0; t0 < NT; t0 += TP) {
        __syncthreads();
#pragma unroll
        for (int t = t0; t < t0 + TP && t < NT; ++t)
#pragma unroll
            for (int r = 0; r < RT; ++r) red[((kg * TP + t - t0) * TILES + rg * RT + r) * 64 + lane] = acc[r][t];
        __syncthreads();
#pragma unroll
        for (int w = 0; w < TW; ++w) {
            const int r = wave + w * kWaves;
            if (r < TILES) {
#pragma unroll
                for (int t = t0; t < t0 + TP && t < NT; ++t) {
                    f32x4 v[kStepGroups];
#pragma unroll
                    for (int q = 0; q < kStepGroups; ++q) v[q] = red[((q * TP + t - t0) * TILES + r) * 64 + lane];
                    sum[w][t] = v[0];
#pragma unroll
                    for (int q = 1; q < kStepGroups; ++q) sum[w][t] += v[q];
                }
            }
        }
    }
    // parts of k: the last workgroup of a tile to arrive adds all parts' sums in k order
    const int item = (int)blockIdx.z * (int)gridDim.x + tile;
    if (split > 1 && !add_parts<kWaves, TILES, NT, NT <= 5 ? 3 : 2>(sum, a_ws, a_counters + item, (size_t)item, part, split, tid, wave, ticket)) return;
    store_tile<kWaves, TILES, NT, RT>(sum, reinterpret_cast<float *>(smem), tid, wave, a_out, a_residual, a_epilogue, row_base, a_m, tok_base, tokens);
}

struct OneMatrix {};
template <int RT, int NT, int BLK, class GROUPS>
hipError_t launch(const BroadPlan &plan, const GROUPS &groups, hipStream_t stream)
{
    static OptInFlag done[16];
    const auto fn = gemm_broad_kernel<RT, NT, BLK, GROUPS>;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 16) return hipErrorInvalidDevice;
    if ((e = ensure_lds_opt_in(done[dev], reinterpret_cast<const void *>(fn))) != hipSuccess) return e;
    const BroadArgs &a = plan.args;
    const size_t lds = lds_bytes(RT, NT, plan.blocks);
    hipLaunchKernelGGL(fn, dim3((unsigned)plan.tiles, (unsigned)plan.split, (unsigned)plan.tok_tiles), dim3(kThreads), lds, stream, a.q, a.x, a.code,
                       a.absmax, a.k, a.n, a.m, plan.part_steps, a.out, a.epilogue, a.residual, a.ws, a.counters, a.blk_shift, (int)lds - 16, groups);
    return hipGetLastError();
}
template <int RT, int NT>
hipError_t launch(const BroadPlan &plan, const BroadGroups *groups, hipStream_t stream)
{
    if constexpr (RT * NT <= 32) {
        if (groups) return launch<RT, NT, SCALES_ROW>(plan, *groups, stream);
        if (!plan.blocks) return launch<RT, NT, SCALES_ROW>(plan, OneMatrix(), stream);
        // (beside the table and the activations of 96 tokens there is no room for scales)
        if constexpr (NT <= 5)
            return plan.unit_scales ? launch<RT, NT, SCALES_UNIT>(plan, OneMatrix(), stream) : launch<RT, NT, SCALES_PART>(plan, OneMatrix(), stream);
        else return hipErrorInvalidConfiguration;
    } else {
        return hipErrorInvalidConfiguration;
    }
}
template <int RT>
hipError_t launch(const BroadPlan &plan, const BroadGroups *groups, hipStream_t stream)
{
    switch (plan.nt) {
    case 4: return launch<RT, 4>(plan, groups, stream);
    case 5: return launch<RT, 5>(plan, groups, stream);
    default: return launch<RT, 6>(plan, groups, stream);
    }
}
}  // namespace

bool plan_gemm_broad(int rows, int nt, int split, int blk_shift, BroadPlan *plan)
{
    BroadArgs &a = plan->args;
    const int rt = rows / (16 * kRowGroups);
    if (rows % (16 * kRowGroups) || rt < 2 || rt > 8 || rt == 7 || nt < 4 || nt > 6 || rt * nt > 32 || split < 1 || split > 65535) return false;
    const int steps = ceil_div_i(a.k, 64), tok_tiles = ceil_div_i(a.n, 16 * nt);
    if (tok_tiles > 65535) return false;
    if (16ll * nt * a.k * 2 > 0x7fffffff || (long long)rows * a.k / 2 > 0x7fffffff) return false;  // 32-bit offsets inside a tile
    plan->rt = rt, plan->nt = nt, plan->tiles = ceil_div_i(a.m, rows), plan->tok_tiles = tok_tiles;
    plan->part_steps = ceil_div_i(ceil_div_i(steps, kStepGroups), split) * kStepGroups;  // (whole units)
    plan->split = ceil_div_i(steps, plan->part_steps);  // (every part has steps)
    const long long items = (long long)plan->tiles * tok_tiles;
    plan->ws_bytes = plan->split > 1 ? (size_t)items * plan->split * kRowGroups * rt * nt * 1024 : 0;
    plan->n_counters = plan->split > 1 ? (size_t)items : 0;
    plan->blocks = 0, plan->unit_scales = false, a.blk_shift = 0;
    if (blk_shift >= 0) {
        if (a.k % 256 || a.k % (64 << blk_shift)) return false;  // (whole units, whole blocks)
        plan->blocks = broad_scale_blocks(rows, nt, plan->part_steps / kStepGroups, plan->split, blk_shift);
        plan->unit_scales = !plan->blocks || a.k >> (6 + blk_shift) < 4;  // (a part's are loaded four blocks at a time)
        if (plan->unit_scales) plan->blocks = 2 * kStepGroups;
        a.blk_shift = blk_shift;
    }
    return loop_bytes(rt, nt, plan->blocks) <= (size_t)kLdsLimit;
}

int broad_scale_blocks(int rows, int nt, int part_units, int parts, int blk_shift)
{
    // the blocks that a part touches: one more than it fills where it starts inside one
    const int steps = part_units * kStepGroups, size = 1 << blk_shift, blocks = ceil_div_i(steps, size) + (parts > 1 && steps % size ? 1 : 0);
    return loop_bytes(rows / (16 * kRowGroups), nt, blocks) <= (size_t)kLdsLimit ? blocks : 0;
}

size_t broad_lds_bytes(const BroadPlan &plan) { return lds_bytes(plan.rt, plan.nt, plan.blocks); }

bool plan_gemm_broad_groups(int rows, int nt, BroadPlan *plan, BroadGroups *groups)
{
    // (a.n: the largest group's tokens)
    if (!plan_gemm_broad(rows, nt, 1, -1, plan)) return false;
    long long items = 0;
    for (int e = 0; e < groups->n; ++e) {
        groups->item[e] = (int)items;
        items += (long long)plan->tiles * ceil_div_i(groups->tok_count[e], 16 * nt);
        if (items > 0x7fffffff) return false;
    }
    plan->tiles = (int)items, plan->tok_tiles = 1;
    return items > 0;
}

hipError_t launch_gemm_broad(const BroadPlan &plan, const BroadGroups *groups, hipStream_t stream)
{
    switch (plan.rt) {
    case 2: return launch<2>(plan, groups, stream);
    case 3: return launch<3>(plan, groups, stream);
    case 4: return launch<4>(plan, groups, stream);
    case 5: return launch<5>(plan, groups, stream);
    case 6: return launch<6>(plan, groups, stream);
    default: return launch<8>(plan, groups, stream);
    }
}

}  // namespace tuna
