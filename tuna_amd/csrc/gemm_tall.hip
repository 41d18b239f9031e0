// Fused FP16 x 4-bit-codebook GEMM for decode batches of up to 64 tokens, weights read once: a workgroup is a tile of 16 RT rows
// (RT 2 .. 8) and all 16 NT tokens, in one of `split` parts of k.
//
// What bounds such a launch is its table reads and the activations it moves besides its weights.  Every row tile decodes against
// all tokens' activations, so these cross the cache, LDS and a CU's one return path once per row tile: per KB of weights 16 NT /
// ROWS KB times 4.  Loads into registers and LDS reads share that path (64 + 55 ns measured alone take 118 together), so tall
// tiles are what saves: as many rows as the CUs leave, chosen by the launch (28672 rows: 112 rows x 256 workgroups; 4096: 64
// rows x four parts of k).
//
// Eight waves split a tile's k-steps of 64 between them, not its rows: each has all 16 RT x 16 NT sums in registers (4 RT NT),
// private activations in LDS, and the loop has no barrier - a wave waits for its own loads alone.  Weights are on their way two
// steps ahead in registers, one dword per lane and row tile of a half step (rows 4 apart make a 16-byte load of four row tiles),
// activations one step ahead, table reads (65536 bytes: each of the 256 pairs of codes for each bank) two turns ahead of the MFMA
// that consumes them.  Each tile starts elsewhere in k (a hash of its number; workgroups that walk k in step ask the same memory
// channels: 101 us became 83 for the weights of 229376 x 4096 alone).  The waves' sums meet in LDS in wave order, parts of k in
// the workspace, added by the last to arrive in k order: results don't depend on the order of arrival.
//
// Measured against the launches that were chosen before, in us on one card (m x k at 16 NT tokens): 5120 x 13824: 19.0 -> 14.4,
// 28.7 -> 15.7, 28.0 -> 18.1, 33.8 -> 20.4 for NT 1 .. 4; for NT 2 .. 4 8192 x 28672: 39 -> 32, 55 -> 37, 54 -> 47; for NT 3 and
// 4 28672 x 4096: 27.8 -> 21.0, 27.7 -> 24.0, 4096 x 14336: 22.9 -> 16.5, 22.6 -> 18.5.  Floors, the weights at the rate of a large
// copy: 7, 23, 12 and 6.  Compute alone (table, scaling, MFMA) runs at 29 .. 36 ns per KB and CU, which is what is left.  Not better,
// and not kept: activations straight into LDS (pieces of 64 bytes 28.4 for 24.9 us at NT 4, of 128 equal), four steps ahead, a
// deeper ring of table reads, part of the decode on the VALU (5 .. 14 per cent slower).
//
// Scales finer than a row (BLK): a part's scales go to LDS once, two bytes each and a lane's of a block together, and a step's
// are read half a step ahead.  28672 x 4096 with blocks of 64: 19.2 -> 17.3 us at 16 tokens, 33.5 -> 25.9 at 64; 8192 x 28672 at 32
// tokens 57 -> 34.
#include "epilogue.hpp"
#include "row_pieces.hpp"

namespace tuna {

namespace {
constexpr int kWaves = 8, kThreads = 64 * kWaves;

// Token tiles whose sums the waves exchange at a time: one, in two buffers, or all.
constexpr int red_tiles(int rt, int nt)
{
    return kWaves * rt * nt * 1024 <= kLutBytes ? nt : 1;
}
constexpr size_t work_bytes(int rt, int nt)  // x of the waves; the waves' sums (from the table on); the outputs
{
    const size_t x = (size_t)kWaves * nt * 2048, out = (size_t)16 * nt * (16 * rt + 4) * 4;
    const size_t both = (size_t)kWaves * rt * red_tiles(rt, nt) * 1024 * (red_tiles(rt, nt) < nt ? 2 : 1);
    const size_t red = both > (size_t)kLutBytes ? both - kLutBytes : 0;
    const size_t a = x > red ? x : red;
    return a > out ? a : out;
}
// Scales in blocks of 64 << blk_shift weights: those of a tile's part of k lie behind the activations, two bytes each and a
// lane's of a block together: [block][16 lanes][scale_dwords], where the waves' sums go in the end.
constexpr int scale_dwords(int rt) { return rt <= 2 ? 1 : rt <= 4 ? 2 : 4; }
constexpr size_t lds_bytes(int rt, int nt, int blocks)
{
    const size_t with_scales = (size_t)kWaves * nt * 2048 + (size_t)blocks * 64 * scale_dwords(rt);
    const size_t work = work_bytes(rt, nt);
    return (size_t)kLutBytes + (with_scales > work ? with_scales : work) + 16;
}

// (separate scalars, the ones the first loads need in front: the first sixteen dwords arrive in scalar registers with the wave)
template <int RT, int NT, bool BLK>
__global__ __launch_bounds__(kThreads, 2) void gemm_tall_kernel(const uint8_t *a_q, const void *a_x, const float *a_code, const float *a_absmax,
                                                                     int a_k, int a_n, int a_m, int a_part_steps, void *a_out, int a_epilogue,
                                                                     const void *a_residual, float *a_ws, unsigned *a_counters, int a_blk_shift, int a_ticket)
{
    using P = Pieces<RT>;
    constexpr int NS = 2;      // steps whose weights are on their way
    constexpr int LR = 2;      // table reads of two turns are on their way
    constexpr int T = 2 * RT;  // turns of a step: a row tile of a half each
    constexpr int ROWS = 16 * RT;
    // kPairs: the loop goes two steps a turn with the odd one behind it, and the first loads are issued in the order of a step's.
    // A wait for a load is a wait for all loads before it, and the compiler counts for the worst way into an instruction: with a
    // branch around the second step (or another order of the first loads) each second step waited for weights requested one step
    // ago, not two.  4096 x 11008 at 16 tokens 10.4 -> 9.9 us, at 37 13.4 -> 13.0, 4096 x 14336 at 64 19.3 -> 18.3; 8192 x 8192 at
    // 16 with blocks of 64 13.6 -> 12.4.  Not where the registers don't allow it (the two steps are one block of instructions:
    // 7 x 4 tiles spill 40 registers, 25 -> 53 us), and not with scale blocks above 64 rows, whose scales take two passes over the
    // rows: there the loads that the branch lets go ahead of them are worth more (24576 x 4096 at 16 15.5 -> 17.2 us).
    constexpr bool kPairs = RT * NT <= 20 && (!BLK || RT <= 4);
    constexpr int XS = kPairs && RT > 6 ? RT - 3 : RT / 2;  // the turn in which the activations' exchange begins
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
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
        const int row = 16 * P::first(p) + P::width(p) * i16;
        w_off[p] = ((uint32_t)(row >> 3) * (uint32_t)kb_total + (uint32_t)g) * 32u + (uint32_t)(row & 7) * 4u;
    }
    // the slots of the last step beyond k read the last slot inside it (and their activations are zeros)
    const int slot_last = (kb_total - 1) & 7, s_tail = (a_k & 63) ? steps_total - 1 : -1;
    const uint32_t back0 = (uint32_t)max(0, g - slot_last) * 32u, back1 = (uint32_t)max(0, 4 + g - slot_last) * 32u;
    // activations: piece i is token lane / 8 + 8 i, 8-k slot lane % 8 of a step
    const uint32_t x_lane = ((uint32_t)(lane >> 3) * (uint32_t)a_k + (uint32_t)(lane & 7) * 8u) * 2u;
    const int x_k_left = a_k - (lane & 7) * 8;
    unsigned char *const xw = work + wave * (NT * 2048);
    unsigned char *const x_dst = xw + (lane >> 3) * 128 + (((lane & 7) ^ ((lane >> 3) & 7)) << 4);
    const int swz = (g ^ (i16 & 7)) << 4;
    const unsigned char *const x_frag0 = xw + i16 * 128 + swz, *const x_frag1 = xw + i16 * 128 + (64 ^ swz);

    const int tile = (int)blockIdx.x, part = (int)blockIdx.y, split = (int)gridDim.y, row_base = tile * ROWS;
    const int s0 = part * a_part_steps, s1 = min(s0 + a_part_steps, steps_total);
    const size_t rows_left = (size_t)(a_m - row_base);
    const __amdgpu_buffer_rsrc_t q_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(a_q) + (size_t)row_base * (size_t)(a_k >> 1), 0,
        (int)(uint32_t)min(rows_left * (size_t)(a_k >> 1), (size_t)0xffffffffu), 0x00020000);
    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        reinterpret_cast<unsigned char *>(const_cast<void *>(a_x)), 0, (int)((uint32_t)a_n * (uint32_t)a_k * 2u), 0x00020000);
    const int nblk = BLK ? a_k >> (6 + a_blk_shift) : 1;
    const __amdgpu_buffer_rsrc_t s_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a_absmax) + (size_t)row_base * (size_t)nblk, 0, (int)(uint32_t)min(rows_left * (size_t)nblk * 4, (size_t)0xffffffffu), 0x00020000);

    f32x4 acc[RT][NT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    // the wave's steps: s0 + wave, + 8 ..., from one that depends on the item on and around (workgroups that walk k in
    // step ask the same memory channels)
    const int mine = max(0, (s1 - s0 - wave + kWaves - 1) >> 3);
    const int s_first = min(s0 + wave, s1 - 1);  // (a wave without a step of its own loads one all the same)
    const unsigned turn = ((((unsigned)tile * 2654435761u) >> 16) * (unsigned)mine) >> 16;
    int s_w = s_first + 8 * (int)turn, s_x = s_w;
    auto next = [&](int s) { return s + 8 < s1 ? s + 8 : s_first; };

    uint32_t wq[NS][2][RT];
    u32x4 xr[2 * NT];
#define TALL_LOAD_W(set, h)                                                                                   \
    {                                                                                                         \
        const uint32_t at_ = (uint32_t)s_w * 256u + (h) * 128u - (s_w == s_tail ? ((h) ? back1 : back0) : 0u); \
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
        if (h) s_w = next(s_w);                                                                               \
    }
#define TALL_LOAD_X(i)                                                                                        \
    {                                                                                                         \
        const uint32_t l_ = s_x * 64 < x_k_left ? x_lane : 0x7fffffffu;                                       \
        xr[i] = __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, (int)(l_ + (uint32_t)(i) * 16u * (uint32_t)a_k), s_x * 128, 0); \
        if ((i) == 2 * NT - 1) s_x = next(s_x);                                                               \
    }
    // (the address path takes these one after the other: what the first step needs goes in front of the table, the rest behind)
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i) TALL_LOAD_X(i)
    TALL_LOAD_W(0, 0)
    float sc32[RT];
    if constexpr (!BLK) {
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int p = P::of(r);
            sc32[r] = __builtin_bit_cast(float, (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(
                                                    s_rsrc, (16 * P::first(p) + P::width(p) * i16 + r - P::first(p)) * 4, 0, 0));
        }
    }
    TALL_LOAD_W(0, 1)
    f16x2 sc[BLK ? 2 : 1][(RT + 1) / 2];  // of the step at hand and of the next one
    f16x8 fa[2], fb[2][NT];
    uint32_t lt[LR][4];
    // (turn tau of step u: row tile tau % RT of half tau / RT; u and tau may run over into the next step)
#define TALL_LUT(u, tau)                                                                                      \
    {                                                                                                         \
        const int u_ = ((u) + (tau) / T) % NS, h_ = (tau) % T / RT, r_ = (tau) % RT, l_ = ((u) * T + (tau)) % LR; \
        _Pragma("unroll") for (int b = 0; b < 4; ++b) lt[l_][b] = *reinterpret_cast<const lds_u32 *>(         \
            (uintptr_t)__builtin_amdgcn_perm(wq[u_][h_][r_], lane4, 0x0c0c0400u + 0x100u * b));               \
        if (r_ == RT - 1) TALL_LOAD_W(u_, h_) /* the half's registers are free */                             \
    }
#define TALL_SCALE(u, tau)                                                                                    \
    {                                                                                                         \
        const int r_ = (tau) % RT, l_ = ((u) * T + (tau)) % LR, f_ = (tau) & 1; /* (as for TALL_LUT) */       \
        _Pragma("unroll") for (int b = 0; b < 4; ++b)                                                         \
        {                                                                                                     \
            f16x2 v_;                                                                                         \
            if (r_ & 1) asm volatile("v_pk_mul_f16 %0, %1, %2 op_sel:[0,1] op_sel_hi:[1,1]" : "=v"(v_) : "v"(lt[l_][b]), "v"(sc[BLK ? ((u) + (tau) / T) % NS : 0][r_ / 2])); \
            else asm volatile("v_pk_mul_f16 %0, %1, %2 op_sel:[0,0] op_sel_hi:[1,0]" : "=v"(v_) : "v"(lt[l_][b]), "v"(sc[BLK ? ((u) + (tau) / T) % NS : 0][r_ / 2])); \
            fa[f_][2 * b] = v_[0];                                                                            \
            fa[f_][2 * b + 1] = v_[1];                                                                        \
        }                                                                                                     \
    }
#define TALL_READ_B(h, t) fb[h][t] = *reinterpret_cast<const f16x8 *>(((h) ? x_frag1 : x_frag0) + (t) * 2048);
/* a turn: the products of its row tile, the scaling of the next one, the table reads of the one after it; between them the
   activations: this step's second half from LDS, the next step's into it (one wave's LDS operations happen in order), its
   first half from there, and the step after it is requested */
#define TALL_STEP(u)                                                                                          \
    _Pragma("unroll") for (int tau = 0; tau < T; ++tau)                                                       \
    {                                                                                                         \
        _Pragma("unroll") for (int t = 0; t < NT; ++t) acc[tau % RT][t] =                                     \
            __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[tau & 1], fb[tau / RT][t], acc[tau % RT][t], 0, 0, 0);  \
        TALL_SCALE(u, tau + 1)                                                                                \
        TALL_LUT(u, tau + 2)                                                                                  \
        _Pragma("unroll") for (int t = 0; t < NT; ++t) if (tau == t * RT / (2 * NT)) TALL_READ_B(1, t)        \
        _Pragma("unroll") for (int i = 0; i < 2 * NT; ++i) if (tau == XS + i * RT / (2 * NT)) {               \
            *reinterpret_cast<u32x4 *>(x_dst + i * 1024) = xr[i];                                             \
            TALL_LOAD_X(i)                                                                                    \
        }                                                                                                     \
        _Pragma("unroll") for (int t = 0; t < NT; ++t) if (tau == 3 * RT / 2 + t * RT / (2 * NT)) TALL_READ_B(0, t) \
        if (BLK && tau == RT) TALL_READ_SCALES(((u) + 1) % NS)                                                \
        __builtin_amdgcn_sched_barrier(0);                                                                    \
    }
    // (the scales of the step after the one at hand)
#define TALL_READ_SCALES(set)                                                                                 \
    {                                                                                                         \
        s_sc = next(s_sc);                                                                                    \
        const lds_u32 *const from_ = sc_lane + ((s_sc >> a_blk_shift) - b0) * (16 * SD);                      \
        _Pragma("unroll") for (int j = 0; j < (RT + 1) / 2; ++j) sc[BLK ? (set) : 0][j] = __builtin_bit_cast(f16x2, from_[j]); \
    }
    constexpr int SD = scale_dwords(RT);
    const int b0 = BLK ? s0 >> a_blk_shift : 0;
    int s_sc = s_first + 8 * (int)turn;
    unsigned char *const scales = work + (size_t)kWaves * NT * 2048;
    const lds_u32 *const sc_lane = reinterpret_cast<const lds_u32 *>((uintptr_t)(uint32_t)(kLutBytes + kWaves * NT * 2048 + i16 * (SD * 4)));
    // Four blocks of a row a lane, 64 rows a wave: the LDS banks of a store are those of 16 lanes and two or four pairs of
    // row tiles.  (The last four of a row where four from here on would go beyond it: what is in front of the part or
    // behind it isn't stored.)
    constexpr int RG = (ROWS + 63) / 64, PIECES = 4;  // groups of 64 rows; loads on their way
    const int nb = BLK ? ((s1 - 1) >> a_blk_shift) + 1 - b0 : 0, pieces = RG * ((nb + 3) >> 2);
    u32x4 sv[BLK ? PIECES : 1];
    const auto load_scales = [&](int j0) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const int j = min(j0 + kWaves * i, pieces - 1), rg = RG == 1 ? 0 : j & 1, c = min(b0 + 4 * (RG == 1 ? j : j >> 1), nblk - 4);
            sv[BLK ? i : 0] = __builtin_amdgcn_raw_buffer_load_b128(s_rsrc, ((64 * rg + lane) * nblk + c) * 4, 0, 0);
        }
    };
    const auto store_scales = [&](int j0) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const int j = min(j0 + kWaves * i, pieces - 1), rg = RG == 1 ? 0 : j & 1, c = min(b0 + 4 * (RG == 1 ? j : j >> 1), nblk - 4) - b0;
            const int row = 64 * rg + lane, r16 = row >> 4;
            const int width = P::width_at(r16), first = P::first_at(r16);
            const int in = row - 16 * first, lane16 = in / width, r = first + in % width;
            if (row < ROWS)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t bits = sv[BLK ? i : 0][e];  // (a copy: a bit cast of a vector's element would take the first)
                    if (c + e >= 0 && c + e < nb)
                        *reinterpret_cast<f16 *>(scales + ((c + e) * 16 + lane16) * (SD * 4) + r * 2) = (f16)__builtin_bit_cast(float, bits);
                }
        }
    };
    const auto stage_scales = [&](int j0) {
        for (; j0 < pieces; j0 += kWaves * PIECES) {
            load_scales(j0);
            store_scales(j0);
        }
    };
    if constexpr (BLK && kPairs) load_scales(wave);
    if constexpr (BLK && !kPairs) stage_scales(wave);
    build_pair_table<kThreads>(smem, tid, code_lane);
    TALL_LOAD_W(1, 0)
    if constexpr (BLK && kPairs) {
        store_scales(wave);
        stage_scales(wave + kWaves * PIECES);
    }
    // (kPairs: the loads in the order of a step's, turn by turn: waiting for one of them is waiting for all before it)
    if (!kPairs) TALL_LOAD_W(1, 1)
    __syncthreads();
#pragma unroll
    for (int tau = 0; tau < T; ++tau) {
        if (kPairs && tau == T - 3) TALL_LOAD_W(1, 1)
#pragma unroll
        for (int i = 0; i < 2 * NT; ++i)
            if (tau == XS + i * RT / (2 * NT)) {
                *reinterpret_cast<u32x4 *>(x_dst + i * 1024) = xr[i];
                TALL_LOAD_X(i)
            }
        if (kPairs) __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (BLK) {
        const lds_u32 *const from = sc_lane + ((s_sc >> a_blk_shift) - b0) * (16 * SD);
#pragma unroll
        for (int j = 0; j < (RT + 1) / 2; ++j) sc[0][j] = __builtin_bit_cast(f16x2, from[j]);
    } else {
#pragma unroll
        for (int r = 0; r < RT; ++r) sc[0][r / 2][r & 1] = (f16)sc32[r];
    }
    TALL_LUT(0, 0)
    TALL_SCALE(0, 0)
    TALL_LUT(0, 1)
#pragma unroll
    for (int t = 0; t < NT; ++t) TALL_READ_B(0, t)
    if constexpr (kPairs) {
        for (int pairs = mine >> 1; pairs > 0; --pairs) {
            TALL_STEP(0)
            TALL_STEP(1)
        }
        if (mine & 1) {
            TALL_STEP(0)
        }
    } else if (mine > 0) {
        int left = mine;
        do {
            TALL_STEP(0)
            if (left > 1) {
                TALL_STEP(1)
            } else {
                __builtin_amdgcn_s_waitcnt(0x0070);  // (one wait here, where the two paths' would differ)
            }
            left -= NS;
        } while (left > 0);
    }
#undef TALL_STEP
#undef TALL_READ_SCALES
#undef TALL_READ_B
#undef TALL_SCALE
#undef TALL_LUT
#undef TALL_LOAD_X
#undef TALL_LOAD_W

    // ---- the waves' sums, added in wave order: wave r ends with row tile r ------------------------------------
    // (two buffers, the table's room among them: a pass is written while the one before it is read.  One buffer and two barriers a
    // pass: 28672 x 4096 at 64 tokens 25.6 us, now 24.4)
    f32x4 sum[1][NT];
    f32x4 *const red = reinterpret_cast<f32x4 *>(smem);
    constexpr int TP = red_tiles(RT, NT), BUF = kWaves * TP * RT * 64;  // token tiles a pass
    __syncthreads();
#pragma unroll
    for (int t0 = 0; t0 < NT; t0 += TP) {
        f32x4 *const buf = red + t0 / TP % 2 * BUF;
#pragma unroll
        for (int t = t0; t < t0 + TP && t < NT; ++t)
#pragma unroll
            for (int r = 0; r < RT; ++r) buf[((wave * TP + t - t0) * RT + r) * 64 + lane] = acc[r][t];
        __syncthreads();
        if (wave < RT) {
#pragma unroll
            for (int t = t0; t < t0 + TP && t < NT; ++t) {
                f32x4 v[kWaves];
#pragma unroll
                for (int w = 0; w < kWaves; ++w) v[w] = buf[((w * TP + t - t0) * RT + wave) * 64 + lane];
                sum[0][t] = v[0];
#pragma unroll
                for (int w = 1; w < kWaves; ++w) sum[0][t] += v[w];
            }
        }
    }
    // parts of k: the last workgroup of a tile to arrive adds all parts' sums in k order
    if (split > 1 && !add_parts<kWaves, RT, NT, 16 / NT>(sum, a_ws, a_counters + tile, (size_t)tile, part, split, tid, wave, ticket)) return;
    store_tile<kWaves, RT, NT, RT>(sum, reinterpret_cast<float *>(work), tid, wave, a_out, a_residual, a_epilogue, row_base, a_m, 0, a_n);
}

template <int RT, int NT, bool BLK>
hipError_t launch(const TallPlan &plan, hipStream_t stream)
{
    static OptInFlag done[16];
    const auto fn = gemm_tall_kernel<RT, NT, BLK>;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 16) return hipErrorInvalidDevice;
    if ((e = ensure_lds_opt_in(done[dev], reinterpret_cast<const void *>(fn))) != hipSuccess) return e;
    const TallArgs &a = plan.args;
    const size_t lds = lds_bytes(RT, NT, plan.part_blocks);
    hipLaunchKernelGGL(fn, dim3((unsigned)plan.tiles, (unsigned)plan.split), dim3(kThreads), lds, stream, a.q, a.x, a.code, a.absmax, a.k, a.n, a.m,
                       plan.part_steps, a.out, a.epilogue, a.residual, a.ws, a.counters, a.blk_shift, (int)lds - 16);
    return hipGetLastError();
}
template <int RT>
hipError_t launch(const TallPlan &plan, hipStream_t stream)
{
    const bool blk = plan.part_blocks != 0;
    switch (plan.nt) {
    case 1: return blk ? launch<RT, 1, true>(plan, stream) : launch<RT, 1, false>(plan, stream);
    case 2: return blk ? launch<RT, 2, true>(plan, stream) : launch<RT, 2, false>(plan, stream);
    case 3: return blk ? launch<RT, 3, true>(plan, stream) : launch<RT, 3, false>(plan, stream);
    default:
        if constexpr (RT <= 7) return blk ? launch<RT, 4, true>(plan, stream) : launch<RT, 4, false>(plan, stream);
        else return hipErrorInvalidConfiguration;
    }
}
}  // namespace

bool plan_gemm_tall(int row_tiles16, int nt, int split, int blk_shift, TallPlan *plan)
{
    TallArgs &a = plan->args;
    if (row_tiles16 < 2 || row_tiles16 > 8 || nt < 1 || nt > 4 || (row_tiles16 == 8 && nt == 4) || split < 1 || split > 65535) return false;
    const int rows = 16 * row_tiles16, steps = ceil_div_i(a.k, 64);
    if (16ll * nt * a.k * 2 > 0x7fffffff || (long long)rows * a.k / 2 > 0x7fffffff) return false;  // 32-bit offsets inside a tile
    plan->rt = row_tiles16, plan->nt = nt, plan->tiles = ceil_div_i(a.m, rows);
    plan->part_steps = ceil_div_i(steps, split);
    plan->split = ceil_div_i(steps, plan->part_steps);  // (every part has steps)
    plan->ws_bytes = plan->split > 1 ? (size_t)plan->tiles * plan->split * row_tiles16 * nt * 1024 : 0;
    plan->n_counters = plan->split > 1 ? (size_t)plan->tiles : 0;
    plan->part_blocks = 0;
    if (blk_shift >= 0) {
        // the blocks that a part touches: one more than it fills where it starts inside one
        const int size = 1 << blk_shift, nblk = a.k >> (6 + blk_shift);
        if (a.k % (64 << blk_shift) || nblk < 4) return false;
        plan->part_blocks = ceil_div_i(plan->part_steps, size) + (plan->split > 1 && plan->part_steps % size ? 1 : 0);
        a.blk_shift = blk_shift;
        if (lds_bytes(row_tiles16, nt, plan->part_blocks) > (size_t)kLdsLimit) return false;
    }
    return true;
}

size_t tall_lds_bytes(const TallPlan &plan) { return lds_bytes(plan.rt, plan.nt, plan.part_blocks); }

hipError_t launch_gemm_tall(const TallPlan &plan, hipStream_t stream)
{
    switch (plan.rt) {
    case 2: return launch<2>(plan, stream);
    case 3: return launch<3>(plan, stream);
    case 4: return launch<4>(plan, stream);
    case 5: return launch<5>(plan, stream);
    case 6: return launch<6>(plan, stream);
    case 7: return launch<7>(plan, stream);
    default: return launch<8>(plan, stream);
    }
}

}  // namespace tuna
