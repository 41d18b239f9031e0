// FP16-activation x 4-bit-codebook-weight GEMM for a decode batch (up to 64 tokens, or that many per group of a grouped
// launch) over many rows: the k-steps of all 256-row tiles are laid end to end and divided evenly over the workgroups.
//
//   * Four waves of 64 rows x all tokens (1 .. 4 token tiles of 16) per workgroup, up to two workgroups per compute unit.  As in
//     gemm_wide.hip a dword of the packed layout, through the decode table and scaled, is a lane's MFMA operand, and the
//     work of a k-step is one even sequence: per byte pair one scaling, one address, one table read, the MFMAs and fragment
//     reads dealt out between them, one barrier.
//   * Weights, activations and scales of the next four steps are on their way in registers, across tile and group
//     boundaries: a share streams without a gap.  A unit is those four steps, so that the loop is unrolled over the register
//     sets; the accumulators of a tile end with a unit, in code that exists once.
//   * The table (a copy per 32 lanes) takes the lower half of every 256 bytes of LDS and the activations' three stages the
//     upper halves: 64 KB in all.
//
// What bounds it: no single unit.  With one workgroup on a compute unit (256 shares: 28672 x 8192 at 37 tokens, eight experts
// of 28672 x 4096 at 16 each) the LDS is busy 28 .. 31 % of the cycles, the vector ALUs 23 .. 29 %, the matrix pipes 12 .. 21 %,
// HBM streams 2.8 .. 3.9 TB/s and the waves wait 40 % of their time at a counter or barrier; a second workgroup fills some
// of that (229376 x 4096 at 32 tokens 132 us on 256 shares, 107 on 512), but costs more for short launches.  Around the loop 6 us
// in all, and 3 .. 10 for handing over tiles that several shares contribute to (120064 x 3968 at 16 tokens: 46 us on 469 shares of
// a tile each, 59 on 512; without the hand-over 47).  No gain: each share's part of a tile walked from elsewhere in k on.
// Against the kernels the launches took before (general, streaming, many-token; one card, launch loop): 17920 x 23168 at 30
// tokens 154 -> 60 us, 32128 x 13312 at 36 tokens 129 -> 68, 28672 x 8192 at 37 tokens 51 -> 43; eight experts of 28672 x 4096 on 128 tokens 148 -> 128, and 100 on 512 shares (117 on 256 on that box).
#include "epilogue.hpp"

namespace tuna {

constexpr int kFlowThreads = 256;
constexpr int kFlowRows = 256;  // (flow_ws_bytes counts on it)
constexpr int kFlowRing = 4;  // k-steps requested ahead, and the k-steps of a unit

template <int NT>
constexpr size_t flow_slot_bytes() { return (size_t)kFlowRows * 16 * NT * 4; }

// Position in the units (kFlowRing k-steps of 64) of the tiles laid end to end.
struct FlowPos {
    int tile, unit;
};
__device__ __forceinline__ FlowPos flow_share_begin(const FlowArgs &a, int share)
{
    const unsigned total = (unsigned)a.tiles * (unsigned)a.units;
    const unsigned p = (unsigned)((unsigned long long)total * (unsigned)share / (unsigned)a.n_shares);
    return FlowPos{(int)(p / (unsigned)a.units), (int)(p % (unsigned)a.units)};
}

template <int NT, bool BLK>
__global__ __launch_bounds__(kFlowThreads, 2) void gemm_flow_kernel(const FlowArgs a)
{
    constexpr int XP = (NT + 1) / 2;          // 16-byte pieces of a step's activations per thread (an odd NT's last: half the threads)
    constexpr int STAGE_ROWS = 16 * NT;
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i16 = lane & 15, g = lane >> 4;
    const uint32_t lane4 = (uint32_t)(lane & 31) << 2;
    const int kb_total = a.k >> 3;
    const int nblk = BLK ? a.k >> (6 + a.blk_shift) : 1;

    const int grid = (int)gridDim.x, xcd = (int)blockIdx.x & 7;
    const int place = xcd * (grid >> 3) + min(xcd, grid & 7) + ((int)blockIdx.x >> 3);
    const FlowPos begin = flow_share_begin(a, place), end = flow_share_begin(a, place + 1);
    const int share_units = (end.tile - begin.tile) * a.units + end.unit - begin.unit;

    // per-lane offsets: weights (rows 4 i16 .. + 3 of the wave's 64, block column g of a half), activations (token tid / 8 +
    // 32 i, 8-k slot tid % 8), scales
    const uint32_t a_off = tile_weight_lane(tid, kFlowRows / 8, kb_total);
    uint32_t x_off[XP];
#pragma unroll
    for (int i = 0; i < XP; ++i) x_off[i] = ((uint32_t)((tid >> 3) + 32 * i) * (uint32_t)a.k + (uint32_t)(tid & 7) * 8u) * 2u;
    const int x_k_left = a.k - (tid & 7) * 8;  // the thread's slot of step s lies inside k while 64 s < x_k_left
    const uint32_t s_off = (uint32_t)(wave * 64 + 4 * i16) * (uint32_t)nblk * 4u;

    // load cursor: the tile whose steps are being requested (beyond the share's end it stays on the last step)
    int l_group = begin.tile / a.row_tiles, l_row = begin.tile - l_group * a.row_tiles;
    int l_unit = begin.unit, l_left = share_units;
    __amdgpu_buffer_rsrc_t q_rsrc, x_rsrc, s_rsrc;
    auto point = [&](int group, int row_tile) {
        const size_t first_row = (size_t)a.id[group] * (size_t)a.m + (size_t)row_tile * kFlowRows, rows_left = (size_t)a.m_total - first_row;
        q_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(a.q) + first_row * (size_t)(a.k >> 1), 0,
                                                   (int)(uint32_t)min(rows_left * (size_t)(a.k >> 1), (size_t)0xffffffffu), 0x00020000);
        x_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            reinterpret_cast<unsigned char *>(const_cast<void *>(a.x)) + (size_t)a.tok_begin[group] * (size_t)a.k * 2, 0,
            (int)((uint32_t)a.tok_count[group] * (uint32_t)a.k * 2u), 0x00020000);
        s_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.absmax) + first_row * (size_t)nblk, 0,
                                                   (int)(uint32_t)min(rows_left * (size_t)nblk * 4, (size_t)0xffffffffu), 0x00020000);
    };
    point(l_group, l_row);

    u32x4 wq[kFlowRing][2];
    u32x4 xr[kFlowRing][XP];
    u32x4 sq[BLK ? kFlowRing : 1];
    // Step `p` of the cursor's unit into register set `p`.  (Steps and slots beyond k: the activations are requested out
    // of range, which gives zeros, so what the weights there hold - of the last step, of the next block row, zeros at the
    // matrix' end - adds nothing.  The weights' offset is all in the vector register: flow_weight_offset says why.  The
    // uniform offsets of activations and scales stay inside a token's k values and a row's scales, so below the
    // descriptors' ends.)
#define FLOW_LOAD(p)                                                                                          \
    {                                                                                                         \
        const int s_ = l_unit * kFlowRing + (p), c_ = min(s_, a.steps_total - 1);                             \
        wq[p][0] = __builtin_amdgcn_raw_buffer_load_b128(q_rsrc, (int)flow_weight_offset(a_off, c_, 0), 0, 2); \
        wq[p][1] = __builtin_amdgcn_raw_buffer_load_b128(q_rsrc, (int)flow_weight_offset(a_off, c_, 1), 0, 2); \
        _Pragma("unroll") for (int i = 0; i < XP; ++i) xr[p][i] = __builtin_amdgcn_raw_buffer_load_b128(      \
            x_rsrc, s_ * 64 < x_k_left ? (int)x_off[i] : 0x7fffffff, c_ * 128, 0);                            \
        if constexpr (BLK) {                                                                                  \
            const int b_ = (c_ >> a.blk_shift) * 4;                                                           \
            _Pragma("unroll") for (int j = 0; j < 4; ++j) sq[p][j] =                                          \
                (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(s_rsrc, (int)(s_off + (uint32_t)(j * nblk) * 4u), b_, 0); \
        } else {                                                                                              \
            if ((p) == 0) sq[0] = __builtin_amdgcn_raw_buffer_load_b128(s_rsrc, (int)s_off, 0, 0);            \
        }                                                                                                     \
    }
    auto advance = [&]() {  // the cursor to the share's next unit (at its end it stays: what is loaded is not used)
        if (l_left > 1) {
            --l_left;
            if (++l_unit == a.units) {
                l_unit = 0;
                if (++l_row == a.row_tiles) l_row = 0, ++l_group;
                point(l_group, l_row);
                __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): no scalar load pending, whose order is free
            }
        }
    };
#pragma unroll
    for (int u = 0; u < kFlowRing; ++u) FLOW_LOAD(u)

    // decode table at LDS address 0: entry (byte << 8) | ((lane & 31) << 2) - a copy per 32 lanes, in the lower 128 bytes of
    // every 256; the upper 128 hold the activation stages: row r of the ring of three stages at r * 256 + 128
    {
        // (as in pair_table.hpp: a thread's entries share their low code, a wave's their high one)
        const int code_bits = (int)(uint32_t)__builtin_bit_cast(uint16_t, (f16)a.code[lane & 15]);
        const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(((tid >> 3) & 15) << 2, code_bits) << 16;
        const int high = __builtin_amdgcn_readfirstlane(tid >> 7);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t v = lo | (uint32_t)__builtin_amdgcn_readlane(code_bits, high + 2 * i);
            *reinterpret_cast<u32x4 *>(smem + ((tid >> 3) + 32 * i) * 256 + (tid & 7) * 16) = u32x4{v, v, v, v};
        }
        static_assert(kFlowThreads == 256, "eight entries of 128 bytes a thread");
    }
    unsigned char *const x_dst = smem + (tid >> 3) * 256 + 128 + (((tid & 7) ^ ((tid >> 3) & 7)) << 4);
    const int swz = (g ^ (i16 & 7)) << 4;
    const unsigned char *x_frag0 = smem + i16 * 256 + 128 + swz, *x_frag1 = smem + i16 * 256 + 128 + (64 ^ swz);
    constexpr int STAGE = STAGE_ROWS * 256;

    f32x4 acc[4][NT];
    f16x8 fa[2][4], fb[NT];
    uint32_t lt[16];
    f16x2 sc[4];
#define FLOW_LUT(l, set, half)                                                                                \
    lt[l] = *reinterpret_cast<const lds_u32 *>(                                                               \
        (uintptr_t)__builtin_amdgcn_perm(wq[set][half][(l) >> 2], lane4, 0x0c0c0400u + 0x100u * ((l) & 3)));
#define FLOW_SCALE(l, ab)                                                                                     \
    {                                                                                                         \
        f16x2 h_; /* (volatile: the compiler would sink it to the next step's block, where it is used) */     \
        asm volatile("v_pk_mul_f16 %0, %1, %2" : "=v"(h_) : "v"(lt[l]), "v"(sc[(l) >> 2]));                   \
        fa[ab][(l) >> 2][2 * ((l) & 3)] = h_[0];                                                              \
        fa[ab][(l) >> 2][2 * ((l) & 3) + 1] = h_[1];                                                          \
    }
#define FLOW_SCALES(set)                                                                                      \
    _Pragma("unroll") for (int j = 0; j < 4; ++j)                                                             \
    {                                                                                                         \
        const uint32_t e_ = sq[set][j];                                                                       \
        const f16 h_ = (f16)__builtin_bit_cast(float, e_);                                                    \
        sc[j] = f16x2{h_, h_};                                                                                \
    }
#define FLOW_STORE_X(set, off)                                                                                \
    _Pragma("unroll") for (int i = 0; i < XP; ++i)                                                            \
        if ((NT & 1) == 0 || i < XP - 1 || tid < 128)                                                         \
            *reinterpret_cast<u32x4 *>(x_dst + (off) + i * 32 * 256) = xr[set][i];
#define FLOW_READ_B(half, off, t) \
    fb[t] = *reinterpret_cast<const f16x8 *>(((half) ? x_frag1 : x_frag0) + (off) + (t) * 16 * 256);
    // Half h of the step at hand; `set` holds the next step.
#define FLOW_HALF(set, h)                                                                                     \
    _Pragma("unroll") for (int u = 0; u < 16; ++u)                                                            \
    {                                                                                                         \
        _Pragma("unroll") for (int i = u * 4 * NT / 16; i < (u + 1) * 4 * NT / 16; ++i)                       \
            acc[i & 3][i >> 2] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[h][i & 3], fb[i >> 2], acc[i & 3][i >> 2], 0, 0, 0); \
        if ((h) == 1 && u == 0) {                                                                             \
            if (BLK || (set) == 0) FLOW_SCALES(set)                                                           \
            __builtin_amdgcn_s_waitcnt(0xC07F | (6 << 8)); /* lgkmcnt: the stores of half 0 are done */       \
            __builtin_amdgcn_s_barrier();                                                                     \
            asm volatile("" ::: "memory");                                                                    \
        }                                                                                                     \
        FLOW_SCALE(u, (h) ^ 1)                                                                                \
        FLOW_LUT(u, set, h)                                                                                   \
        /* a token fragment is replaced by the next half's right behind its last MFMA */                      \
        _Pragma("unroll") for (int t = 0; t < NT; ++t)                                                        \
            if (u == (16 * (t + 1) + NT - 1) / NT - 1) FLOW_READ_B((h) ^ 1, (h) ? nxt : cur, t)              \
        if ((h) == 0 && u == 8) FLOW_STORE_X(set, nxt)                                                        \
        __builtin_amdgcn_sched_barrier(0);                                                                    \
    }

#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[j][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    int cur = 0, nxt = STAGE, nx2 = 2 * STAGE;
    FLOW_STORE_X(0, 0)
    FLOW_SCALES(0)
    __syncthreads();
#pragma unroll
    for (int l = 0; l < 16; ++l) FLOW_LUT(l, 0, 0)
#pragma unroll
    for (int l = 0; l < 16; ++l) FLOW_SCALE(l, 0)
#pragma unroll
    for (int l = 0; l < 16; ++l) FLOW_LUT(l, 0, 1)
#pragma unroll
    for (int t = 0; t < NT; ++t) FLOW_READ_B(0, 0, t)
    advance();
    FLOW_LOAD(0)

    FlowPos at = begin;
    int seg0 = begin.unit;  // first unit of the segment
    int todo = share_units, left = min(todo, a.units - begin.unit);
    while (todo > 0) {
#define FLOW_STEP(p)                                                                                          \
        {                                                                                                     \
            FLOW_HALF(((p) + 1) % kFlowRing, 0)                                                               \
            FLOW_HALF(((p) + 1) % kFlowRing, 1)                                                               \
            const int c_ = cur;                                                                               \
            cur = nxt, nxt = nx2, nx2 = c_;                                                                   \
        }
        do {
#pragma unroll
            for (int p = 0; p < kFlowRing; ++p) {
                FLOW_STEP(p)
                if (p + 1 == kFlowRing) advance();
                FLOW_LOAD((p + 1) % kFlowRing)
            }
        } while (--left != 0);
#undef FLOW_STEP
        // ---- the segment ends: a whole tile is stored, a shared one handed over as in gemm_wide.hip ----------------
        const int seg1 = at.tile == end.tile ? end.unit : a.units;
        todo -= seg1 - seg0;
        const int group = at.tile / a.row_tiles, row_base = (at.tile - group * a.row_tiles) * kFlowRows;
        const int tokens = a.tok_count[group], tok0 = a.tok_begin[group];
        const uint32_t lane_off = (uint32_t)(wave * (4 * NT) * 64 + lane) * 16u;  // of the partial sums: [wave][t][j][lane]
        int c_lo = 0, c_hi = -1, lo = place, lo_slot = 0, my_slot = 0;
        bool own = true, store = true;
        auto slot = [&](int share) {
            const int which = share == place ? my_slot : share == lo ? lo_slot : 0;
            return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<unsigned char *>(a.ws) + (size_t)(a.slots * share + which) * flow_slot_bytes<NT>(), 0,
                                                     (int)flow_slot_bytes<NT>(), 0x00020000);
        };
        if (seg0 != 0 || seg1 != a.units) {
            auto before = [](const FlowPos &p, int tile, int unit) { return p.tile < tile || (p.tile == tile && p.unit < unit); };
            int hi = place;
            while (!before(flow_share_begin(a, lo), at.tile, 1)) --lo;
            while (before(flow_share_begin(a, hi + 1), at.tile + 1, 0)) ++hi;
            lo_slot = before(flow_share_begin(a, lo), at.tile, 0) ? 1 : 0;
            my_slot = before(begin, at.tile, 0) ? 1 : 0;
            const unsigned others = (unsigned)(hi - lo);
            unsigned *counter = a.counters + at.tile;
            volatile unsigned *ticket = reinterpret_cast<volatile unsigned *>(smem + 255 * 256 + 128);
            // (two contributors: the one that finds the other arrived adds its partial sums to its own registers; more: the
            // last to arrive adds all of them from memory, in k order)
            __syncthreads();
            if (tid == 0) *ticket = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            store = others == 1 && *ticket == 1;
            if (!store) {
                const auto mine = slot(place);
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[j][t]), mine, (int)lane_off, (4 * t + j) * 1024, 16);
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
        }
        if (store) {
            f16 *outp = reinterpret_cast<f16 *>(a.out);
            const f16 *resp = reinterpret_cast<const f16 *>(a.residual);
            const int row = row_base + wave * 64 + 16 * g;
            f32x4 sum[NT][4];
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j) sum[t][j] = own ? acc[j][t] : f32x4{0.f, 0.f, 0.f, 0.f};
            // (several contributors' loads issued before the first is awaited: the pass is a chain of memory round trips)
            constexpr int CB = NT == 1 ? 4 : NT == 2 ? 2 : 1;
#pragma unroll 1
            for (int c = c_lo; c <= c_hi; c += CB) {
                f32x4 v[CB][NT][4];
#pragma unroll
                for (int b = 0; b < CB; ++b) {
                    const auto src = slot(min(c + b, c_hi));
#pragma unroll
                    for (int t = 0; t < NT; ++t)
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            v[b][t][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(src, (int)lane_off, (4 * t + j) * 1024, 16));
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int b = 0; b < CB; ++b)
                    if (c + b <= c_hi) {
#pragma unroll
                        for (int t = 0; t < NT; ++t)
#pragma unroll
                            for (int j = 0; j < 4; ++j) sum[t][j] += v[b][t][j];
                    }
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int tl = 16 * t + i16;
                const size_t tok = (size_t)(tok0 + tl);
                if (tl < tokens && row + 8 <= a.m)
                    store_features8(outp, resp, a.epilogue, tok, a.m, row, f32x4{sum[t][0][0], sum[t][1][0], sum[t][2][0], sum[t][3][0]},
                                    f32x4{sum[t][0][1], sum[t][1][1], sum[t][2][1], sum[t][3][1]});
                if (tl < tokens && row + 16 <= a.m)
                    store_features8(outp, resp, a.epilogue, tok, a.m, row + 8, f32x4{sum[t][0][2], sum[t][1][2], sum[t][2][2], sum[t][3][2]},
                                    f32x4{sum[t][0][3], sum[t][1][3], sum[t][2][3], sum[t][3][3]});
            }
        }
        __builtin_amdgcn_s_waitcnt(0x0070);  // (no load or scalar load pending: the loop's own waits then count from here)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[j][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        at = FlowPos{at.tile + 1, 0};
        seg0 = 0;
        left = min(todo, a.units);
    }
#undef FLOW_HALF
#undef FLOW_READ_B
#undef FLOW_STORE_X
#undef FLOW_SCALES
#undef FLOW_SCALE
#undef FLOW_LUT
#undef FLOW_LOAD
}

bool plan_gemm_flow(int nt, int shares, FlowPlan *plan)
{
    FlowArgs &a = plan->args;
    a.steps_total = ceil_div_i(a.k, 64);
    a.units = ceil_div_i(a.steps_total, kFlowRing);
    a.row_tiles = ceil_div_i(a.m, kFlowRows);
    const long long tiles = (long long)a.row_tiles * a.n_groups, units = tiles * a.units;
    if (nt < 1 || nt > 4 || shares < 1 || tiles < 1 || units > 0x7fffffff) return false;
    if (16ll * nt * a.k * 2 > 0x7fffffff || (long long)kFlowRows * a.k / 2 > 0x7fffffff) return false;  // 32-bit offsets inside a tile
    a.tiles = (int)tiles;
    plan->nt = nt;
    a.n_shares = shares > units ? (int)units : shares;
    a.slots = flow_slots(a.tiles, a.n_shares);
    plan->ws_bytes = flow_ws_bytes(a.tiles, a.n_shares, nt);
    plan->n_counters = a.slots ? (size_t)tiles : 0;
    return true;
}

hipError_t launch_gemm_flow(const FlowPlan &plan, bool scale_blocks, hipStream_t stream)
{
    typedef void (*Fn)(const FlowArgs);
    static const Fn kFn[2][4] = {{gemm_flow_kernel<1, false>, gemm_flow_kernel<2, false>, gemm_flow_kernel<3, false>, gemm_flow_kernel<4, false>},
                                 {gemm_flow_kernel<1, true>, gemm_flow_kernel<2, true>, gemm_flow_kernel<3, true>, gemm_flow_kernel<4, true>}};
    hipLaunchKernelGGL(kFn[scale_blocks][plan.nt - 1], dim3((unsigned)plan.args.n_shares), dim3(kFlowThreads), 65536, stream, plan.args);
    return hipGetLastError();
}

}  // namespace tuna
