// FP16-activation x 4-bit-codebook-weight GEMM for MANY tokens: tiles of 256 weight rows x up to 256 tokens (gemm_wide.hpp), divided
// between workgroups.  A launch has tiles of one kind, or of several (the groups of a grouped call, each with its tokens divided
// evenly into as few tiles as the launch's width allows; 256 x 256 tiles with narrower ones behind them).  A workgroup takes whole
// tiles and then a share of the k-steps of the remaining ones, or such a share alone; how tiles become workgroups is
// plan_gemm_wide's choice.  Tiles that nothing divides are gemm_wide_whole.hip's.
//
// What a divided tile costs: its partial sums and the wait for the other contributors, 8 us and what they weigh by wide_kinds_time's
// fit, and that shares which cross tiles meet fewer of their neighbours' activations in the L2.
#include "gemm_wide.hpp"

namespace tuna {

// Position in the k-steps of the shared tiles laid end to end: tile and step.
struct WidePos {
    int tile, step;
};
__device__ __forceinline__ bool before(const WidePos &a, const WidePos &b) { return a.tile < b.tile || (a.tile == b.tile && a.step < b.step); }
// (tile_end, weight_end: the lane's group's; with one group nothing is looked up)
__device__ __forceinline__ WidePos wide_share_begin(const WideArgs &a, int tile_end, unsigned weight_end, int share)
{
    if (share >= a.n_shares) return WidePos{a.tiles, 0};
    unsigned p = a.share_each * (unsigned)share + a.share_rest * (unsigned)share / (unsigned)a.n_shares;
    int group = 0, first = a.whole;
    if (a.n_groups > 1) {
        group = __builtin_popcountll(__ballot(weight_end <= p));
        if (group > 0) {
            first = max(first, __builtin_amdgcn_readlane(tile_end, group - 1));
            p -= (unsigned)__builtin_amdgcn_readlane((int)weight_end, group - 1);
        }
    }
    p /= wide_step_weight(a.g.nt[group]);
    const unsigned t = p / (unsigned)a.steps_total;
    return WidePos{first + (int)t, (int)(p - t * (unsigned)a.steps_total)};
}

// What a workgroup does with one tile, or with its share of one.
struct WideSegment {
    int place, tok0;  // the workgroup, the tile's first token
    int s0, s1;       // k-steps
    bool first;       // of the workgroup
    WidePos at, begin, end;  // of a divided tile: where this segment starts, and the workgroup's share
};
template <int NT, bool KTAIL, bool BLK, class ShareBegin>
__device__ __forceinline__ void wide_segment(const WideArgs &a, const WideTile &w, const WideSegment &seg, unsigned char *smem, const ShareBegin &share_begin)
{
    constexpr int kTiles = (NT + 3) / 4 * 4;  // (outputs are stored four token tiles at a time)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // (what follows from it is worked out again for each segment, not kept in registers that the loop lacks)
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int place = seg.place, tok0 = seg.tok0, s0 = seg.s0, s1 = seg.s1;
    const WidePos at = seg.at, begin = seg.begin, end = seg.end;
    unsigned char *const xs = smem + kLutBytes;
    // accumulators: [j][t] element v of lane (i16, g) is weight row 16 g + 4 v + j of the wave's 64, token 16 t + i16
    f32x4 acc[4][kTiles];
    wide_steps<NT, KTAIL, BLK>(acc, w, smem, a.code, seg.first, s0, s1, tid);

    // Straight-line code for 64 accumulators and every way a tile can end would be long, so the sums of four token tiles at a time go
    // through LDS (gemm_wide.hpp), where a loop can index them.
    const uint32_t lane_off = (uint32_t)(wave * 64 * 64 + lane) * 16u;  // of the partial sums: [wave][t][v][lane] of 16 bytes
    auto piece = [&](int t, int v) { return f32x4{acc[0][t][v], acc[1][t][v], acc[2][t][v], acc[3][t][v]}; };
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
        const WidePos head{at.tile, 0}, past{at.tile + 1, 0};
        int hi = place;
        WidePos lo_begin = begin;
        while (before(head, lo_begin)) lo_begin = share_begin(--lo);
        for (WidePos next = end; before(next, past); next = share_begin(hi + 1)) ++hi;
        lo_slot = before(lo_begin, head) ? 1 : 0;
        my_slot = before(begin, head) ? 1 : 0;
        const int others = hi - lo;
        unsigned *counter = a.counters + (at.tile - a.whole);
        volatile unsigned *ticket = reinterpret_cast<volatile unsigned *>(xs);
        if (tid == 0) *ticket = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        store = others == 1 && __builtin_amdgcn_readfirstlane((int)*ticket) == 1;
        if (!store) {
            const auto mine = slot(place);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, piece(t, v)), mine, (int)lane_off, (4 * t + v) * 1024, 16);
            }
            __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the partial sums have left this CU
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            __syncthreads();
            if (tid == 0) *ticket = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            store = __builtin_amdgcn_readfirstlane((int)*ticket) == others;
        }
        if (store && tid == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        own = others == 1;
        c_lo = lo, c_hi = hi;
        if (own) c_lo = c_hi = lo == place ? hi : lo;
        __syncthreads();  // the ticket has been read: its LDS is free
    }
    if (store) {
        unsigned char *const mine = xs + wave * 16384;
        WideOut out = wide_out(lane, a.out, a.residual, a.epilogue, a.m, tok0, w.tokens, w.row_base + wave * 64);
#pragma unroll 1
        for (int tb = 0; tb < NT; tb += 4) {
            auto at_piece = [&](int t, int v) { return wide_piece(mine, lane, t, v); };
            if (own) {
#pragma unroll
                for (int b = 0; b < kTiles; b += 4)
                    if (tb == b) {
#pragma unroll
                        for (int i = 0; i < 16; ++i) asm volatile("" : "+a"(acc[i & 3][b + (i >> 2)]));  // (here, not ahead of the loop)
#pragma unroll
                        for (int t = 0; t < 4; ++t)
#pragma unroll
                            for (int v = 0; v < 4; ++v) *at_piece(t, v) = piece(b + t, v);
                    }
            }
            if (c_lo <= c_hi) {
                f32x4 sum[4][4];
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int v = 0; v < 4; ++v) sum[t][v] = own ? *at_piece(t, v) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
                for (int c = c_lo; c <= c_hi; ++c) {
                    // (all loads issued before the first is awaited: the pass is a chain of memory round trips)
                    const auto src = slot(c);
                    f32x4 p[4][4];
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                            p[t][v] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(src, (int)lane_off, (4 * (tb + t) + v) * 1024, 16));
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int v = 0; v < 4; ++v) sum[t][v] += p[t][v];
                }
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int v = 0; v < 4; ++v) *at_piece(t, v) = sum[t][v];
            }
            wide_store(out, mine, lane);
        }
    }
}

template <bool KTAIL, bool BLK>
__global__ __launch_bounds__(kWideThreads, 1) void gemm_wide_kernel(const WideArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];  // the byte-pair table at LDS address 0, three stages of activations
    const int lane = threadIdx.x & 63;

    // Workgroups are dealt to the 8 XCDs in turn (workgroup L sits on XCD L % 8): an XCD takes consecutive tiles - the
    // token tiles of a few row tiles, which share the weights through its L2 - or consecutive shares.
    const int grid = (int)gridDim.x, xcd = (int)blockIdx.x & 7;
    const int place = xcd * (grid >> 3) + min(xcd, grid & 7) + ((int)blockIdx.x >> 3);

    int tile_end = 0;
    unsigned weight_end = 0;
    if (a.n_groups > 1) tile_end = a.g.tile_end[lane], weight_end = a.weight_end[lane];
    auto share_begin = [&](int share) { return wide_share_begin(a, tile_end, weight_end, share); };

    int tile = place, s0 = 0, s1 = a.steps_total;  // the segment at hand
    WidePos at{0, 0}, begin{0, 0}, end{0, 0};
    bool shared = a.whole <= place, first = true;
    if (a.n_shares) begin = share_begin(place), end = share_begin(place + 1);
    if (shared) {
        if (!a.n_shares) return;
        at = begin;
    }
    for (;;) {
        if (shared) {
            if (!before(at, end)) return;
            tile = at.tile;
            s0 = at.step;
            s1 = end.tile == at.tile ? end.step : a.steps_total;
        }
        // the tile's group, rows and tokens
        int group = 0, index = tile;
        if (a.n_groups > 1) {
            group = __builtin_popcountll(__ballot(tile_end <= tile));
            if (group > 0) index -= __builtin_amdgcn_readlane(tile_end, group - 1);
        }
        const int id = a.g.id[group], nt = a.g.nt[group], width = a.g.width[group], count = a.g.tok_count[group], per_row = a.g.tok_tiles[group];
        const int row_tile = index / per_row, tok_tile = index - row_tile * per_row, tok0 = a.g.tok_begin[group] + tok_tile * width;
        WideTile w;
        w.q = a.q + (size_t)id * (size_t)(a.m >> 3) * (size_t)(a.k >> 3) * 32;
        w.x = reinterpret_cast<const unsigned char *>(a.x) + (size_t)tok0 * (size_t)a.k * 2;
        w.absmax = a.absmax + (size_t)id * (size_t)a.m * (size_t)(BLK ? a.k >> (6 + a.blk_shift) : 1);
        w.m = a.m, w.k = a.k, w.row_base = row_tile * kWideRows;
        w.tokens = min(count - tok_tile * width, width);
        w.steps_total = a.steps_total, w.blk_shift = a.blk_shift;

        const WideSegment seg{place, tok0, s0, s1, first, at, begin, end};
        if (nt == 16) wide_segment<16, KTAIL, BLK>(a, w, seg, smem, share_begin);
        else if (nt == 14) wide_segment<14, KTAIL, BLK>(a, w, seg, smem, share_begin);
        else if (nt == 12) wide_segment<12, KTAIL, BLK>(a, w, seg, smem, share_begin);
        else if (nt == 10) wide_segment<10, KTAIL, BLK>(a, w, seg, smem, share_begin);
        else wide_segment<8, KTAIL, BLK>(a, w, seg, smem, share_begin);
        first = false;
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

bool plan_gemm_wide(int split, int cus, WidePlan *plan)
{
    WideArgs &a = plan->args;
    a.steps_total = ceil_div_i(a.k, 64);
    a.row_tiles = ceil_div_i(a.m, kWideRows);
    a.n_shares = 0;
    long long tiles = 0, weight = 0, widest = 0;  // widest: tiles of the first group's kind
    long long total[kMaxGroups];
    for (int e = 0; e < a.n_groups; ++e) {
        a.g.tok_tiles[e] = ceil_div_i(a.g.tok_count[e], a.g.width[e]);
        const int nt = wide_token_tiles(a.g.tok_count[e] < a.g.width[e] ? a.g.tok_count[e] : a.g.width[e]);
        a.g.nt[e] = split == 1 ? nt : wide_divided_token_tiles(nt);
        const long long here = (long long)a.row_tiles * a.g.tok_tiles[e];
        tiles += here;
        if (tiles > kWideMostTiles) return false;
        weight += here * a.steps_total * wide_step_weight(a.g.nt[e]);
        a.g.tile_end[e] = (int)tiles, total[e] = weight;
        if (a.g.nt[e] == a.g.nt[0]) widest += here;
    }
    if (tiles < 1) return false;
    a.tiles = (int)tiles;
    a.whole = (int)tiles;
    if (split > 1 && tiles * split <= 0xffff) {  // (more shares are no use, and their bounds are worked out in 32 bits)
        a.whole = 0;
        a.n_shares = (int)(tiles * split);
    } else if (split == 0) {
        wide_balance(tiles, widest, weight, wide_step_weight(a.g.nt[0]), a.steps_total, cus, &a.whole, &a.n_shares);
    }
    const long long skipped = (long long)a.whole * a.steps_total * wide_step_weight(a.g.nt[0]);
    long long divided_weight = a.n_shares ? weight - skipped : 0;
    if (divided_weight > 0x7fffffff) a.whole = (int)tiles, a.n_shares = 0, divided_weight = 0;  // (as above: whole tiles have no such bounds)
    // (a share is at least a step of a wide tile, so that every share between a tile's first and last has a part of it)
    const int most = (int)(divided_weight / wide_step_weight(a.g.nt[0]));
    if (a.n_shares > most) a.n_shares = most > 0 ? most : 1;
    if (a.n_shares) a.share_each = (unsigned)(divided_weight / a.n_shares), a.share_rest = (unsigned)(divided_weight % a.n_shares);
    for (int e = 0; e < kMaxGroups; ++e) {
        if (e >= a.n_groups) a.g.tile_end[e] = 0x7fffffff, a.weight_end[e] = 0xffffffffu;
        else a.weight_end[e] = a.n_shares && total[e] > skipped ? (unsigned)(total[e] - skipped) : 0u;
    }
    plan->grid = (unsigned)(a.n_shares ? a.n_shares : tiles);
    const long long divided = tiles - a.whole;
    bool alike = true;  // the divided tiles are of one kind: shares are equal parts of them
    for (int e = 0; e < a.n_groups; ++e) alike = alike && (a.g.tile_end[e] <= a.whole || a.g.nt[e] == a.g.nt[a.n_groups - 1]);
    a.slots = !a.n_shares || (alike && divided % a.n_shares == 0) ? 0 : alike && a.n_shares % divided == 0 ? 1 : 2;
    plan->ws_bytes = (size_t)a.n_shares * a.slots * kWideSlot;
    plan->n_counters = a.slots ? (size_t)divided : 0;
    return true;
}

hipError_t launch_gemm_wide(const WidePlan &plan, bool scale_blocks, hipStream_t stream)
{
    // (tiles that nothing divides: the kernels without bookkeeping)
    if (!plan.args.n_shares && (plan.args.n_groups == 1 || (!scale_blocks && plan.args.epilogue == TUNA_EPILOGUE_NONE)))
        return launch_gemm_wide_whole(plan.args, scale_blocks, stream);
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
