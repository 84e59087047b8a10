// Selection for batches whose roots have few visitors each (at most kBlockVisitors): a block a root.
//
// What it computes is what omk_select_kernels.h computes (see there), for crowds that fit a wavefront: a node's
// visitors are one per lane, a subtree's lists and work items live in LDS, and a wavefront that has settled a node goes
// on with the child most of them chose and leaves the others to the idle wavefronts of its block.  Nothing is shared
// between blocks: no queue in memory, no reset before the launch, no wait that could have to give up.  Handing a node
// on costs an LDS round trip where the queue in memory takes 3 us (release, poll, acquire, the item's own trip).
//
// What bounds it is the latency of a chain of crowded nodes: one dependent trip to memory a level, and the instruction
// issue of the wavefront that settles the node.
#pragma once

#include "omk_select_kernels.h"

namespace omk {

constexpr int kBlockVisitors = kBlockMax;  // of one root: a lane each
constexpr int kBlockDepth = 63;     // deepest bound for which the blocks send rows to the host themselves
constexpr int kBlockWaves = 16;     // wavefronts of a block: 128 registers each

// A node and the visitors that reached it: entries [off, off + m) of the block's list.
struct BlockItem {
    int node, np, cb, cc, depth, off, m, unused;
};

// What a wavefront settles a node in: the children that matter, one per lane, in child order.
template <int RMAX>
struct BlockScratch {
    int child[kWave];  // index in the node
    int n[kWave], vl[kWave], sx[kWave], sy[kWave];
    float w[kWave], p[kWave], q2[kWave];
    int start[kWave];        // first place of the child's visitors in the node's list
    int taken[kWave];        // its visits
    uint64_t entry[2 * kWave + 8];  // merge_heads: the entries being put in order
    uint32_t order[kWave];   // per visitor: child << 21 | number of the visit
    uint8_t lane_of[RMAX * kWave];  // where child i is listed
};

template <int RMAX, bool ROWS>
struct BlockLds {
    int head, tail, open;  // tickets taken, items handed out, visitors that have not reached their leaf
    int ready[kBlockVisitors];  // item i lies in slot i once this is i + 1.  A block hands out at most kBlockVisitors items in
                                // all: each but the first (of the lone roots: their own) makes one group more of the
                                // visitors, who are in no more groups than they are.  So no slot is used twice, and the
                                // tickets beyond wait at slots that never hold their number
    BlockItem item[kBlockVisitors];
    int list[kBlockVisitors];  // visitors by number, partitioned in place
    int trav[kBlockVisitors];  // traversal of a visitor
    // the rows for the host
    int len[ROWS ? kBlockVisitors : 1], leaf[ROWS ? kBlockVisitors : 1], kids[ROWS ? kBlockVisitors : 1],
        visits[ROWS ? kBlockVisitors : 1];
    int path[ROWS ? kBlockVisitors : 1][kBlockDepth + 2];
    BlockScratch<RMAX> scratch[kBlockWaves];
};

// (key, position) of the best of per-lane candidates, like wave_best; without the scalar unit until the end.
__device__ __forceinline__ void wave_best_fast(uint32_t bk, uint32_t bpos, uint32_t &mk, uint32_t &mpos) {
    const uint32_t top = wave_max_all(bk);
    uint64_t tie = __ballot(bk == top);
    mk = (uint32_t)uniform((int)top);
    if (tie & (tie - 1ull)) {
        mpos = wave_min_u32(bk == top ? bpos : 0xFFFFFFFFu);
        return;
    }
    mpos = (uint32_t)__builtin_amdgcn_readlane((int)bpos, __ffsll((long long)tie) - 1);
}

// m visitors of a node settled over the n0 children listed in `s`, one per lane: order[q] for every visitor, and the
// visits of the lane's child.  The score a child shows its j-th visitor of this node depends on nothing but j, and where
// no child's scores increase with j the serial order is the merge of the children's lists.  Twice 64 entries are worked
// out at once, as many of every child (64 of two children, two of 64), independently of each other where the serial
// loop waits for two divisions a visitor.  An entry that is not worked out comes after the last one of its child that is:
// the entries up to the first of these last ones are the next visitors', the best first, and every one finds its place
// by counting the ones before it.  What is left goes on from there.
// floor_key: the children that are not listed have no entry above it.
// False (with `order` overwritten) when a child's entries are not in order, or when an entry at or below floor_key or none
// would be next: the caller plays one visitor after the other.
template <int RMAX, bool RAVE>
__device__ __forceinline__ bool merge_heads(BlockScratch<RMAX> &s, int n0, int m, float ep, uint32_t uvl,
                                            uint32_t floor_key, int lane, int &visits) {
    visits = 0;
    if (n0 == 0) return false;
    const int log_e = n0 <= 1 ? 6 : 6 - (32 - __clz(n0 - 1));  // a child's lanes: the largest power of two that fits
    const int E = 1 << log_e;
    const int c = lane >> log_e, j0 = lane & (E - 1);
    const bool mine = c < n0;
    int cn = 0, cvl = 0;
    float cw = 0.0f, cp = 0.0f, cq2 = 0.0f;
    if (mine) {
        cn = s.n[c];
        cw = s.w[c];
        cp = s.p[c];
        cvl = s.vl[c];
        if (RAVE) cq2 = s.q2[c];
    }
    const bool proven =
        __ballot(mine && !keys_provably_monotone<RAVE>(cn, cw, cp, cvl, cq2, ep, uvl, m - 1)) == 0ull;
    s.taken[lane] = 0;
    wave_sync_memory();
    int base = 0;  // visits of the lane's child so far
    for (int done = 0; done < m;) {
        const int need = m - done;
        uint32_t key[2] = {0u, 0u}, pos[2] = {0u, 0u};
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (h == 1 && E >= need) break;  // uniform: nobody gets more than the first E
            entry_key<1, RAVE>(cn, cw, cp, cvl, cq2, ep, uvl, base + h * E + j0, 0, key[h], pos[h]);
            key[h] = mine && h * E + j0 < need ? key[h] : 0u;  // (nobody gets more than `need`)
        }
        if (!proven) {
            const uint32_t p0 = (uint32_t)__shfl_up((int)key[0], 1, kWave), q0 = (uint32_t)__shfl_up((int)pos[0], 1, kWave);
            const uint32_t l0 = (uint32_t)__shfl((int)key[0], lane + E - 1, kWave), m0 = (uint32_t)__shfl((int)pos[0], lane + E - 1, kWave);
            const uint32_t p1 = (uint32_t)__shfl_up((int)key[1], 1, kWave), q1 = (uint32_t)__shfl_up((int)pos[1], 1, kWave);
            bool bad = j0 > 0 && comes_before(key[0], pos[0], p0, q0);
            if (key[1] != 0u) bad |= j0 > 0 ? comes_before(key[1], pos[1], p1, q1) : comes_before(key[1], pos[1], l0, m0);
            if (__ballot(mine && bad)) return false;
        }
        // ---- up to the first of the children's last entries (those that can be needed are all there, or it counts) ----
        // (equal keys: first scan before second, then the children's order, then the visits')
        uint32_t low[2];
#pragma unroll
        for (int h = 0; h < 2; h++) low[h] = (pos[h] << 24) | (uint32_t)(c << 16) | (uint32_t)(base + h * E + j0);
        const uint32_t last = j0 == E - 1 && 2 * E < need ? key[1] : 0u;
        const uint32_t bar = (uint32_t)uniform((int)wave_max_all(last));
        const uint32_t bar_low = bar == 0u ? 0u : wave_min_u32(last == bar ? low[1] : 0xFFFFFFFFu);
        bool in[2];
#pragma unroll
        for (int h = 0; h < 2; h++) in[h] = key[h] > floor_key && (key[h] > bar || (key[h] == bar && low[h] <= bar_low));
        const uint64_t in0 = __ballot(in[0]), in1 = __ballot(in[1]);
        const int n_in0 = __popcll(in0), total = n_in0 + __popcll(in1);
        if (total == 0) return false;
        const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
        for (int h = 0; h < 2; h++)
            if (in[h])
                s.entry[h == 0 ? __popcll(in0 & below) : n_in0 + __popcll(in1 & below)] = ((uint64_t)~key[h] << 32) | low[h];
        if (lane < 8) s.entry[total + lane] = ~0ull;
        wave_sync_memory();
        // smaller = played earlier, all different; a lane has one of them, or two
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (h * kWave >= total) break;  // uniform
            const int at = h * kWave + lane;
            const uint64_t e = at < total ? s.entry[at] : ~0ull;
            int rank = 0;
            for (int e0 = 0; e0 < total; e0 += 8) {
                uint64_t o[8];
#pragma unroll
                for (int u = 0; u < 8; u++) o[u] = s.entry[e0 + u];
#pragma unroll
                for (int u = 0; u < 8; u++) rank += o[u] < e ? 1 : 0;
            }
            if (at < total && rank < need) {
                const int w = (int)((e >> 16) & 63u);
                s.order[done + rank] = ((uint32_t)s.child[w] << 21) | (uint32_t)(e & 0xFFFFu);
                atomicAdd(&s.taken[w], 1);
            }
        }
        wave_sync_memory();
        base = s.taken[c];
        done += total < need ? total : need;
    }
    visits = s.taken[lane];
    return true;
}

// Blocks [0, n_items): a root with several visitors each.  The blocks behind them: up to kBlockWaves roots with one
// visitor each.  One thread leaves the scheduler words as a reset would have.  ROWS: the block sends its visitors' rows
// to the host when the last of them has reached its leaf.
template <int RMAX, bool RAVE, bool ROWS>
__global__ __launch_bounds__(kBlockWaves *kWave) void k_select_blocks(ForestDev f, SelectArgs a, int n_items, int n_singles,
                                                                      LoneOut out) {
    constexpr int F = RMAX * kWave;
    __shared__ BlockLds<RMAX, ROWS> s;
    const int lane = threadIdx.x & (kWave - 1), wv = uniform((int)threadIdx.x >> 6);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *a.n_singles = n_singles;
        *a.truncated_next = 0;
        a.sched_wait[1] = 0;
        if (a.times) a.times[0] = (int)(wall_clock64() & 0x7FFFFFFF);
    }
    // ---- the block's visitors ----
    int n_here = 0;
    if (wv == 0) {
        s.ready[lane] = 0;
        s.list[lane] = lane;
        int items = 1;
        if ((int)blockIdx.x < n_items) {
            const Item root = a.items0[blockIdx.x];
            n_here = uniform(root.m);
            if (lane < n_here) s.trav[lane] = a.seg0[root.off + lane];
            if (ROWS && lane < n_here) s.path[lane][0] = root.node;
            if (lane == 0) {
                const int2 sp = f.span[root.node];
                s.item[0] = BlockItem{root.node, f.N[root.node], sp.x, sp.y, 0, 0, n_here, 0};
                s.ready[0] = 1;
            }
        } else {
            const int first = ((int)blockIdx.x - n_items) * kBlockWaves;
            n_here = n_singles - first < kBlockWaves ? n_singles - first : kBlockWaves;
            items = n_here;
            if (lane < n_here) {
                const Item root = a.singles0[first + lane];
                const int2 sp = f.span[root.node];
                s.trav[lane] = root.off;
                if (ROWS) s.path[lane][0] = root.node;
                s.item[lane] = BlockItem{root.node, f.N[root.node], sp.x, sp.y, 0, lane, 1, 0};
                s.ready[lane] = lane + 1;
            }
        }
        if (lane == 0) {
            s.head = 0;
            s.tail = items;
            s.open = n_here;
        }
    }
    __syncthreads();
    BlockScratch<RMAX> &my = s.scratch[wv];
    const uint32_t uvl = a.vl > 0 ? (uint32_t)a.vl : 0u;
    for (;;) {
        const int ticket = take_ticket(&s.head, lane);
        bool got = false;
        for (;;) {  // (ends: a visitor goes down one level with every node settled)
            const int open = uniform(__hip_atomic_load(&s.open, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
            const int r = uniform(__hip_atomic_load(&s.ready[ticket & (kBlockVisitors - 1)], __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_WORKGROUP));
            got = r == ticket + 1;
            if (got || open <= 0) break;
            __builtin_amdgcn_s_sleep(1);
        }
        if (!got) break;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        const BlockItem it = s.item[ticket & (kBlockVisitors - 1)];
        int node = uniform(it.node), np = uniform(it.np), cb = uniform(it.cb), cc = uniform(it.cc);
        int depth = uniform(it.depth), off = uniform(it.off), m = uniform(it.m);
        int v = 0, t = 0;  // the lane's visitor and its traversal
        if (lane < m) {
            v = s.list[off + lane];
            t = s.trav[v];
        }
        // ---- down from this node, with the child most visitors choose ----
        for (;;) {
            const long long tr0 = a.trace ? wall_clock64() : 0ll;
            bool leaf = cc <= 0 || depth >= a.max_depth;
            int run_child = -1, run_np = 0, run_sx = 0, run_sy = 0;
            int n0 = 0, visits = 0;  // of the lane's listed child
            bool serial = false;
            Kids<RMAX, RAVE> k;
            int2 sp[RMAX];
            if (!leaf) {
                int nelig = cc;
                if (a.pw) {
                    const int kk = ceil_sqrt_i32(np);
                    nelig = kk < cc ? kk : cc;
                }
                {
                    // one trip to memory: statistics, legality bits and child ranges together (a lane without a child
                    // asks for the last one's)
                    const int32_t *const bN = f.N + cb, *const bVL = f.VL + cb;
                    const float *const bW = f.W + cb, *const bP = f.P + cb, *const bq = RAVE ? f.q2 + cb : nullptr;
                    const int2 *const bs = f.span + cb;
                    uint32_t word[RMAX];
#pragma unroll
                    for (int r = 0; r < RMAX; r++) {
                        word[r] = 0u;
                        k.n[r] = k.vl[r] = 0;
                        k.w[r] = k.p[r] = k.q2[r] = 0.0f;
                        sp[r] = int2{0, 0};
                        if (r * kWave >= nelig) continue;  // uniform
                        const int i = r * kWave + lane;
                        const uint32_t at = (uint32_t)(i < nelig ? i : nelig - 1) & 0xFFFFu;
                        word[r] = f.legal ? f.legal[((uint32_t)cb + at) >> 5] : 0xFFFFFFFFu;
                        k.n[r] = bN[at];
                        k.w[r] = bW[at];
                        k.p[r] = bP[at];
                        k.vl[r] = bVL[at];
                        if (RAVE) k.q2[r] = bq[at];
                        sp[r] = bs[at];
                    }
                    const float ep = a.c_puct * sqrtf((float)np);
#pragma unroll
                    for (int r = 0; r < RMAX; r++) {
                        const int i = r * kWave + lane;
                        k.part[r] = i < nelig && ((word[r] >> ((uint32_t)(cb + i) & 31u)) & 1u);
                        k.k1[r] = k.k2[r] = 0u;
                        if (r * kWave >= nelig) continue;  // uniform
                        child_keys<RAVE>(k.n[r], k.w[r], k.p[r], k.vl[r], k.q2[r], ep, k.k1[r], k.k2[r]);
                        k.k1[r] = k.part[r] ? k.k1[r] : 0u;
                        k.k2[r] = k.part[r] ? k.k2[r] : 0u;
                    }
                    // All of them have arrived, the child ranges too (vmcnt(0)), and the compiler knows it.  Else it may wait
                    // for a round that was skipped where the loop comes round, and with it for the stores and atomics of
                    // the level before its next loads: 8 visitors of a Gomoku tree 35 or 38 us, by how registers fall.
                    __builtin_amdgcn_s_waitcnt(0x0F70);
                }
                const float ep = a.c_puct * sqrtf((float)np);
                bool odd = false;  // (select_group: such a node is played one visitor after the other)
                if (RAVE) {
                    bool any1 = false, o = false;
#pragma unroll
                    for (int r = 0; r < RMAX; r++) {
                        any1 |= k.k1[r] != 0u;
                        o |= k.part[r] && !(fabsf(k.w[r]) <= 3.0e38f);
                    }
                    odd = __ballot(o) != 0ull;
                    if (__ballot(any1) == 0ull) {  // no real score in the first scan: the second is never run
#pragma unroll
                        for (int r = 0; r < RMAX; r++) k.k2[r] = 0u;
                    }
                }
                uint32_t bk, bpos, hk, hp;
                lane_best<RMAX, RAVE>(k, lane, bk, bpos);
                wave_best_fast(bk, bpos, hk, hp);
                const int best = (int)(hp >= (uint32_t)F ? hp - (uint32_t)F : hp);
                serial = true;
                if (hk != 0u && (m == 1 || a.vl <= 0)) {
                    run_child = best;
                } else if (hk != 0u && !odd) {
                    // ---- does the best child win every time?  (single_run) ----
                    int tn = 0, tvl = 0;
                    float tw = 0.0f, tp = 0.0f, tq2 = 0.0f;
#pragma unroll
                    for (int r = 0; r < RMAX; r++) {
                        if (r == (best >> 6)) {
                            tn = k.n[r];
                            tw = k.w[r];
                            tp = k.p[r];
                            tvl = k.vl[r];
                            tq2 = k.q2[r];
                        }
                    }
                    const int bl = best & 63;
                    const int bn = __builtin_amdgcn_readlane(tn, bl), bvl = __builtin_amdgcn_readlane(tvl, bl);
                    const float bw = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tw), bl));
                    const float bp = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tp), bl));
                    const float bq2 = RAVE ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tq2), bl)) : 0.0f;
                    uint32_t lk, lp;
                    entry_key<RMAX, RAVE>(bn, bw, bp, bvl, bq2, ep, uvl, m - 1, best, lk, lp);
                    lk = (uint32_t)uniform((int)lk);
                    auto heads = [&](uint32_t T) {
                        int c = 0;
#pragma unroll
                        for (int r = 0; r < RMAX; r++) c += __popcll(__ballot(umax32(k.k1[r], k.k2[r]) >= T));
                        return c;
                    };
                    // its entry for the last visitor comes before every other child's next one, and they are in order
                    uint32_t from = lk < hk ? lk : hk, floor_key = from - 1u;
                    int n_heads = from != 0u ? heads(from) : 0;
                    if (n_heads == 1 && entries_in_order<RMAX, RAVE>(bn, bw, bp, bvl, bq2, ep, uvl, best, m, lane))
                        run_child = best;
                    if (run_child < 0) {
                        // ---- the children that can be chosen, one per lane ----
                        // those whose next entry is not below that one (with the best child's entries in order nobody
                        // else is; merge_heads sees to it), or, if there are too many or it is not real, the m best
                        if (from == 0u || n_heads > kWave) {
                            from = first_heads<RMAX, RAVE>(k, bk, m);
                            floor_key = 0u;
                        }
                        if (from != 0u) {
#pragma unroll
                            for (int r = 0; r < RMAX; r++) {
                                const bool in = umax32(k.k1[r], k.k2[r]) >= from;
                                const uint64_t cm = __ballot(in);
                                if (in) {
                                    const int cl = n0 + __popcll(cm & ((1ull << lane) - 1ull));
                                    my.child[cl] = r * kWave + lane;
                                    my.n[cl] = k.n[r];
                                    my.w[cl] = k.w[r];
                                    my.p[cl] = k.p[r];
                                    my.vl[cl] = k.vl[r];
                                    if (RAVE) my.q2[cl] = k.q2[r];
                                    my.sx[cl] = sp[r].x;
                                    my.sy[cl] = sp[r].y;
                                    my.lane_of[r * kWave + lane] = (uint8_t)cl;
                                }
                                n0 += __popcll(cm);
                            }
                            wave_sync_memory();
                            serial = !merge_heads<RMAX, RAVE>(my, n0, m, ep, uvl, floor_key, lane, visits);
                        }
                    }
                }
                if (run_child < 0 && serial) {
                    // ---- one visitor after the other (no real score, values that are not finite, a child that was
                    // not listed) ----
                    int cnt[RMAX];
#pragma unroll
                    for (int r = 0; r < RMAX; r++) cnt[r] = 0;
                    for (int done = 0; done < m; done++) {
                        const int i = wave_pick<RMAX, RAVE>(k, lane, bk, bpos);
                        if (i < 0) {  // no child takes part, for every visitor
                            leaf = true;
                            break;
                        }
                        if (a.vl <= 0) {  // nothing changes between visitors
                            run_child = i;
                            break;
                        }
                        if (lane == (i & 63)) {
#pragma unroll
                            for (int r = 0; r < RMAX; r++) {
                                if (r == (i >> 6)) {
                                    my.order[done] = ((uint32_t)i << 21) | (uint32_t)cnt[r];
                                    cnt[r]++;
                                    k.vl[r] = (int)((uint32_t)k.vl[r] + uvl);
                                    score_round<RMAX, RAVE>(k, r, ep);
                                }
                            }
                            lane_best<RMAX, RAVE>(k, lane, bk, bpos);
                        }
                    }
                    if (!leaf && run_child < 0) {
                        n0 = 0;
#pragma unroll
                        for (int r = 0; r < RMAX; r++) {
                            const uint64_t cm = __ballot(cnt[r] > 0);
                            if (cnt[r] > 0) {
                                const int cl = n0 + __popcll(cm & ((1ull << lane) - 1ull));
                                my.child[cl] = r * kWave + lane;
                                my.n[cl] = k.n[r];
                                my.vl[cl] = cnt[r];
                                my.sx[cl] = sp[r].x;
                                my.sy[cl] = sp[r].y;
                                my.lane_of[r * kWave + lane] = (uint8_t)cl;
                            }
                            n0 += __popcll(cm);
                        }
                        wave_sync_memory();
                        visits = lane < n0 ? my.vl[lane] : 0;
                    }
                }
                if (a.stats && lane == 0 && m > 1 && !leaf) {
                    atomicAdd(a.stats + 0, 1);
                    atomicAdd(a.stats + 1, serial && run_child < 0 ? 0 : 1);
                    atomicAdd(a.stats + 2, serial && run_child < 0 ? 0 : m);
                    atomicAdd(a.stats + 3, serial && run_child < 0 ? m : 0);
                    // (without a real score, or with values that are not finite, no merge was tried)
                    if (serial && run_child < 0 && hk != 0u && !odd) atomicAdd(a.stats + 4, 1);
                    if (!serial) {
                        atomicAdd(a.stats + 7, 1);
                        atomicAdd(a.stats + 13, 1);
                    }
                }
                if (a.stats && lane == 0 && m == 1 && !leaf) atomicAdd(a.stats + 6, 1);
                if (run_child >= 0) {
                    int tn = 0, tx = 0, ty = 0;
#pragma unroll
                    for (int r = 0; r < RMAX; r++) {
                        if (r == (run_child >> 6)) {
                            tn = k.n[r];
                            tx = sp[r].x;
                            ty = sp[r].y;
                        }
                    }
                    run_np = __builtin_amdgcn_readlane(tn, run_child & 63);
                    run_sx = __builtin_amdgcn_readlane(tx, run_child & 63);
                    run_sy = __builtin_amdgcn_readlane(ty, run_child & 63);
                }
            }
            if (a.trace && lane == 0) {
                const int ti = atomicAdd(a.trace_n, 1);
                if (ti < a.trace_cap) {
                    a.trace[12 * ti + 0] = tr0;
                    a.trace[12 * ti + 1] = wall_clock64();
                    a.trace[12 * ti + 2] = (long long)m | ((long long)depth << 32) | ((m > 1 ? 0ll : 6ll) << 60);
                    a.trace[12 * ti + 3] = (long long)node;
                    for (int q = 0; q < 8; q++) a.trace[12 * ti + 4 + q] = 0;
                }
            }
            if (leaf) {
                if (lane < m) {
                    a.leaf[t] = node;
                    a.path_len[t] = depth + 1;
                    if (ROWS) {
                        s.len[v] = depth + 1;
                        s.leaf[v] = node;
                        s.kids[v] = cc;
                        s.visits[v] = np;
                    }
                }
                if (lane == 0) {
                    if (cc > 0 && depth >= a.max_depth) atomicAdd(a.truncated, m);
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
                    atomicSub(&s.open, m);
                }
                break;
            }
            if (run_child >= 0) {
                // ---- all of them go down together ----
                const int child = cb + run_child;
                if (lane < m) {
                    a.paths[(size_t)(depth + 1) * a.stride + t] = child;
                    if (ROWS) s.path[v][depth + 1] = child;
                }
                if (lane == 0 && a.vl > 0) atomicAdd(f.VL + child, (int)((uint32_t)a.vl * (uint32_t)m));
                node = child;
                np = run_np;
                cb = run_sx;
                cc = run_sy;
                depth++;
                continue;
            }
            // ---- the partition: the list in child order, each child's visitors in theirs ----
            const bool has = lane < n0 && visits > 0;
            const int inc = wave_inclusive_sum(has ? visits : 0, lane);
            const int start = inc - (has ? visits : 0);
            int child = 0, sx = 0, sy = 0, cn = 0;
            if (has) {
                child = my.child[lane];
                sx = my.sx[lane];
                sy = my.sy[lane];
                cn = my.n[lane];
                my.start[lane] = start;
                if (a.vl > 0) atomicAdd(f.VL + cb + child, (int)((uint32_t)a.vl * (uint32_t)visits));
            }
            const bool deep = depth + 1 >= a.max_depth;
            const bool on = has && sy > 0 && !deep;  // the visitors of this lane's child go on from it
            wave_sync_memory();
            bool ends = false, cut = false;
            if (lane < m) {
                const uint32_t o = my.order[lane];
                const int i = (int)(o >> 21), cl = my.lane_of[i];
                const int next = cb + i, kids = my.sy[cl];
                a.paths[(size_t)(depth + 1) * a.stride + t] = next;
                if (ROWS) s.path[v][depth + 1] = next;
                s.list[off + my.start[cl] + (int)(o & 0x1FFFFFu)] = v;
                ends = kids <= 0 || deep;
                cut = kids > 0 && deep;
                if (ends) {
                    a.leaf[t] = next;
                    a.path_len[t] = depth + 2;
                    if (ROWS) {
                        s.len[v] = depth + 2;
                        s.leaf[v] = next;
                        s.kids[v] = kids;
                        s.visits[v] = my.n[cl];
                    }
                }
            }
            wave_sync_memory();
            const uint64_t going = __ballot(on);
            const int n_end = __popcll(__ballot(ends)), n_cut = __popcll(__ballot(cut));
            int keep = -1;
            if (going) {
                const uint32_t most = wave_max_all(on ? ((uint32_t)visits << 6) | (63u - (uint32_t)lane) : 0u);
                keep = 63 - (int)((uint32_t)uniform((int)most) & 63u);
                const uint64_t others = going & ~(1ull << keep);
                if (others) {
                    int at = 0;
                    if (lane == 0) at = atomicAdd(&s.tail, __popcll(others));
                    at = uniform(at) + __popcll(others & ((1ull << lane) - 1ull));
                    if (on && lane != keep) {
                        s.item[at & (kBlockVisitors - 1)] = BlockItem{cb + child, cn, sx, sy, depth + 1, off + start, visits, 0};
                        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
                        __hip_atomic_store(&s.ready[at & (kBlockVisitors - 1)], at + 1, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_WORKGROUP);
                    }
                }
            }
            if (lane == 0 && n_end > 0) {
                if (n_cut > 0) atomicAdd(a.truncated, n_cut);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
                atomicSub(&s.open, n_end);
            }
            if (keep < 0) break;
            node = cb + __builtin_amdgcn_readlane(child, keep);
            np = __builtin_amdgcn_readlane(cn, keep);
            off += __builtin_amdgcn_readlane(start, keep);
            m = __builtin_amdgcn_readlane(visits, keep);
            cb = __builtin_amdgcn_readlane(sx, keep);
            cc = __builtin_amdgcn_readlane(sy, keep);
            depth++;
            if (lane < m) {
                v = s.list[off + lane];
                t = s.trav[v];
            }
        }
    }
    // (NULL unless somebody reads them: stamps of every launch, with the call in their upper half, cost it up to 3 %)
    auto left = [&]() {
        if (a.times && threadIdx.x == 0) atomicMax(a.times + 1, (int)(wall_clock64() & 0x7FFFFFFF));
    };
    if (!ROWS) {
        left();
        return;
    }
    // ---- the rows, straight into pinned host memory (see k_export) ----
    __syncthreads();
    n_here = (int)blockIdx.x < n_items ? a.items0[blockIdx.x].m
                                       : min(kBlockWaves, n_singles - ((int)blockIdx.x - n_items) * kBlockWaves);
    const ExportOut &o = out.rows;
    if ((int)threadIdx.x < n_here) {
        const int v = threadIdx.x, t = s.trav[v];
        host_store(o.len + t, s.len[v]);
        host_store(o.leaf + t, s.leaf[v]);
        host_store(o.children + t, s.kids[v]);
        host_store(o.visits + t, s.visits[v]);
    }
    for (int v = wv; v < n_here; v += kBlockWaves) {
        const int t = s.trav[v], len = s.len[v];
        const int id = lane < len ? s.path[v][lane] : -1;
        const int act = lane < len ? (f.action ? f.action[id] : id) : -1;
        if (lane <= a.max_depth) host_store(o.paths + (size_t)t * (a.max_depth + 1) + lane, id);
        if (lane >= 1 && lane <= a.max_depth) host_store(o.actions + (size_t)t * a.max_depth + lane - 1, act);
    }
    host_signal(out.sig.count, out.sig.flag, out.sig.seq, gridDim.x);
    left();
}

}  // namespace omk
