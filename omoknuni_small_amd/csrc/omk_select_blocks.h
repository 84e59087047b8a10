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
constexpr int kPlayQueue = 4;       // entries of a child worked out ahead
constexpr uint32_t kPlayEmpty = 0xFFFFFFFFu;  // above every real key: they have run out

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
    uint32_t order[kWave];   // per visitor: child << 21 | number of the visit
    uint8_t lane_of[RMAX * kWave];  // where child i is listed
};

template <int RMAX, bool ROWS>
struct BlockLds {
    int head, tail, open;  // tickets taken, items handed out, visitors that have not reached their leaf
    int ready[kBlockVisitors];  // item i lies in slot i % kBlockVisitors once this is i + 1 (an item has a visitor of its
                                // own, so that a slot is free again when its turn comes)
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

// m visitors of a node played over the n0 children listed in `s`, one per lane: order[q] for every visitor, and the
// visits of the lane's child.  It is the serial loop itself (the best of the current entries, first scan before second,
// lowest child first), but not one visitor at a time:
//   * every lane has its child's next kPlayQueue entries worked out, independently of each other;
//   * the next entries that come before every entry after the next are the next visitors', all at once, the best first:
//     each lane counts the ones before its own;
//   * a child whose entries run out becomes the leader, with 64 of its entries spread over the lanes: the visitors it
//     wins in a row are taken at once.
// Nothing is assumed about the order of a child's entries.  The children that are not listed have no entry above
// floor_key: false (with `order` overwritten) when an entry at or below it, or none, would be next.
template <int RMAX, bool RAVE>
__device__ __forceinline__ bool play_heads(BlockScratch<RMAX> &s, int n0, int m, float ep, uint32_t uvl,
                                           uint32_t floor_key, int lane, int &visits) {
    constexpr int K = kPlayQueue;
    int child = 0, cn = 0, cvl = 0, cnt = 0;
    float cw = 0.0f, cp = 0.0f, cq2 = 0.0f;
    if (lane < n0) {
        child = s.child[lane];
        cn = s.n[lane];
        cw = s.w[lane];
        cp = s.p[lane];
        cvl = s.vl[lane];
        if (RAVE) cq2 = s.q2[lane];
    }
    uint32_t q[K], second = 0u;  // bit j of `second`: entry j is a candidate of the second scan
    int lead = -1;               // lane of the leader, whose queue holds nothing
    auto refill = [&]() {
        second = 0u;
#pragma unroll
        for (int j = 0; j < K; j++) {
            uint32_t pos;
            entry_key<1, RAVE>(cn, cw, cp, cvl, cq2, ep, uvl, cnt + j, 0, q[j], pos);
            if (lane >= n0 || lane == lead) q[j] = 0u;
            second |= pos != 0u ? 1u << j : 0u;
        }
    };
    int l_child = 0, l_n = 0, l_vl = 0, l_base = 0, l_pos = 0;  // the leader; entry l_base + l_pos is its next
    float l_w = 0.0f, l_p = 0.0f, l_q2 = 0.0f;
    uint32_t l_key = 0u;                // entry l_base + lane
    uint64_t l_second = 0u, l_ok = 0u;  // which of them are of the second scan, and above floor_key
    auto lead_entries = [&]() {
        uint32_t pos;
        entry_key<1, RAVE>(l_n, l_w, l_p, l_vl, l_q2, ep, uvl, l_base + lane, 0, l_key, pos);
        l_second = __ballot(pos != 0u);
        l_ok = __ballot(l_key > floor_key);
        l_pos = 0;
    };
    refill();
    const uint32_t id = (uint32_t)lane;
    for (int done = 0; done < m;) {
        const uint32_t after = (uint32_t)uniform((int)wave_max_all(q[1]));
        if (after == kPlayEmpty) {  // somebody's entries run out
            const int x = __ffsll((long long)__ballot(q[1] == kPlayEmpty)) - 1;
            if (lane == lead) cnt = l_base + l_pos;
            lead = x;
            l_child = __builtin_amdgcn_readlane(child, x);
            l_n = __builtin_amdgcn_readlane(cn, x);
            l_vl = __builtin_amdgcn_readlane(cvl, x);
            l_w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cw), x));
            l_p = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cp), x));
            if (RAVE) l_q2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cq2), x));
            l_base = __builtin_amdgcn_readlane(cnt, x);
            refill();
            lead_entries();
            continue;
        }
        // the next entries above all entries after the next, above the leader's and above floor_key
        uint32_t bar = after > floor_key ? after : floor_key;
        if (lead >= 0) {
            const uint32_t l_next = (uint32_t)__builtin_amdgcn_readlane((int)l_key, l_pos);
            bar = bar > l_next ? bar : l_next;
        }
        const uint64_t set = __ballot(q[0] > bar);
        if (set) {
            const uint64_t mine = ((uint64_t)q[0] << 32) | ((second & 1u) ? 63u - id : 127u - id);  // larger: earlier
            int rank = 0;
            for (uint64_t rest = set; rest; rest &= rest - 1ull) {
                const int x = __ffsll((long long)rest) - 1;
                const uint64_t other = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(mine >> 32), x) << 32) |
                                       (uint32_t)__builtin_amdgcn_readlane((int)mine, x);
                rank += other > mine ? 1 : 0;
            }
            if (q[0] > bar && rank < m - done) {
                s.order[done + rank] = ((uint32_t)child << 21) | (uint32_t)cnt;
#pragma unroll
                for (int j = 0; j + 1 < K; j++) q[j] = q[j + 1];
                q[K - 1] = kPlayEmpty;
                second >>= 1;
                cnt++;
            }
            done += __popcll(set);
            continue;
        }
        // one at a time: the best of the next entries, or the leader's as long as they come before it
        const uint32_t best = wave_max_all(q[0]);
        const uint64_t tied = __ballot(q[0] == best), first = __ballot(q[0] == best && !(second & 1u));
        const int x = __ffsll((long long)(first ? first : tied)) - 1;
        const uint32_t key = (uint32_t)uniform((int)best);
        if (lead >= 0) {
            uint64_t wins = __ballot(l_key > key);
            const uint64_t same = __ballot(l_key == key);
            if (same) {
                const uint64_t lower = lead < x ? ~0ull : 0ull;
                wins |= same & (first ? ~l_second & lower : ~l_second | lower);
            }
            const uint64_t lost = ~(wins & l_ok) & (~0ull << l_pos);
            int run = (lost ? __ffsll((long long)lost) - 1 : kWave) - l_pos;
            run = run < m - done ? run : m - done;
            if (run > 0) {
                if (lane >= l_pos && lane < l_pos + run)
                    s.order[done + lane - l_pos] = ((uint32_t)l_child << 21) | (uint32_t)(l_base + lane);
                done += run;
                l_pos += run;
                if (l_pos == kWave && done < m) {
                    l_base += kWave;
                    lead_entries();
                }
                continue;
            }
        }
        if (key <= floor_key) return false;
        if (lane == x) {
            s.order[done] = ((uint32_t)child << 21) | (uint32_t)cnt;
#pragma unroll
            for (int j = 0; j + 1 < K; j++) q[j] = q[j + 1];
            q[K - 1] = kPlayEmpty;
            second >>= 1;
            cnt++;
        }
        done++;
    }
    visits = lane == lead ? l_base + l_pos : cnt;
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
        a.times[0] = (int)(wall_clock64() & 0x7FFFFFFF);
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
        int ticket = 0;
        if (lane == 0) ticket = atomicAdd(&s.head, 1);
        ticket = uniform(ticket);
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
                uint32_t lk = 0u;  // the best child's entry for the last visitor, where others come before it
                if (hk != 0u && (m == 1 || a.vl <= 0)) {
                    run_child = best;
                } else if (hk != 0u && !odd) {
                    // ---- does the best child win every time?  (single_run) ----
                    uint32_t ok = 0u, opos = 0xFFFFFFFFu;
#pragma unroll
                    for (int r = 0; r < RMAX; r++)
                        if (r * kWave + lane != best && k.k1[r] > ok) { ok = k.k1[r]; opos = (uint32_t)(r * kWave + lane); }
#pragma unroll
                    for (int r = 0; r < RMAX; r++)
                        if (r * kWave + lane != best && k.k2[r] > ok) { ok = k.k2[r]; opos = (uint32_t)(F + r * kWave + lane); }
                    uint32_t sk, spos, lp;
                    wave_best_fast(ok, opos, sk, spos);
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
                    entry_key<RMAX, RAVE>(bn, bw, bp, bvl, bq2, ep, uvl, m - 1, best, lk, lp);
                    lk = (uint32_t)uniform((int)lk);
                    lp = (uint32_t)uniform((int)lp);
                    if (lk != 0u && (sk == 0u || comes_before(lk, lp, sk, spos))) {
                        if (entries_in_order<RMAX, RAVE>(bn, bw, bp, bvl, bq2, ep, uvl, best, m, lane)) run_child = best;
                        lk = 0u;
                    }
                    if (run_child < 0) {
                        // ---- the children that can be chosen, one per lane ----
                        // those whose next entry is not below lk (with the best child's entries in order nobody else
                        // is; play_heads sees to it), or, if there are too many or no lk, the m best
                        uint32_t from = lk < hk ? lk : hk, floor_key = from - 1u;
                        auto heads = [&](uint32_t T) {
                            int c = 0;
#pragma unroll
                            for (int r = 0; r < RMAX; r++) c += __popcll(__ballot(umax32(k.k1[r], k.k2[r]) >= T));
                            return c;
                        };
                        if (RMAX == 1) {
                            from = 1u;
                            floor_key = 0u;
                        } else if (from == 0u || heads(from) > kWave) {
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
                            serial = !play_heads<RMAX, RAVE>(my, n0, m, ep, uvl, floor_key, lane, visits);
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
                if (a.stats && lane == 0 && m > 1) {
                    atomicAdd(a.stats + 0, 1);
                    atomicAdd(a.stats + 1, serial && run_child < 0 ? 0 : 1);
                    atomicAdd(a.stats + 2, serial && run_child < 0 ? 0 : m);
                    atomicAdd(a.stats + 3, serial && run_child < 0 ? m : 0);
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
    if (threadIdx.x == 0) a.times[1] = a.times[2] = (int)(wall_clock64() & 0x7FFFFFFF);
    if (!ROWS) return;
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
}

}  // namespace omk
