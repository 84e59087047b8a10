// Selection for batches whose roots have few visitors each (at most kBlockVisitors): a block a root.
//
// What it computes is what omk_select_kernels.h computes (see there), for crowds that fit a wavefront: a node's
// visitors are one per lane, a subtree's lists and work items live in LDS, and a wavefront that has settled a node goes
// on with the child most of them chose and leaves the others to the idle wavefronts of its block.  Nothing is shared
// between blocks: no queue in memory, no reset before the launch, no wait that could have to give up.  Handing a node
// on costs an LDS round trip where the queue in memory takes 3 us (release, poll, acquire, the item's own trip).
//
// What bounds it is the latency of a chain of crowded nodes: one dependent trip to memory a level (0.3 us), and the
// instruction issue of the wavefront that settles the node, 5 cycles an instruction and 8 to 10 where each needs the one
// before.  So most children are ruled out by bounds of their scores (score_about: two reciprocals where the score takes two
// IEEE divisions), which settles a node whose visitors stay together, and a lone visitor's, without a division: a level of
// four rounds 2.5 -> 1.8 us in the timeline.  Where the bounds leave several children the exact scores of these few decide.
// A selection and its reverting, us, with scores first and with bounds first, the median of five seeds: of trees fresh from an
// upload 8 visitors of a Gomoku tree 25 -> 19, 64 49 -> 32, 48 of a Go tree with RAVE 36 -> 22, 64 of a chess-like one 39 -> 31,
// 64 in each of 16 47 -> 35; of trees that 2000 batches have been backed up into, where most nodes are contested, 26 -> 22,
// 37 -> 34, 53 -> 44, 34 -> 35, 32 -> 33: nodes of one round have two divisions to lose and contested ones keep them.  (Lone
// visitors of 200 such chess-like trees 15 -> 16; 8 in one 26 -> 26, 16 in each of 64 31 -> 32.)
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
struct BlockScratch {
    int child[kWave];  // index in the node
    int n[kWave], vl[kWave], sx[kWave], sy[kWave];
    float w[kWave], p[kWave], q2[kWave];
    int start[kWave];        // first place of the child's visitors in the node's list
    int taken[kWave];        // its visits
    uint64_t entry[2 * kWave + 8];         // merge_heads: the entries being put in order
    alignas(16) uint32_t slot[2 * kWave];  // merge_rest: the same
    uint32_t order[kWave];   // per visitor: listed child << 16 | number of the visit
};

// The ceiling of a lane without a child: the least finite number, so that the sum that looks for others passes over it.  Children
// are listed from kLeastScore on at the lowest, which no lane without a child reaches; what lies below is left to the serial loop.
constexpr float kNoChild = -3.402823466e38f, kLeastScore = -3.0e38f;

template <bool ROWS>
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
    BlockScratch scratch[kBlockWaves];
};

// A contested node: m visitors over the n0 children listed in `s`, one per lane.  order[q] receives the listed child and the
// number of its visit for every visitor, `visits` the visits of the lane's child.  The score a child shows its j-th visitor of
// this node depends on nothing but j, and where no child's scores increase with j the serial order is the merge of the
// children's lists.  A prefix of every list is worked out at once, 128 entries in all, independently of each other where the
// serial loop waits for two divisions a visitor.  An entry that is not worked out comes after the last one of its child that
// is, or is a child's very next one: the entries up to the first of these are the next visitors', the best first, and every
// one finds its place by counting the ones before it.  What is left goes on from there.
// floor_key: the children that are not listed have no entry above it.
// False (with `order` overwritten) when a child's entries are not in order, or when an entry at or below floor_key or none
// would be next: the caller plays one visitor after the other.
//
// At first as many entries of every child (merge_heads).  One child that most visitors go to gets two or four of many
// children's 128 that way, and a pass settles little more than these: then as many of every child as the closed form says
// lie at or above a threshold with enough of them, and one more (merge_rest; team_merge).  40 visitors of a Gomoku node, 25
// passes before: 23 -> 6.5 us; 16 of a Go node, 8 passes: 12 -> 6.

template <bool RAVE>
__device__ __forceinline__ bool merge_rest(BlockScratch &s, int n0, int m, float ep, uint32_t uvl,
                                           uint32_t floor_key, int lane, int done, int &visits) {
    constexpr int kSlots = 2 * kWave;
    constexpr int kScaled = 16;  // children up to which a threshold is not looked for where 128 entries are not enough
    const bool mine = lane < n0;
    uint32_t *const slot = s.slot;
    int took = visits;  // of the lane's child so far
    while (done < m) {
        const int need = m - done;
        // As many of every child, all that are asked for if there is room (`all`); where that is not a quarter of them, as
        // many as a threshold says.
        const int log_need = need <= 1 ? 0 : 32 - __clz(need - 1), log_room = n0 <= 1 ? 7 : 7 - (32 - __clz(n0 - 1));
        const int log_e = log_need < log_room ? log_need : log_room;
        const bool all = log_need <= log_room;
        int total = n0 << log_e, c = 1 << log_e, start = lane << log_e;  // slots in all; the lane's child's
        c = c < need ? c : need;
        uint32_t bk = 0u, bl = ~0u;  // the first entry behind which one may be missing
        int from[2] = {lane >> log_e << log_e, (kWave + lane) >> log_e << log_e};  // of the lane's slots
        int child[2] = {lane >> log_e, (kWave + lane) >> log_e};
        uint64_t starts0 = 0ull, starts1 = 0ull;
        const uint64_t upto = ~0ull >> (63 - lane);
        auto last_of = [&](uint64_t m0, uint64_t m1, int h) {  // the last marked slot up to the lane's own in half h
            if (h == 0) return 63 - __clzll((long long)(m0 & upto));
            return m1 & upto ? 2 * kWave - 1 - __clzll((long long)(m1 & upto)) : 63 - __clzll((long long)m0);
        };
        if (!all) {
            // ---- how many of every child ----
            slot[lane] = ~0u;
            slot[kWave + lane] = ~0u;
            int cn = 0, cvl = 0;
            float cw = 0.0f, cp = 0.0f, cq2 = 0.0f;
            if (mine) {
                cn = s.n[lane];
                cw = s.w[lane];
                cp = s.p[lane];
                cvl = (int)((uint32_t)s.vl[lane] + (uint32_t)took * uvl);
                if (RAVE) cq2 = s.q2[lane];
            }
            // (its next entry is not above `head`)
            float head = score_ceiling<RAVE>(cn, cw, cp, cvl, cq2, ep) + kBoundTiny;
            if (!mine) head = -__builtin_inff();
            auto entries_from = [&](uint32_t key) {
                const float tau = key_score(key);
                const int n = predict_count<RAVE>(cn, cw, cp, cvl, cq2, ep, uvl, tau, need,
                                                  RAVE ? 0.5f * (tau - key_score(key - 1u)) : 0.0f);
                return !(head >= tau) ? 0 : n > 1 ? n : 1;
            };
            auto with_next = [&](int n) { return n > 0 && n < need ? n + 1 : n; };
            uint32_t T = floor_key + 1u;
            {  // the last one a child could be asked for: it alone has `need` entries at or above that
                float tail = score_floor<RAVE>(cn, cw, cp, (int)((uint32_t)cvl + (uint32_t)(need - 1) * uvl), cq2, ep);
                if (!mine) tail = -__builtin_inff();
                const uint32_t best = (uint32_t)uniform((int)wave_max_all(ordered_bits(tail)));
                T = best > T ? best : T;
            }
            int n = entries_from(T);
            c = with_next(n);
            int inc = wave_inclusive_sum(c, lane);
            total = __builtin_amdgcn_readlane(inc, 63);
            if (total == 0) return false;
            if (total > kSlots && n0 > kScaled) {
                // false position in y = 1 / (score + 1), in which the counts are nearly a straight line (search_threshold)
                auto y_of = [](uint32_t key) {
                    const float d = key_score(key) + 1.0f;
                    return __builtin_amdgcn_rcpf(d > 1e-6f ? d : 1e-6f);
                };
                const uint32_t hi_key = (uint32_t)uniform((int)wave_max_all(ordered_bits(head)));
                uint32_t klo = T, khi = hi_key + 1u;
                const float aim = (float)(need + (need >> 2) + 1);
                float ylo = y_of(klo), yhi = y_of(hi_key), flo = fmaxf((float)wave_sum_i32(n) - aim, 1.0f), fhi = 1.0f - aim;
                T = hi_key;
                int last = 0;
                for (int it = 0; it < 8 && khi - klo > 1u; it++) {
                    const float ym = (ylo * fhi - yhi * flo) * __builtin_amdgcn_rcpf(fhi - flo);
                    uint32_t mid = score_key(__builtin_amdgcn_rcpf(ym) - 1.0f);
                    if (!(mid > klo)) mid = klo + 1u;
                    if (!(mid < khi)) mid = khi - 1u;
                    mid = (uint32_t)uniform((int)mid);
                    const int e = entries_from(mid);
                    const int both = wave_sum_i32(e | (with_next(e) << 16));
                    const int sum = both & 0xFFFF, slots = both >> 16;
                    if (slots > kSlots) {
                        klo = mid;
                        ylo = y_of(mid);
                        flo = fmaxf((float)sum - aim, 1.0f);
                        if (last > 0) fhi *= 0.5f;
                        last = 1;
                        continue;
                    }
                    T = mid;
                    if (sum >= need) break;
                    khi = mid;
                    yhi = y_of(mid);
                    fhi = (float)sum - aim;
                    if (last < 0) flo *= 0.5f;
                    last = -1;
                }
                n = entries_from(T);
                c = with_next(n);
                inc = wave_inclusive_sum(c, lane);
                total = __builtin_amdgcn_readlane(inc, 63);
            }
            if (total > kSlots) {  // (few children, or many entries on one key)  In proportion, and one at least
                const float f = (float)(kSlots - kScaled) * __builtin_amdgcn_rcpf((float)total);
                if (c > 1) c = 1 + (int)((float)(c - 1) * (n0 > kScaled ? 0.5f : 1.0f) * f);
                inc = wave_inclusive_sum(c, lane);
                total = __builtin_amdgcn_readlane(inc, 63);
            }
            if (c == 0 && mine) {
                bk = ordered_bits(head);
                bl = 0u;
            }
            // ---- which child a slot's entry belongs to: the last one that starts at or before it ----
            start = inc - c;
            wave_sync_memory();
            if (c > 0) slot[start] = (uint32_t)lane;
            wave_sync_memory();
            const int w0 = (int)slot[lane], w1 = (int)slot[kWave + lane];
            starts0 = __ballot(w0 >= 0);
            starts1 = __ballot(w1 >= 0);
            from[0] = last_of(starts0, starts1, 0);
            child[0] = __shfl(w0, from[0], kWave);
            if (total > kWave) {
                from[1] = last_of(starts0, starts1, 1);
                const int x1 = __shfl(w1, from[1] & 63, kWave), x0 = __shfl(w0, from[1] & 63, kWave);
                child[1] = from[1] >= kWave ? x1 : x0;
            }
        }
        const bool wide = total > kWave;  // uniform
        // ---- work them out ----
        uint32_t key[2] = {0u, 0u}, low[2] = {~0u, ~0u};
        bool valid[2] = {lane < total, kWave + lane < total};
        if (all) {
#pragma unroll
            for (int h = 0; h < 2; h++) valid[h] = valid[h] && child[h] < n0 && h * kWave + lane - from[h] < need;
        }
        wave_sync_memory();
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (h == 1 && !wide) break;
            const int w = child[h] & (kWave - 1), j = s.taken[w] + h * kWave + lane - from[h];
            uint32_t kk, pp;
            entry_key<1, RAVE>(s.n[w], s.w[w], s.p[w], s.vl[w], RAVE ? s.q2[w] : 0.0f, ep, uvl, j, 0, kk, pp);
            if (valid[h]) {
                key[h] = kk;
                low[h] = (pp << 24) | (uint32_t)(w << 16) | (uint32_t)j;
            }
        }
        // ---- in order?  And up to the first behind which one may be missing ----
        // (equal keys: first scan before second, then the children's order, then the visits')
        bool bad = false;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (h == 1 && !wide) break;
            const int e = h * kWave + lane;
            uint32_t pk = (uint32_t)__shfl_up((int)key[h], 1, kWave), pl = (uint32_t)__shfl_up((int)low[h], 1, kWave);
            if (h == 1 && lane == 0) {
                pk = (uint32_t)__builtin_amdgcn_readlane((int)key[0], 63);
                pl = (uint32_t)__builtin_amdgcn_readlane((int)low[0], 63);
            }
            const bool first = e == from[h];
            bad |= valid[h] && !first && comes_before(key[h], low[h], pk, pl);
            if (!all) {
                const uint64_t next = h == 0 ? (starts0 >> 1) | (starts1 << 63) : starts1 >> 1;
                const bool end = e + 1 == total || ((next >> lane) & 1ull);  // of its child's
                if (valid[h] && end && e + 1 - from[h] < need && comes_before(key[h], low[h], bk, bl)) {
                    bk = key[h];
                    bl = low[h];
                }
            }
        }
        if (__ballot(bad)) return false;
        uint32_t bar = 0u;
        if (!all) bar = (uint32_t)uniform((int)wave_max_all(bk));
        const uint32_t above = bar > floor_key ? bar : floor_key;
        uint64_t in0 = __ballot(key[0] > above), in1 = __ballot(key[1] > above);
        int n_in = __popcll(in0) + __popcll(in1);
        if (n_in < need && bar > floor_key) {  // (those on the bar's own key)
            const uint32_t bar_low = wave_min_u32(bk == bar ? bl : ~0u);
            in0 |= __ballot(key[0] == bar && low[0] <= bar_low);
            in1 |= __ballot(key[1] == bar && low[1] <= bar_low);
            n_in = __popcll(in0) + __popcll(in1);
        }
        if (n_in == 0) return false;
        // ---- far more than are needed: those from a key on that few lie above ----
        if (n_in > need + 32) {
            float lo = key_score(above + 1u), hi = key_score((uint32_t)uniform((int)wave_max_all(key[0] > key[1] ? key[0] : key[1])));
            uint32_t cut = 0u;
            for (int it = 0; it < 12; it++) {
                const float mid = 0.5f * (lo + hi);
                if (!(mid > lo && mid < hi)) break;
                const uint32_t k = (uint32_t)uniform((int)score_key(mid));
                const int n = __popcll(in0 & __ballot(key[0] >= k)) + __popcll(in1 & __ballot(key[1] >= k));
                if (n < need) {
                    hi = mid;
                } else {
                    lo = mid;
                    cut = k;
                    if (n <= need + 8) break;
                }
            }
            in0 &= __ballot(key[0] >= cut);
            in1 &= __ballot(key[1] >= cut);
        }
        // ---- every one's place: behind the better ones, on equal keys behind the first scan's and the slots before ----
        const bool in[2] = {((in0 >> lane) & 1ull) != 0ull, ((in1 >> lane) & 1ull) != 0ull};
        const bool second[2] = {(low[0] >> 30) != 0u, (low[1] >> 30) != 0u};
        const uint64_t f0 = __ballot(in[0] && !second[0]), f1 = __ballot(in[1] && !second[1]);
        const int n_first = __popcll(f0) + __popcll(f1), n_list = __popcll(in0) + __popcll(in1);
        int at[2];  // in a list of the first scan's and then the second's, each in the order of their slots
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint64_t b0 = second[h] ? in0 & ~f0 : f0, b1 = second[h] ? in1 & ~f1 : f1;
            at[h] = (second[h] ? n_first : 0) + __popcll(b0 & (h == 0 ? upto >> 1 : ~0ull)) + (h == 0 ? 0 : __popcll(b1 & (upto >> 1)));
        }
        wave_sync_memory();
        slot[lane] = 0u;
        slot[kWave + lane] = 0u;
        wave_sync_memory();
#pragma unroll
        for (int h = 0; h < 2; h++)
            if (in[h]) slot[at[h]] = key[h];
        wave_sync_memory();
        int rank[2] = {0, 0};
        const uint4 *const four = reinterpret_cast<const uint4 *>(slot);
        for (int e0 = 0; e0 < n_list; e0 += 16) {
            uint4 o[4];
#pragma unroll
            for (int u = 0; u < 4; u++) o[u] = four[(e0 >> 2) + u];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                if (h == 1 && in1 == 0ull) break;  // uniform
                int r0 = 0, r1 = 0;  // (sums that do not wait for one another)
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const uint32_t k = key[h] - ((e0 >> 2) + u < (at[h] >> 2) ? 1u : 0u);  // (in front of it equal ones count too)
                    r0 += o[u].x > k ? 1 : 0;
                    r1 += o[u].y > k ? 1 : 0;
                    r0 += o[u].z > k ? 1 : 0;
                    r1 += o[u].w > k ? 1 : 0;
                }
                rank[h] += r0 + r1;
            }
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {  // (and of its own four)
            const uint4 o = four[(in[h] ? at[h] : 0) >> 2];
            const int q = at[h] & 3;
            rank[h] += (q > 0 && o.x == key[h] ? 1 : 0) + (q > 1 && o.y == key[h] ? 1 : 0) + (q > 2 && o.z == key[h] ? 1 : 0);
        }
        bool takes[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            takes[h] = in[h] && rank[h] < need;
            if (takes[h]) s.order[done + rank[h]] = low[h] & 0x3FFFFFu;
        }
        wave_sync_memory();
        // ---- what every child took: so many of its slots ----
        const uint64_t t0 = __ballot(takes[0]), t1 = __ballot(takes[1]);
        if (!wide) {
            took += mine && c > 0 ? __popcll((t0 >> start) & (~0ull >> (kWave - c))) : 0;
        } else {
            auto below = [](uint64_t b0, uint64_t b1, int e) {  // marked slots before slot e
                const int e0 = e < kWave ? e : kWave, e1 = e - e0;
                return (e0 ? __popcll(b0 << (kWave - e0)) : 0) + (e1 ? __popcll(b1 << (kWave - e1)) : 0);
            };
            took += below(t0, t1, start + c) - below(t0, t1, start);
        }
        done += n_in < need ? n_in : need;
        if (done < m) {
            s.taken[lane] = took;
            wave_sync_memory();
        }
    }
    visits = took;
    return true;
}

template <bool RAVE>
__device__ __forceinline__ bool merge_heads(BlockScratch &s, int n0, int m, float ep, uint32_t uvl,
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
                s.order[done + rank] = (uint32_t)(e & 0x3FFFFFu);
                atomicAdd(&s.taken[w], 1);
            }
        }
        wave_sync_memory();
        base = s.taken[c];
        done += total < need ? total : need;
        // As many of every child is not what it takes.  (That it seldom comes to that is said because the compiler gives registers
        // to the deepest loops otherwise, which are merge_rest's: 64 visitors of a worn Gomoku tree 28, 39, 37, 41, 29 us, and
        // 27, 36, 36, 40, 28 with this.  With RAVE it is not seldom: 48 visitors of a fresh Go tree took 4 % longer with this.)
        const bool poor = done < m && 4 * total < need;
        if (RAVE ? poor : __builtin_expect_with_probability(poor, 0, 0.999)) {
            visits = s.taken[lane];
            return merge_rest<RAVE>(s, n0, m, ep, uvl, floor_key, lane, done, visits);
        }
    }
    visits = s.taken[lane];
    return true;
}

// A node settled by the serial loop itself, over at most one child a lane, on the next two entries of every child, worked
// out side by side: a visitor is then a search for the best of the lanes' and no more.  order[q] and the visits of the
// lane's child as above; `who`: the lane of the last visitor's child.  mine: the lane has a child, number `child` of the
// node.  The children that are not in a lane have no entry above floor_key: false when one at or below it would be next, or
// where a child's entries are not in order (as above, though nothing here depends on it).
constexpr int kPickFew = 3;  // visitors up to which that is done
template <bool RAVE>
__device__ __forceinline__ bool pick_few(uint32_t *order, bool mine, int child, int cn, float cw, float cp, int cvl, float cq2,
                                         int m, float ep, uint32_t uvl, uint32_t floor_key, int lane, int &visits, int &who) {
    visits = 0;
    for (int done = 0; done < m;) {
        uint32_t key[2], pos[2];
#pragma unroll
        for (int g = 0; g < 2; g++) {
            entry_key<1, RAVE>(cn, cw, cp, cvl, cq2, ep, uvl, visits + g, 0, key[g], pos[g]);
            key[g] = mine ? key[g] : 0u;
        }
        if (__ballot(mine && comes_before(key[1], pos[1], key[0], pos[0]))) return false;
        int used = 0;
        for (bool left = true; left && done < m; done++) {
            const uint32_t top = (uint32_t)uniform((int)wave_max_all(key[0]));
            if (top <= floor_key) return false;
            uint64_t ties = __ballot(key[0] == top);
            if (ties & (ties - 1ull)) {  // first scan before second, then the children's order
                const uint32_t place = pos[0] * 1024u + (uint32_t)child;
                const uint32_t least = wave_min_u32(key[0] == top ? place : ~0u);
                ties = __ballot(key[0] == top && place == least);
            }
            who = __ffsll((long long)ties) - 1;
            if (lane == who) {
                order[done] = (uint32_t)(lane << 16) | (uint32_t)visits;
                visits++;
                used++;
                key[0] = key[1];
                pos[0] = pos[1];
            }
            left = __builtin_amdgcn_readlane(used, who) < 2;
        }
    }
    wave_sync_memory();
    return true;
}

// Blocks [0, n_items): a root with several visitors each.  The blocks behind them: up to kBlockWaves roots with one
// visitor each.  One thread leaves the scheduler words as a reset would have.  ROWS: the block sends its visitors' rows
// to the host when the last of them has reached its leaf.
template <int RMAX, bool RAVE, bool ROWS>
__global__ __launch_bounds__(kBlockWaves *kWave) void k_select_blocks(ForestDev f, SelectArgs a, int n_items, int n_singles,
                                                                      LoneOut out) {
    __shared__ BlockLds<ROWS> s;
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
    BlockScratch &my = s.scratch[wv];
    const uint32_t uvl = a.vl > 0 ? (uint32_t)a.vl : 0u;
    float c_puct = a.c_puct;
    asm volatile("" : "+v"(c_puct));  // (as above)
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
        bool owed = false;
        for (;;) {
            const long long tr0 = a.trace ? wall_clock64() : 0ll;
            bool leaf = cc <= 0 || depth >= a.max_depth;
            int run_child = -1, run_np = 0, run_sx = 0, run_sy = 0;
            int n0 = 0, visits = 0;  // of the lane's listed child
            bool serial = false;
            Kids<RMAX, RAVE> k;
            int2 sp[RMAX];
            bool replayed = false;
            // what the level before left to be stored when all of its visitors went on together: once this level's loads
            // are on their way
            auto arrive = [&]() {
                if (!owed) return;
                if (lane < m) {
                    a.paths[(size_t)depth * a.stride + t] = node;
                    if (ROWS) s.path[v][depth] = node;
                }
                if (lane == 0 && a.vl > 0) atomicAdd(f.VL + node, (int)((uint32_t)a.vl * (uint32_t)m));
                owed = false;
            };
            if (leaf) arrive();
            if (!leaf) {
                int nelig = cc;
                if (__builtin_expect_with_probability(a.pw, 0, 0.99)) {
                    const int kk = ceil_sqrt_i32(np);
                    nelig = kk < cc ? kk : cc;
                }
                // one trip to memory: statistics, legality bits and child ranges together.  A lane without a child asks for
                // the last one's, and so does a round without any: a branch around its loads costs more than them, in
                // registers set to nothing and in waits for loads that only the other way would have made.
                uint32_t word[RMAX];
                auto ask = [&]() {
                    const int32_t *const bN = f.N + cb, *const bVL = f.VL + cb;
                    const float *const bW = f.W + cb, *const bP = f.P + cb, *const bq = RAVE ? f.q2 + cb : nullptr;
                    const int2 *const bs = f.span + cb;
                    const __attribute__((address_space(1))) uint32_t *legal = (const __attribute__((address_space(1))) uint32_t *)f.legal;
                    asm volatile("" : "+s"(legal));  // (in registers: not a trip to the arguments per round)
                    uint32_t at[RMAX];
#pragma unroll
                    for (int r = 0; r < RMAX; r++) {
                        const int i = r * kWave + lane;
                        at[r] = (uint32_t)(i < nelig ? i : nelig - 1) & 0xFFFFu;
                        word[r] = 0xFFFFFFFFu;
                    }
                    if (legal) {
#pragma unroll
                        for (int r = 0; r < RMAX; r++) word[r] = legal[((uint32_t)cb + at[r]) >> 5];
                    }
#pragma unroll
                    for (int r = 0; r < RMAX; r++) {
                        k.n[r] = bN[at[r]];
                        k.vl[r] = bVL[at[r]];
                        k.w[r] = bW[at[r]];
                        k.p[r] = bP[at[r]];
                        if (RAVE) k.q2[r] = bq[at[r]];
                        sp[r] = bs[at[r]];
                    }
                };
                ask();
                arrive();
                float ep_ahead = c_puct * sqrtf((float)np);
                asm volatile("" : "+v"(ep_ahead));  // (while the loads are on their way)
                // All of them have arrived, the child ranges too (vmcnt(0)), and the compiler knows it.  Else it may wait
                // where the loop comes round, and with it for the stores and atomics of the level before its next loads:
                // 8 visitors of a Gomoku tree 35 or 38 us, by how registers fall.
                __builtin_amdgcn_s_waitcnt(0x0F70);
                const float ep = __int_as_float(uniform(__float_as_int(ep_ahead)));
                // ---- no child's score is above ceil[] (score_ceiling): the lane's two highest ----
                float ceil[RMAX], c1 = kNoChild, c2 = kNoChild, odd = 0.0f;
                int r1 = 0, tn = 0, tvl = 0, tx = 0, ty = 0;  // the highest: its round and statistics
                float tw = 0.0f, tp = 0.0f, tq2 = 0.0f;
                auto bound = [&](int r, bool in) {
                    float c = score_ceiling<RAVE>(k.n[r], k.w[r], k.p[r], k.vl[r], k.q2[r], ep);
                    // (an unvisited child's score does not look at its sum, its later ones do: when those of the first scan run
                    // out, the blends of the second must not decide)
                    if (RAVE) c = fmaf(k.w[r], 0.0f, c);
                    odd = fmaf(c, 0.0f, odd);  // not a number from the first value on that is not finite
                    in = in && ((word[r] >> ((uint32_t)(cb + r * kWave + lane) & 31u)) & 1u);
                    ceil[r] = in ? c : kNoChild;
                    c2 = __builtin_amdgcn_fmed3f(c1, c2, ceil[r]);
                    const bool up = ceil[r] > c1;
                    r1 = up ? r : r1;
                    tn = up ? k.n[r] : tn;
                    tvl = up ? k.vl[r] : tvl;
                    tw = up ? k.w[r] : tw;
                    tp = up ? k.p[r] : tp;
                    if (RAVE) tq2 = up ? k.q2[r] : tq2;
                    tx = up ? sp[r].x : tx;
                    ty = up ? sp[r].y : ty;
                    c1 = up ? ceil[r] : c1;
                };
                if (RMAX > 1 && nelig > (RMAX - 1) * kWave) {
#pragma unroll
                    for (int r = 0; r < RMAX; r++) bound(r, r < RMAX - 1 || r * kWave + lane < nelig);
                } else {
#pragma unroll
                    for (int r = 0; r < RMAX; r++) {
                        ceil[r] = kNoChild;
                        if (r * kWave < nelig) bound(r, r * kWave + lane < nelig);  // uniform
                    }
                }
                // its entry for the last visitor: of the lane's highest, for whichever lane has the node's (while that is being
                // found; what not every node asks for is worked out where it is, which lone visitors and splits gain 1 to 4 % by)
                const bool together = m == 1 || a.vl <= 0;  // nothing changes between the visitors
                const int j_last = together ? 0 : m - 1;
                const float lane_last = score_floor<RAVE>(tn, tw, tp, (int)((uint32_t)tvl + (uint32_t)j_last * uvl), tq2, ep);
                const uint32_t lane_top = ordered_bits(c1), top = (uint32_t)uniform((int)wave_max_all(lane_top));
                const uint64_t tops = __ballot(lane_top == top);
                serial = true;
                bool real = __ballot(!(odd == 0.0f)) == 0ull;
                if (__builtin_expect_with_probability(!real, 0, 0.999)) {
                    // (not of what stands in an empty slot.  In the loop above that would put up to 61 registers into memory;
                    // between it and the reductions just made it would keep them apart: 64 visitors of a Go tree 37 -> 39 us)
                    odd = 0.0f;
#pragma unroll
                    for (int r = 0; r < RMAX; r++) odd = fmaf(ceil[r], 0.0f, odd);
                    real = __ballot(!(odd == 0.0f)) == 0ull;
                }
                if (__builtin_expect_with_probability(real && top > ordered_bits(kLeastScore), 1, 0.999)) {
                    // ---- does that child win every time?  Its last entry comes before every other child's next one ----
                    const int bl = __ffsll((long long)tops) - 1;
                    const float last = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(lane_last), bl));
                    bool wins = __ballot(c1 >= last) == 1ull << bl && __ballot(c2 >= last) == 0ull;
                    const auto in_order = [&]() { return __ballot(in_order_at_once(tn, tw, tp, tvl, ep, uvl, j_last)); };
                    if (__builtin_expect_with_probability(wins && !together && !((in_order() >> bl) & 1ull), 0, 0.99))
                        wins = entries_in_order<RMAX, RAVE>(
                            __builtin_amdgcn_readlane(tn, bl), __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tw), bl)),
                            __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tp), bl)), __builtin_amdgcn_readlane(tvl, bl),
                            __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tq2), bl)), ep, uvl, 0, m, lane);
                    if (__builtin_expect_with_probability(wins, 1, 0.999)) {
                        run_child = __builtin_amdgcn_readlane(r1, bl) * kWave + bl;
                        run_np = __builtin_amdgcn_readlane(tn, bl);
                        run_sx = __builtin_amdgcn_readlane(tx, bl);
                        run_sy = __builtin_amdgcn_readlane(ty, bl);
                    } else {
                        // ---- the children that can be chosen, one per lane: no other has a score of `from` or more, and m
                        // entries of these have (that child's, or, where too many would be left, the heads of m) ----
                        const float lane_first = score_floor<RAVE>(tn, tw, tp, tvl, tq2, ep);
                        const float first = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(lane_first), bl));
                        float from = fmaxf(last < first ? last : first, kLeastScore);
                        const bool few = together || m <= kPickFew;
                        // (a lane's highest child is the only one of its that can: nothing needs to be moved)
                        const bool direct = __ballot(c2 >= from) == 0ull;
                        auto listed = [&](float t) {
                            int c = 0;
#pragma unroll
                            for (int r = 0; r < RMAX; r++) c += __popcll(__ballot(ceil[r] >= t));
                            return c;
                        };
                        if (!direct) {
                            if (listed(from) > kWave) {
                                float lo = from, hi = key_score(top);
                                int n = 0;
                                for (int it = 0; it < 24; it++) {
                                    const float mid = 0.5f * (lo + hi);
                                    if (!(mid > lo && mid < hi)) break;
                                    n = listed(mid);
                                    if (n < m) hi = mid;
                                    else lo = mid;
                                    if (n >= m && n <= kWave) break;
                                }
                                from = listed(lo) <= kWave ? lo : __builtin_inff();  // (too many alike)
                            }
#pragma unroll
                            for (int r = 0; r < RMAX; r++) {
                                const bool in = ceil[r] >= from;
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
                                }
                                n0 += __popcll(cm);
                            }
                            wave_sync_memory();
                        }
                        const uint32_t floor_key = floor_key_of(from);
                        if (direct && !few) {
                            const bool in = c1 >= from;
                            int cl = 0;  // (in child order, which the merge goes by where keys are equal)
#pragma unroll
                            for (int r = 0; r < RMAX; r++) {
                                const uint64_t cm = __ballot(in && r1 == r);
                                if (r1 == r) cl = n0 + __popcll(cm & ((1ull << lane) - 1ull));
                                n0 += __popcll(cm);
                            }
                            if (in) {
                                my.child[cl] = r1 * kWave + lane;
                                my.n[cl] = tn;
                                my.w[cl] = tw;
                                my.p[cl] = tp;
                                my.vl[cl] = tvl;
                                if (RAVE) my.q2[cl] = tq2;
                                my.sx[cl] = tx;
                                my.sy[cl] = ty;
                            }
                            wave_sync_memory();
                        }
                        if (few && (direct || n0 > 0)) {
                            bool mine = c1 >= from;
                            int child = r1 * kWave + lane, who = 0;
                            if (!direct) {
                                mine = lane < n0;
                                child = my.child[lane];
                                tn = my.n[lane];
                                tvl = my.vl[lane];
                                tw = my.w[lane];
                                tp = my.p[lane];
                                if (RAVE) tq2 = my.q2[lane];
                                tx = my.sx[lane];
                                ty = my.sy[lane];
                            }
                            const bool settled = pick_few<RAVE>(my.order, mine, child, tn, tw, tp, tvl, tq2, together ? 1 : m, ep, uvl,
                                                                floor_key, lane, visits, who);
                            if (settled && together) {
                                run_child = __builtin_amdgcn_readlane(child, who);
                                run_np = __builtin_amdgcn_readlane(tn, who);
                                run_sx = __builtin_amdgcn_readlane(tx, who);
                                run_sy = __builtin_amdgcn_readlane(ty, who);
                            } else if (settled) {
                                serial = false;
                                if (direct && visits > 0) {
                                    my.child[lane] = child;
                                    my.n[lane] = tn;
                                    my.sx[lane] = tx;
                                    my.sy[lane] = ty;
                                }
                                if (direct) n0 = kWave;
                                wave_sync_memory();
                            }
                        } else if (n0 > 0) {
                            serial = !merge_heads<RAVE>(my, n0, m, ep, uvl, floor_key, lane, visits);
                        }
                        replayed = serial && !together;
                    }
                }
                if (__builtin_expect_with_probability(run_child < 0 && serial, 0, 0.999)) {
                    // ---- one visitor after the other (no real score, values that are not finite, a child that was
                    // not listed); the children once more, which spares the ways above the registers ----
                    ask();
                    __builtin_amdgcn_s_waitcnt(0x0F70);  // (as above: else the loop waits in front of its loads, on every way)
                    int cnt[RMAX];
#pragma unroll
                    for (int r = 0; r < RMAX; r++) {
                        const int i = r * kWave + lane;
                        cnt[r] = 0;
                        k.part[r] = i < nelig && ((word[r] >> ((uint32_t)(cb + i) & 31u)) & 1u);
                        score_round<RMAX, RAVE>(k, r, ep);
                    }
                    uint32_t bk, bpos;
                    lane_best<RMAX, RAVE>(k, lane, bk, bpos);
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
                                    my.order[done] = ((uint32_t)i << 16) | (uint32_t)cnt[r];
                                    cnt[r]++;
                                    k.vl[r] = (int)((uint32_t)k.vl[r] + uvl);
                                    score_round<RMAX, RAVE>(k, r, ep);
                                }
                            }
                            lane_best<RMAX, RAVE>(k, lane, bk, bpos);
                        }
                    }
                    if (run_child >= 0) {
#pragma unroll
                        for (int r = 0; r < RMAX; r++) {
                            if (r == (run_child >> 6)) {
                                run_np = __builtin_amdgcn_readlane(k.n[r], run_child & 63);
                                run_sx = __builtin_amdgcn_readlane(sp[r].x, run_child & 63);
                                run_sy = __builtin_amdgcn_readlane(sp[r].y, run_child & 63);
                            }
                        }
                    } else if (!leaf) {
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
                            }
                            n0 += __popcll(cm);
                        }
                        wave_sync_memory();
                        visits = lane < n0 ? my.vl[lane] : 0;
                        if (lane < m) {  // (from the node's children to the listed ones)
                            const uint32_t o = my.order[lane];
                            int cl = 0;
                            while (my.child[cl] != (int)(o >> 16)) cl++;
                            my.order[lane] = ((uint32_t)cl << 16) | (o & 0xFFFFu);
                        }
                    }
                }
                if (a.stats && lane == 0 && m > 1 && !leaf) {
                    atomicAdd(a.stats + 0, 1);
                    atomicAdd(a.stats + 1, serial && run_child < 0 ? 0 : 1);
                    atomicAdd(a.stats + 2, serial && run_child < 0 ? 0 : m);
                    atomicAdd(a.stats + 3, serial && run_child < 0 ? m : 0);
                    // (without a real score, or with values that are not finite, no merge was tried)
                    if (replayed) atomicAdd(a.stats + 4, 1);
                    if (!serial) {
                        atomicAdd(a.stats + 7, 1);
                        atomicAdd(a.stats + 13, 1);
                    }
                }
                if (a.stats && lane == 0 && m == 1 && !leaf) atomicAdd(a.stats + 6, 1);
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
            if (__builtin_expect_with_probability(run_child >= 0, 1, 0.999)) {
                // ---- all of them go down together ----
                node = cb + run_child;
                owed = true;
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
                const int cl = (int)(o >> 16);
                const int next = cb + my.child[cl], kids = my.sy[cl];
                a.paths[(size_t)(depth + 1) * a.stride + t] = next;
                if (ROWS) s.path[v][depth + 1] = next;
                s.list[off + my.start[cl] + (int)(o & 0xFFFFu)] = v;
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
