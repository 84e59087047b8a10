// Host check of the rules by which the selection settles a node whose visitors split: pick_few, merge_heads and merge_rest
// (csrc/omk_select_blocks.h, up to 64 visitors) and team_merge (csrc/omk_select_kernels.h).  The same steps, one "lane" at
// a time, with the score arithmetic of csrc/omk_score.h, on random nodes; what a rule accepts is played one visitor at a
// time as well (the serial loop of the reference, mcts_engine_batch_tree_simple.cpp:73-185 applied to one node) and must
// give the same winner order and the same visits per child.
// This pins the RULES (which children are listed, which entries are worked out, the bar up to which they are final, the
// refusals); the device code itself is held against the CPU checker by the GPU tests.
//   merge_check [cases [seed]]
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "omk_score.h"
using namespace omk;

static bool RAVE = true;
struct Kid {
    int n;
    float w, p;
    int vl;
    float q2;
    bool part;
    uint32_t k1, k2;  // of its next visitor
    uint32_t head() const { return k1 > k2 ? k1 : k2; }
};
// An entry: a child's score for its j-th visitor of this node.  Played earlier: larger key, then first scan before second,
// then the children's order, then the visits'.
struct Entry {
    uint32_t key;
    uint64_t place;
    bool before(const Entry &o) const { return key > o.key || (key == o.key && place < o.place); }
    int child() const { return (int)(place >> 21) & 1023; }
    int visit() const { return (int)(place & 0x1FFFFF); }
};
static void keys(const Kid &c, float ep, int vlj, uint32_t &k1, uint32_t &k2) {
    if (RAVE) child_keys<true>(c.n, c.w, c.p, vlj, c.q2, ep, k1, k2);
    else child_keys<false>(c.n, c.w, c.p, vlj, c.q2, ep, k1, k2);
}
static Entry entry(const std::vector<Kid> &k, int child, int j, float ep, uint32_t uvl) {
    uint32_t k1, k2;
    keys(k[child], ep, (int)((uint32_t)k[child].vl + (uint32_t)j * uvl), k1, k2);
    const uint64_t place = ((uint64_t)child << 21) | (uint64_t)j;
    return k2 > k1 ? Entry{k2, place | (1ull << 31)} : Entry{k1, place};
}
static bool monotone(const Kid &c, float ep, uint32_t uvl, int j_last) {
    return RAVE ? keys_provably_monotone<true>(c.n, c.w, c.p, c.vl, c.q2, ep, uvl, j_last)
                : keys_provably_monotone<false>(c.n, c.w, c.p, c.vl, c.q2, ep, uvl, j_last);
}

static float key_score(uint32_t key) {  // what score_key gave it
    const uint32_t b = key & 0x80000000u ? key & 0x7FFFFFFFu : ~key;
    float f;
    memcpy(&f, &b, sizeof(f));
    return f;
}
static long cuts = 0;  // lists of entries that were cut short

struct Played {
    std::vector<Entry> order;
    std::vector<int> taken;  // per child
};

// ---- up to 64 visitors: a lane a child ----
// What is left after `out`: a prefix of every child's list, of whatever lengths, 128 entries in all; the next entry of a
// child of which there is none is not above a bound of its own, here a little above it.
template <typename Lengths, typename Slack>
static bool merge_rest(const std::vector<Kid> &k, const std::vector<int> &L, int m, float ep, uint32_t uvl, uint32_t floor_key,
                       Lengths &&lengths, Slack &&slack, Played &out) {
    while ((int)out.order.size() < m) {
        const int need = m - (int)out.order.size();
        std::vector<int> c;
        int total = 0;
        for (int i : L) {
            const int n = std::min(need, lengths(i, out.taken[i], need));
            c.push_back(n > 0 && n < need ? n + 1 : n);
            total += c.back();
        }
        if (total > 128) {  // in proportion, and one at least
            const float f = (float)(128 - 16) / (float)total;
            total = 0;
            for (int &n : c) {
                if (n > 1) n = 1 + (int)((float)(n - 1) * (L.size() > 16 ? 0.5f : 1.0f) * f);
                total += n;
            }
        }
        if (total == 0 || total > 128) return false;
        std::vector<Entry> all;
        Entry bar{0u, 0};
        for (size_t q = 0; q < L.size(); q++) {
            Entry last{0u, 0};
            for (int j = 0; j < c[q]; j++) {
                const Entry e = entry(k, L[q], out.taken[L[q]] + j, ep, uvl);
                if (j > 0 && e.before(last)) return false;  // not in order
                all.push_back(last = e);
            }
            if (c[q] == 0) last = Entry{entry(k, L[q], out.taken[L[q]], ep, uvl).key + slack(), 0};
            if (c[q] < need && last.key != 0u && (bar.key == 0u || last.before(bar))) bar = last;
        }
        std::vector<Entry> in;
        const uint32_t above = std::max(bar.key, floor_key);
        for (const Entry &e : all)
            if (e.key > above) in.push_back(e);
        if ((int)in.size() < need && bar.key > floor_key)  // (those on the bar's own key)
            for (const Entry &e : all)
                if (e.key == bar.key && !bar.before(e)) in.push_back(e);
        if (in.empty()) return false;
        // far more than are needed: those from a key on that few lie above
        if ((int)in.size() > need + 32) {
            uint32_t top = 0u, cut = 0u;
            for (const Entry &e : in) top = std::max(top, e.key);
            float lo = key_score(above + 1u), hi = key_score(top);
            for (int it = 0; it < 12; it++) {
                const float mid = 0.5f * (lo + hi);
                if (!(mid > lo && mid < hi)) break;
                int n = 0;
                for (const Entry &e : in) n += e.key >= score_key(mid);
                if (n < need) {
                    hi = mid;
                } else {
                    lo = mid;
                    cut = score_key(mid);
                    if (n <= need + 8) break;
                }
            }
            in.erase(std::remove_if(in.begin(), in.end(), [&](const Entry &e) { return e.key < cut; }), in.end());
            cuts++;
        }
        std::sort(in.begin(), in.end(), [](const Entry &a, const Entry &b) { return a.before(b); });
        for (int r = 0; r < (int)in.size() && r < need; r++) {
            out.order.push_back(in[r]);
            out.taken[in[r].child()]++;
        }
    }
    return true;
}
// At first 128 entries, as many of every child; where that settles less than a quarter, as above.
template <typename Lengths, typename Slack>
static bool merge_heads(const std::vector<Kid> &k, const std::vector<int> &L, int m, float ep, uint32_t uvl, uint32_t floor_key,
                        Lengths &&lengths, Slack &&slack, Played &out) {
    const int n0 = (int)L.size();
    int E = 64;
    while (E * n0 > 64) E >>= 1;
    bool proven = true;
    for (int c : L) proven = proven && monotone(k[c], ep, uvl, m - 1);
    while ((int)out.order.size() < m) {
        const int need = m - (int)out.order.size();
        std::vector<Entry> all;
        Entry bar{0u, 0};
        bool bad = false;
        for (int c : L) {
            const int base = out.taken[c], n = std::min(need, E < need ? 2 * E : E);
            Entry last{0u, 0};
            for (int j = 0; j < n; j++) {
                const Entry e = entry(k, c, base + j, ep, uvl);
                if (!proven && j > 0 && e.key != 0u && e.before(last)) bad = true;
                all.push_back(last = e);
            }
            if (2 * E < need && last.key != 0u && (bar.key == 0u || last.before(bar))) bar = last;
        }
        if (bad) return false;
        std::vector<Entry> in;
        for (const Entry &e : all)
            if (e.key > floor_key && !bar.before(e)) in.push_back(e);
        if (in.empty()) return false;
        std::sort(in.begin(), in.end(), [](const Entry &a, const Entry &b) { return a.before(b); });
        for (int r = 0; r < (int)in.size() && r < need; r++) {
            out.order.push_back(in[r]);
            out.taken[in[r].child()]++;
        }
        if (4 * (int)in.size() < need) return merge_rest(k, L, m, ep, uvl, floor_key, lengths, slack, out);
    }
    return true;
}
// Three visitors or fewer: the serial loop over the listed children, while their entries are in order and above the floor.
static bool pick_few(const std::vector<Kid> &k, const std::vector<int> &L, int m, float ep, uint32_t uvl, uint32_t floor_key,
                     Played &out) {
    for (int v = 0; v < m; v++) {
        Entry b{0u, 0};
        for (int i : L) {
            const Entry e = entry(k, i, out.taken[i], ep, uvl), next = entry(k, i, out.taken[i] + 1, ep, uvl);
            if (next.before(e)) return false;
            if (e.key != 0u && (b.key == 0u || e.before(b))) b = e;
        }
        if (b.key <= floor_key) return false;
        out.order.push_back(b);
        out.taken[b.child()]++;
    }
    return true;
}
// Which children a root's block lists for it: those that a bound a little above their next entry's score does not rule out
// against `from`, which lies a little below the best child's last entry (or its first, if that is lower), or where that
// leaves more than 64, with at least m of them.
template <typename Lengths, typename Slack>
static bool by_block(const std::vector<Kid> &k, int m, float ep, uint32_t uvl, Lengths &&lengths, Slack &&slack, Played &out) {
    out.order.clear();
    out.taken.assign(k.size(), 0);
    std::vector<uint32_t> ceiling(k.size(), 0u);
    int best = -1;
    for (int i = 0; i < (int)k.size(); i++)
        if (k[i].head()) {
            ceiling[i] = k[i].head() + slack();
            if (best < 0 || ceiling[i] > ceiling[best]) best = i;
        }
    if (best < 0) return false;
    auto listed = [&](uint32_t T) {
        int n = 0;
        for (uint32_t c : ceiling) n += c >= T;
        return n;
    };
    const uint32_t low = std::min(entry(k, best, m - 1, ep, uvl).key, k[best].head());
    uint32_t from = low > 64u ? low - slack() : 1u;
    if (listed(from) > 64) {
        uint32_t lo = from, hi = ceiling[best];
        while (hi - lo > 1u) {
            const uint32_t mid = lo + ((hi - lo) >> 1);
            const int n = listed(mid);
            (n < m ? hi : lo) = mid;
            if (n >= m && n <= 64) break;
        }
        if (listed(lo) > 64) return false;
        from = lo;
    }
    std::vector<int> L;
    for (int i = 0; i < (int)k.size(); i++)
        if (ceiling[i] >= from) L.push_back(i);
    if (m <= 3) return pick_few(k, L, m, ep, uvl, from - 1u, out);
    return merge_heads(k, L, m, ep, uvl, from - 1u, lengths, slack, out);
}

// ---- any number of visitors: a prefix of every child's list, of whatever lengths ----
// lengths: what is said of child i's entries at or above the threshold, `need` to go (the device: the closed form; here
// anything, since nothing may depend on it)
template <typename Lengths>
static bool team_merge(const std::vector<Kid> &k, int m, float ep, uint32_t uvl, Lengths &&lengths, Played &out) {
    const int nk = (int)k.size(), kBatch = 2048;
    out.order.clear();
    out.taken.assign(nk, 0);
    for (int pass = 0; (int)out.order.size() < m; pass++) {
        if (pass >= 12) return false;
        const int need = m - (int)out.order.size();
        std::vector<int> c(nk, 0);
        int total = 0;
        for (int i = 0; i < nk; i++) {
            if (!k[i].part) continue;
            const Entry head = entry(k, i, out.taken[i], ep, uvl);
            const int n = head.key == 0u ? 0 : std::min(need, lengths(i, out.taken[i], need));
            c[i] = n > 0 && n < need ? n + 1 : n;
            total += c[i];
        }
        if (total > kBatch) {
            const float f = (float)(kBatch - 1024) / (float)total * 0.999f;
            total = 0;
            for (int i = 0; i < nk; i++) {
                if (c[i] > 1) c[i] = 1 + (int)((float)(c[i] - 1) * f);
                total += c[i];
            }
            if (total > kBatch) return false;
        }
        std::vector<Entry> all;
        Entry bar{0u, 0};
        for (int i = 0; i < nk; i++) {
            if (!k[i].part) continue;
            Entry last{0u, 0};
            for (int j = 0; j < c[i]; j++) {
                const Entry e = entry(k, i, out.taken[i] + j, ep, uvl);
                if (j > 0 && e.before(last)) return false;  // not in order
                all.push_back(last = e);
            }
            const Entry head = entry(k, i, out.taken[i], ep, uvl);
            if (c[i] == 0 && head.key != 0u) last = head;
            if ((c[i] == 0 ? head.key != 0u : c[i] < need) && (bar.key == 0u || last.before(bar)) && last.key != 0u) bar = last;
        }
        std::vector<Entry> in;
        for (const Entry &e : all)
            if (!bar.before(e)) in.push_back(e);
        if (in.empty()) return false;
        std::sort(in.begin(), in.end(), [](const Entry &a, const Entry &b) { return a.before(b); });
        for (int r = 0; r < (int)in.size() && r < need; r++) {
            if (in[r].key == 0u) return false;
            out.order.push_back(in[r]);
            out.taken[in[r].child()] = std::max(out.taken[in[r].child()], in[r].visit() + 1);
        }
    }
    return true;
}

int main(int argc, char **argv) {
    const long cases = argc > 1 ? atol(argv[1]) : 100000;
    std::mt19937_64 rng(argc > 2 ? atoll(argv[2]) : 1);
    long block_yes = 0, block_no = 0, team_yes = 0, team_no = 0, wrong = 0;
    auto U = [&](double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); };
    for (long cs = 0; cs < cases; cs++) {
        RAVE = rng() & 1;
        const int nk = 2 + (int)(rng() % (rng() % 4 == 0 ? 380 : 40));
        const int m = 2 + (int)(rng() % (rng() % 2 == 0 ? 63 : rng() % 4 == 0 ? 1500 : 300));
        const uint32_t uvl = 1 + (uint32_t)(rng() % 4);
        const float ep = 1.4f * sqrtf((float)(100 + rng() % 100000));
        std::vector<Kid> k(nk);
        const int style = (int)(rng() % 6);
        for (int i = 0; i < nk; i++) {
            Kid &c = k[i];
            c.part = rng() % 10 != 0;
            c.n = style == 3 ? (int)(rng() % 3) : style >= 4 ? 0 : (int)(rng() % 60);
            if (rng() % 5 == 0) c.n = 0;
            c.w = (float)(U(-0.3, 0.6) * c.n);
            if (rng() % 7 == 0) c.w = floorf(c.w);
            if (rng() % (style == 5 ? 3 : 200) == 0) c.w = -1.5f * (float)c.n - (float)U(0.0, 4.0);  // scores that rise with virtual loss
            if (style == 5 && rng() % 2) c.p *= 30.0f;
            c.p = (float)U(1e-5, style == 1 ? 0.05 : 0.005);
            c.vl = rng() % 5 == 0 ? (int)(rng() % 9) : 0;
            const int rn = (int)(rng() % 40);
            c.q2 = RAVE ? combined_value(c.n, c.w, rn, (float)(U(-0.5, 0.5) * rn), 1000.0f) : 0.0f;
        }
        if (style < 4)
            for (int r = 0; r < (style == 2 ? 4 : 1); r++) {  // a child that dominates, rivals close to it
                Kid &c = k[rng() % nk];
                c.part = true;
                c.n = 20 + (int)(rng() % (r == 0 ? 100000 : 3000));
                c.w = (float)(U(0.6, 0.95) * c.n);
                c.p = (float)U(1e-4, 0.05);
                if (RAVE) c.q2 = combined_value(c.n, c.w, 400, (float)U(-150, 300), 1000.0f);
            }
        for (int r = (int)(rng() % 6); r >= 4; r--) k[rng() % nk] = k[rng() % nk];  // children exactly alike: ties at every visit
        if (rng() % 9 == 0) std::fill(k.begin(), k.end(), Kid(k[0]));
        for (auto &c : k) {
            c.k1 = c.k2 = 0;
            if (c.part) keys(c, ep, c.vl, c.k1, c.k2);
        }
        bool any1 = false;
        for (auto &c : k) any1 = any1 || c.k1 != 0;
        if (!any1) continue;  // (the caller plays such a node one visitor after the other)
        Played serial;
        serial.taken.assign(nk, 0);
        for (int v = 0; v < m; v++) {
            Entry b{0u, 0};
            for (int i = 0; i < nk; i++) {
                if (!k[i].part) continue;
                const Entry e = entry(k, i, serial.taken[i], ep, uvl);
                if (e.key != 0u && (b.key == 0u || e.before(b))) b = e;
            }
            if (b.key == 0u) break;
            serial.order.push_back(b);
            serial.taken[b.child()]++;
        }
        auto hold = [&](bool accepted, const Played &got, const char *who, long &yes, long &no) {
            (accepted ? yes : no)++;
            if (!accepted) return;
            bool same = got.order.size() == serial.order.size() && got.taken == serial.taken;
            for (size_t i = 0; same && i < got.order.size(); i++) same = got.order[i].place == serial.order[i].place;
            if (!same && ++wrong < 5)
                printf("WRONG: %s, case %ld, rave %d, %d children, %d visitors, virtual loss %u\n", who, cs, (int)RAVE, nk, m, uvl);
        };
        Played got;
        // lengths about right, far too short, far too long
        const int how = (int)(rng() % 3);
        auto lengths = [&](int i, int had, int need) {
            const int right = std::max(0, serial.taken[i] - had) + (int)(rng() % 3);
            if (how == 0) return right;
            if (how == 1) return right / (int)(1 + rng() % 4) + (rng() % 8 == 0);
            return right + (int)(rng() % (need + 1));
        };
        auto slack = [&]() { return (uint32_t)(rng() % 17); };
        if (m <= 64) hold(by_block(k, m, ep, uvl, lengths, slack, got), got, "block", block_yes, block_no);
        hold(team_merge(k, m, ep, uvl, lengths, got), got, "team", team_yes, team_no);
    }
    printf("lists cut short: %ld\n", cuts);
    printf("blocks: merged %ld, declined %ld; teams: merged %ld, declined %ld; wrong %ld\n", block_yes, block_no, team_yes, team_no,
           wrong);
    return wrong != 0;
}
