// Host check of the bounds by which the selection rules children out without dividing (score_about, in_order_at_once,
// csrc/omk_score.h): with reciprocals off by up to two units in the last place either way the exact score (child_keys) lies
// between floor and ceiling, and what in_order_at_once says keys_provably_monotone says too.  Inputs over their whole
// range: counts to 2^31, sums and priors of any magnitude, blends, children without visits, values that are not finite.
//   bound_check [cases [seed]]
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>

#include "omk_score.h"
using namespace omk;

static float off(float x, std::mt19937_64 &rng) {
    for (int by = (int)(rng() % 5) - 2; by != 0 && std::isfinite(x); by += by < 0 ? 1 : -1)
        x = std::nextafter(x, by < 0 ? -INFINITY : INFINITY);
    return x;
}

template <bool RAVE>
static long run(long cases, uint64_t seed, long *decided) {
    std::mt19937_64 rng(seed);
    auto any = [&]() {  // of any magnitude
        const float f = std::ldexp((float)(rng() % (1u << 24)), (int)(rng() % 60) - 50);
        return rng() % 2 ? f : -f;
    };
    long bad = 0;
    for (long c = 0; c < cases; c++) {
        const int n = rng() % 4 == 0 ? 0 : (int)(rng() >> (33 + rng() % 31));
        const int vl = rng() % 2 ? 0 : rng() % 8 == 0 ? (int)(rng() >> 33) : (int)(rng() % 200);
        float w = rng() % 8 == 0 ? any() : (float)(((double)(rng() % 2001) / 1000.0 - 1.0) * n);
        float p = rng() % 8 == 0 ? any() : (float)(rng() % 100000) * 1e-5f;
        float q2 = rng() % 8 == 0 ? any() : (float)(rng() % 2001) * 1e-3f - 1.0f, ep = 1.4f * std::sqrt((float)(rng() % 1000000));
        if (rng() % 50 == 0) (rng() % 2 ? w : p) = rng() % 3 == 0 ? NAN : rng() % 2 ? INFINITY : -INFINITY;
        if (rng() % 50 == 0) w = std::ldexp(w, 100);
        if (rng() % 50 == 0) p = std::ldexp(p, -140);
        if (rng() % 50 == 0) {  // nothing but quotients that underflow
            w = rng() % 2 ? 0.0f : std::ldexp((float)(rng() % 64), -149);
            p = std::ldexp((float)(rng() % 64), -149);
            q2 = 0.0f;
            ep = (float)(1 + rng() % 40);
        }
        const float x = (float)(int)((uint32_t)n + (uint32_t)vl);
        float s, size;
        score_about<RAVE>(n, w, p, vl, q2, ep, off(1.0f / x, rng), off(1.0f / (1.0f + x), rng), s, size);
        const float ceiling = ceiling_of(s, size), floor = floor_of(s, size);
        if (!(ceiling * 0.0f == 0.0f)) continue;  // not finite: settled without the bounds
        uint32_t k1, k2;
        child_keys<RAVE>(n, w, p, vl, q2, ep, k1, k2);
        // a child that is ruled out by the least `from` above its ceiling has no entry above the floor that goes with it; one
        // from whose floor on others are listed is above the floor that goes with that; and none is above the ceiling and kBoundTiny
        const uint32_t key = k1 > k2 ? k1 : k2, lo = floor_key_of(floor) + 1u;
        const uint32_t hi = std::min(floor_key_of(std::nextafter(ceiling, INFINITY)), score_key(ceiling + kBoundTiny));
        (*decided)++;
        if (k1 == 0u || key < lo || key > hi) {
            if (++bad < 5) printf("outside: rave %d n %d vl %d w %a p %a q2 %a ep %a: %08x not in %08x .. %08x\n", (int)RAVE, n, vl, w, p, q2, ep, key, lo, hi);
        }
        const uint32_t uvl = (uint32_t)(rng() % 5);
        const int j = (int)(rng() % 64);
        if (in_order_at_once(n, w, p, vl, ep, uvl, j) &&
            !keys_provably_monotone<RAVE>(n, w, p, vl, q2, ep, uvl, j) && ++bad < 5)
            printf("order: n %d vl %d w %a p %a ep %a uvl %u j %d\n", n, vl, w, p, ep, uvl, j);
    }
    return bad;
}

int main(int argc, char **argv) {
    const long cases = argc > 1 ? atol(argv[1]) : 1000000;
    const uint64_t seed = argc > 2 ? strtoull(argv[2], nullptr, 10) : 1;
    long decided = 0;
    const long bad = run<false>(cases, seed, &decided) + run<true>(cases, seed + 1, &decided);
    printf("bounds: %ld held, wrong %ld\n", decided, bad);
    return bad != 0;
}
