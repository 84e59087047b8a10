// Priors of an expansion's children from the policy over the action space, on the host.
#pragma once
#include <algorithm>
#include <cstdint>
#if !defined(__HIP_DEVICE_COMPILE__)
#include <immintrin.h>
#endif

namespace omk {

// pr[i] = the policy's value of move mv[i], clamped to [0, 1], or 0.01 for a move outside the action space
// (MCTSNode::setPriorProbabilities, src/mcts/mcts_node.cpp:537-560); mv is copied to `moves`.
static inline void gather_priors_plain(const int32_t *mv, int32_t n, const float *pol, int32_t action_space,
                                       int32_t *moves, float *pr) {
    for (int32_t i = 0; i < n; i++) {
        moves[i] = mv[i];
        pr[i] = mv[i] >= 0 && mv[i] < action_space ? std::min(1.0f, std::max(0.0f, pol[mv[i]])) : 0.01f;
    }
}

#if !defined(__HIP_DEVICE_COMPILE__)
// Eight moves at a time.  Same bits: min and max take their second operand where one is NaN, as std::max(0, x) and
// std::min(1, x) do.  The GPU idles meanwhile: 64 offers of 220 moves took 15 us of a batch's 95 one by one.
__attribute__((target("avx2"))) static inline void gather_priors_avx2(const int32_t *mv, int32_t n, const float *pol,
                                                                      int32_t action_space, int32_t *moves, float *pr) {
    const __m256i bound = _mm256_set1_epi32(action_space), below = _mm256_set1_epi32(-1);
    const __m256 zero = _mm256_setzero_ps(), one = _mm256_set1_ps(1.0f), outside = _mm256_set1_ps(0.01f);
    int32_t i = 0;
    for (; i + 8 <= n; i += 8) {
        const __m256i m = _mm256_loadu_si256((const __m256i *)(mv + i));
        const __m256 in =
            _mm256_castsi256_ps(_mm256_and_si256(_mm256_cmpgt_epi32(m, below), _mm256_cmpgt_epi32(bound, m)));
        const __m256 x = _mm256_mask_i32gather_ps(outside, pol, m, in, 4);  // (reads nothing outside the policy)
        const __m256 clamped = _mm256_min_ps(_mm256_max_ps(x, zero), one);
        _mm256_storeu_si256((__m256i *)(moves + i), m);
        _mm256_storeu_ps(pr + i, clamped);  // 0.01 passes the clamp as it is
    }
    gather_priors_plain(mv + i, n - i, pol, action_space, moves + i, pr + i);
}
#endif

static inline void gather_priors(const int32_t *mv, int32_t n, const float *pol, int32_t action_space, int32_t *moves,
                                 float *pr) {
#if !defined(__HIP_DEVICE_COMPILE__)
    static const bool wide = __builtin_cpu_supports("avx2");
    if (wide) return gather_priors_avx2(mv, n, pol, action_space, moves, pr);
#endif
    gather_priors_plain(mv, n, pol, action_space, moves, pr);
}

}  // namespace omk
