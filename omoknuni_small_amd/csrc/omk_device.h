// Device-side building blocks shared by the kernels: wave64 cross-lane reductions
// written with DPP row operations, the order-preserving score key and the per-child
// score arithmetic of MCTSNode::selectChild (reference src/mcts/mcts_node.cpp:94-95,
// 143-160, 196-214) and getCombinedValue (:657-678).
//
// Everything here assumes all 64 lanes of the wavefront are active at the call site.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "omk_score.h"

namespace omk {

constexpr int kWave = 64;

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_mov(uint32_t v) {
    // lanes whose source lane does not exist keep their own value
    return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xF, 0xF, false);
}

// for patterns in which every lane has a source lane: fuses with the instruction that uses it
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_mov_all(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
}

__device__ __forceinline__ uint32_t umax32(uint32_t a, uint32_t b) { return a > b ? a : b; }
__device__ __forceinline__ uint32_t umin32(uint32_t a, uint32_t b) { return a < b ? a : b; }

// Butterfly inside each row of 16 lanes (quad swaps, then row shifts by 4 and 8), after
// which lane 15 of every row holds the row's result; the four row results are combined
// on the scalar unit.
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    v = umax32(v, dpp_mov<0xB1>(v));   // quad_perm [1,0,3,2]
    v = umax32(v, dpp_mov<0x4E>(v));   // quad_perm [2,3,0,1]
    v = umax32(v, dpp_mov<0x114>(v));  // row_shr:4
    v = umax32(v, dpp_mov<0x118>(v));  // row_shr:8
    uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)v, 15);
    uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)v, 31);
    uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)v, 47);
    uint32_t d = (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
    return umax32(umax32(a, b), umax32(c, d));
}

// The same, in every lane and without the scalar unit: rows of 16 by mirrors, then rows and halves exchanged
// (v_permlane16_swap, v_permlane32_swap).  37 ns where wave_max_u32 takes 57, for a caller that compares lanes with it.
__device__ __forceinline__ uint32_t wave_max_all(uint32_t v) {
    v = umax32(v, dpp_mov_all<0xB1>(v));
    v = umax32(v, dpp_mov_all<0x4E>(v));
    v = umax32(v, dpp_mov_all<0x141>(v));  // row_half_mirror
    v = umax32(v, dpp_mov_all<0x140>(v));  // row_mirror
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = umax32(r[0], r[1]);
    const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return umax32(h[0], h[1]);
}

__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
    v = umin32(v, dpp_mov<0xB1>(v));
    v = umin32(v, dpp_mov<0x4E>(v));
    v = umin32(v, dpp_mov<0x114>(v));
    v = umin32(v, dpp_mov<0x118>(v));
    uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)v, 15);
    uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)v, 31);
    uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)v, 47);
    uint32_t d = (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
    return umin32(umin32(a, b), umin32(c, d));
}

// Sum over the 64 lanes: xor butterfly inside each row of 16 (quad swaps, half-row mirror,
// row mirror leave the row total in every lane), the four row totals added on the scalar unit.
__device__ __forceinline__ int wave_sum_i32(int x) {
    uint32_t v = (uint32_t)x;
    v += dpp_mov<0xB1>(v);   // quad_perm [1,0,3,2]
    v += dpp_mov<0x4E>(v);   // quad_perm [2,3,0,1]
    v += dpp_mov<0x141>(v);  // row_half_mirror
    v += dpp_mov<0x140>(v);  // row_mirror
    uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)v, 0);
    uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)v, 16);
    uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)v, 32);
    uint32_t d = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
    return (int)(a + b + c + d);
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_mov_zero(uint32_t v) {
    // lanes whose source lane does not exist receive 0
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
}

// Inclusive prefix sum over the 64 lanes: log-step scan inside each row of 16 with row
// shifts, then the totals of the rows below are added from the scalar unit.
__device__ __forceinline__ int wave_inclusive_sum(int x, int lane) {
    uint32_t v = (uint32_t)x;
    v += dpp_mov_zero<0x111>(v);  // row_shr:1
    v += dpp_mov_zero<0x112>(v);  // row_shr:2
    v += dpp_mov_zero<0x114>(v);  // row_shr:4
    v += dpp_mov_zero<0x118>(v);  // row_shr:8
    uint32_t t0 = (uint32_t)__builtin_amdgcn_readlane((int)v, 15);
    uint32_t t1 = (uint32_t)__builtin_amdgcn_readlane((int)v, 31);
    uint32_t t2 = (uint32_t)__builtin_amdgcn_readlane((int)v, 47);
    const int row = lane >> 4;
    uint32_t add = row >= 1 ? t0 : 0u;
    add += row >= 2 ? t1 : 0u;
    add += row >= 3 ? t2 : 0u;
    return (int)(v + add);
}

// smallest k >= 1 with k*k >= n
__device__ __forceinline__ int ceil_sqrt_i32(int n) {
    if (n <= 1) return 1;
    long long k = (long long)sqrt((double)n);
    while (k * k < (long long)n) k++;
    while ((k - 1) * (k - 1) >= (long long)n) k--;
    return (int)k;
}

// A float as an unsigned number with the same order (score_key without its special cases: not a number in particular).
__device__ __forceinline__ uint32_t ordered_bits(float x) {
    const uint32_t b = __float_as_uint(x);
    return b ^ ((uint32_t)((int32_t)b >> 31) | 0x80000000u);
}

// No score of the child is above this and kBoundTiny (score_about; v_rcp_f32 is within one unit in the last place) ..
template <bool RAVE>
__device__ __forceinline__ float score_ceiling(int n, float w, float p, int vl, float q2, float ep) {
    const float x = (float)(int)((uint32_t)n + (uint32_t)vl);
    float s, size;
    score_about<RAVE>(n, w, p, vl, q2, ep, __builtin_amdgcn_rcpf(x), __builtin_amdgcn_rcpf(1.0f + x), s, size);
    return ceiling_of(s, size);
}
// .. and none below this.
template <bool RAVE>
__device__ __forceinline__ float score_floor(int n, float w, float p, int vl, float q2, float ep) {
    const float x = (float)(int)((uint32_t)n + (uint32_t)vl);
    float s, size;
    score_about<RAVE>(n, w, p, vl, q2, ep, __builtin_amdgcn_rcpf(x), __builtin_amdgcn_rcpf(1.0f + x), s, size);
    return floor_of(s, size);
}

// Results for a host that polls: pinned memory is written with stores of system scope, which go past the L2 of
// the XCD they come from (a plain store may stay in it, and the release of another XCD's block does not write it
// back: with plain stores 1 % of 4 MB had not arrived when the flag had).
template <typename T>
__device__ __forceinline__ void host_store(T *p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Until this wavefront's own stores have been acknowledged.  For a wavefront that hands what it stored to another one, whose
// release of agent scope announces it to other blocks: that one waits for its own stores only, and a release of workgroup
// scope or a block barrier waits for none in memory.
__device__ __forceinline__ void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// The end of a kernel whose results the host waits for (all threads of all blocks take part): every wavefront
// waits until its own host_stores have been acknowledged, and the last of the grid's `blocks` blocks stores the
// call's number to the host's flag.  The host polls that word.  Measured on an MI355X from the launch to the
// host's seeing it: 7.1 us for 1 KB, 7.6 for 64 KB, 27 for 1 MB, 82 for 4 MB (50 GB/s, the link's rate); a
// second kernel that raises the flag costs 1.6 us more, a release of system scope per block 27 % more at 1 MB.
// One kernel and hipStreamSynchronize take 11 us, a copy back into pageable memory 14 more.
__device__ __forceinline__ void host_signal(int32_t *count, int32_t *flag, int32_t seq, int blocks) {
    wait_stores();
    __syncthreads();
    if (threadIdx.x != 0) return;
    if (blocks > 1) {
        const int before = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (before != blocks - 1) return;
        __hip_atomic_store(count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    host_store(flag, seq);
}

}  // namespace omk
