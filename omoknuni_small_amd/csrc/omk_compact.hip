// Breadth-first renumbering of a subtree on the device, for the compaction that follows
// re-rooting (tree reuse between moves: MCTSEngine::searchWithTreeReuse,
// reference src/mcts/mcts_engine_search.cpp:1029-1075, keeps the subtree of the move played
// and drops the rest; with arrays instead of pointers the kept nodes are renumbered so that
// siblings stay contiguous).
//
// order[] receives the old id of every new node: new id 0 is the new root, then level after
// level, a level in the order of its parents, the children of a parent in slot order.
// new_begin[] receives the new id of every node's first child (0 for a node without children).
//
// Two kernels per level, a fixed grid each: every block sums the child counts of its share of the level; then
// every block adds up the sums before its own and writes its nodes' children to the next level.  Where a level
// lies is passed on in device memory (BfsLevel), so the host enqueues several levels at once and reads the sizes
// back once per kBfsLevels levels: 2.5 us a kernel where a scan by the library, two copies back and the wait for
// them took 60 us a level.
#include "omk_internal.h"

namespace omk {

constexpr int kBfsBlocks = 256;  // the second kernel adds up the sums before its own with one load per thread

// This block's share of a level of `cnt` nodes.
__device__ __forceinline__ void bfs_share(int64_t cnt, int64_t &from, int64_t &to) {
    const int64_t per = (cnt + kBfsBlocks - 1) / kBfsBlocks;
    from = per * blockIdx.x;
    to = from + per < cnt ? from + per : cnt;
}

__device__ __forceinline__ int block_sum_256(int v, int *s_part) {
    v = wave_sum_i32(v);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = v;
    __syncthreads();
    const int sum = s_part[0] + s_part[1] + s_part[2] + s_part[3];
    __syncthreads();
    return sum;
}

__global__ __launch_bounds__(256) void k_bfs_counts(const int2 *span, const int32_t *order, const BfsLevel *levels,
                                                    int level, int *sums) {
    __shared__ int s_part[4];
    const BfsLevel l = levels[level];
    if (l.cnt <= 0) return;
    int64_t from, to;
    bfs_share(l.cnt, from, to);
    int c = 0;
    for (int64_t p = from + threadIdx.x; p < to; p += 256) {
        const int y = span[order[l.lo + p]].y;
        c += y > 0 ? y : 0;
    }
    c = block_sum_256(c, s_part);
    if (threadIdx.x == 0) sums[blockIdx.x] = c;
}

// room: ids the order array holds.  A level that does not fit says so (cnt -1) and ends the walk: the child
// ranges then do not form a tree.
__global__ __launch_bounds__(256) void k_bfs_place(const int2 *span, int32_t *order, int32_t *new_begin, BfsLevel *levels,
                                                   int level, const int *sums, int64_t room) {
    __shared__ int s_part[4];
    __shared__ int s_wave[4];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const BfsLevel l = levels[level];
    if (l.cnt <= 0) {
        if (blockIdx.x == 0 && tid == 0) levels[level + 1] = BfsLevel{l.lo, l.cnt};
        return;
    }
    // (a level of a tree holds fewer than 2^31 nodes; a sum that wraps is caught by the room check as it grows)
    int64_t below = block_sum_256(tid < (int)blockIdx.x ? sums[tid] : 0, s_part);
    const int64_t total = block_sum_256(sums[tid], s_part);
    const int64_t next = l.lo + l.cnt;
    const bool fits = total >= 0 && next + total <= room;
    if (blockIdx.x == 0 && tid == 0) levels[level + 1] = BfsLevel{next, fits ? total : -1};
    if (!fits) return;
    int64_t from, to;
    bfs_share(l.cnt, from, to);
    for (int64_t tile = from; tile < to; tile += 256) {
        const int64_t p = tile + tid;
        int2 sp = int2{0, 0};
        if (p < to) sp = span[order[l.lo + p]];
        if (sp.y < 0) sp.y = 0;
        const int upto = wave_inclusive_sum(sp.y, lane);
        if (lane == 63) s_wave[w] = upto;
        __syncthreads();
        int64_t first = next + below + upto - sp.y;
        for (int q = 0; q < w; q++) first += s_wave[q];
        below += s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
        __syncthreads();
        if (p < to) new_begin[l.lo + p] = sp.y > 0 ? (int32_t)first : 0;
        // the wavefront writes the children of one of its nodes after another, most nodes having none
        for (uint64_t todo = __ballot(sp.y > 0); todo; todo &= todo - 1) {
            const int src = __ffsll((long long)todo) - 1;
            const int64_t at = __shfl((long long)first, src);
            const int cb = __shfl(sp.x, src), cc = __shfl(sp.y, src);
            for (int j = lane; j < cc; j += 64) order[at + j] = cb + j;
        }
    }
}

hipError_t launch_bfs(const int2 *span, int32_t *order, int32_t *new_begin, BfsLevel *levels, int from, int n_levels,
                      int *sums, int64_t room, hipStream_t s) {
    for (int l = from; l < from + n_levels; l++) {
        hipLaunchKernelGGL(k_bfs_counts, dim3(kBfsBlocks), dim3(256), 0, s, span, order, levels, l, sums);
        hipLaunchKernelGGL(k_bfs_place, dim3(kBfsBlocks), dim3(256), 0, s, span, order, new_begin, levels, l, sums, room);
    }
    return hipGetLastError();
}

__global__ void k_bfs_start(int32_t *order, BfsLevel *levels, int32_t root) {
    order[0] = root;
    levels[0] = BfsLevel{0, 1};
}

hipError_t launch_bfs_start(int32_t *order, BfsLevel *levels, int32_t root, hipStream_t s) {
    hipLaunchKernelGGL(k_bfs_start, dim3(1), dim3(1), 0, s, order, levels, root);
    return hipGetLastError();
}

// New node i takes word map[i] of every array of `g` (64-bit words where step is 2); the child range (q == span)
// keeps its length and starts at new_begin[i].  Everything of one node in one pass over the map, into tmp, array
// after array, and back by one copy: the gathers of different arrays overlap, where one launch per array and
// another to copy it back were eighteen.
__global__ __launch_bounds__(256) void k_compact_gather(CompactFields g, uint32_t *tmp, const int32_t *map,
                                                        const int32_t *new_begin, int64_t k) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= k) return;
    const int64_t old = map[i];
    int64_t at = 0;
    for (int q = 0; q < g.n; q++) {
        if (g.kind[q] == 1) {
            tmp[at + i] = g.array[q][old];
            at += k;
            continue;
        }
        uint2 v = reinterpret_cast<const uint2 *>(g.array[q])[old];
        if (g.kind[q] == 3) v.x = (int)v.y > 0 ? (uint32_t)new_begin[i] : 0u;
        reinterpret_cast<uint2 *>(tmp + at)[i] = v;
        at += 2 * k;
    }
}

__global__ __launch_bounds__(256) void k_compact_back(CompactFields g, const uint32_t *tmp, int64_t k) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= k) return;
    int64_t at = 0;
    for (int q = 0; q < g.n; q++) {
        if (g.kind[q] == 1) {
            g.array[q][i] = tmp[at + i];
            at += k;
            continue;
        }
        reinterpret_cast<uint2 *>(g.array[q])[i] = reinterpret_cast<const uint2 *>(tmp + at)[i];
        at += 2 * k;
    }
}

hipError_t launch_compact(const CompactFields &g, uint32_t *tmp, const int32_t *map, const int32_t *new_begin, int64_t k,
                          hipStream_t s) {
    if (k <= 0 || g.n == 0) return hipSuccess;
    const dim3 grid((unsigned)((k + 255) / 256)), block(256);
    hipLaunchKernelGGL(k_compact_gather, grid, block, 0, s, g, tmp, map, new_begin, k);
    hipLaunchKernelGGL(k_compact_back, grid, block, 0, s, g, tmp, k);
    return hipGetLastError();
}

// legal bit of new node i = legal bit of old node order[i]: a node per lane, a word of the new mask per half
// wavefront (one thread per word took 32 dependent trips: 10 us for 140 k nodes)
__global__ __launch_bounds__(256) void k_gather_legal(uint32_t *dst, const uint32_t *src, const int32_t *order,
                                                      int64_t k) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    bool bit = false;
    if (i < k) {
        const uint32_t old = (uint32_t)order[i];
        bit = (src[old >> 5] >> (old & 31u)) & 1u;
    }
    const uint64_t mask = __ballot(bit);
    if (i < k && (threadIdx.x & 31) == 0) dst[i >> 5] = (threadIdx.x & 32) ? (uint32_t)(mask >> 32) : (uint32_t)mask;
}

// Plain fill kernel: used instead of hipMemsetAsync wherever a caller might capture the stream
// into a graph.
__global__ __launch_bounds__(256) void k_fill_words(uint32_t *dst, uint32_t value, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t step = (int64_t)gridDim.x * 256;
    for (; i < n; i += step) dst[i] = value;
}

hipError_t launch_fill_words(void *dst, uint32_t value, int64_t n_words, hipStream_t s) {
    if (n_words <= 0) return hipSuccess;
    int64_t blocks = (n_words + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_fill_words, dim3((unsigned)blocks), dim3(256), 0, s, (uint32_t *)dst, value, n_words);
    return hipGetLastError();
}

hipError_t launch_gather_legal(uint32_t *dst, const uint32_t *src, const int32_t *order, int64_t k, hipStream_t s) {
    if (k <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_gather_legal, dim3((unsigned)((k + 255) / 256)), dim3(256), 0, s, dst, src, order, k);
    return hipGetLastError();
}

}  // namespace omk
