// The selection's entry: the reset launch, then the kernels of the forest's fan-out class.  The kernels are in
// omk_select_kernels.h; every class is compiled by a file of its own (omk_select_r*.hip), because they are what the
// build waits for.
#include "omk_internal.h"

namespace omk {

// The scheduler's words before a selection.
__device__ __forceinline__ void reset_words(const SelectArgs &a, int n_items0, int n_singles0, int open0, int n_hctx0) {
    *a.truncated = 0;
    *a.truncated_next = 0;
    *a.n_singles = n_singles0;
    *a.sched_head = 0;
    *a.singles_head = 0;
    *a.sched_tail = n_items0;
    a.sched_wait[0] = open0;
    a.sched_wait[1] = 0;
    *a.hctx_n = n_hctx0;  // the contexts of heavy roots are handed out when the roots are set
    *a.trace_n = 0;
}

// Four arrays from one staging block in pinned memory: a word per thread, so that every read of the host link is in
// flight at once (three synchronous copies and the wait before them took 51 us, this launch 3 us of the host).
// With `prepare` the reset of the next selection as well, from the same words: a search sets its roots before every
// batch, and one launch is then left of two (4 us a batch of a selection's 45).
__global__ __launch_bounds__(256) void k_set_roots(SelectArgs a, int32_t *seg0, int32_t *items0, int32_t *singles0,
                                                   const int32_t *staged, int n, int n_items, int n_singles, int n_hctx0,
                                                   bool prepare) {
    constexpr int W = (int)(sizeof(Item) / 4);
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (prepare) {
        if (i == 0) reset_words(a, n_items, n_singles, n - n_singles, n_hctx0);
        if (i < 3) a.times[i] = 0;
        if (i < n) {
            // a traversal that the selection does not finish (the kernel gave up) has an empty path
            a.path_len[i] = 0;
            a.leaf[i] = -1;
            a.list_flag[i] = 0;
        }
        if (i < n_items) a.q_ready[i] = a.epoch;
        if (i < n_singles) a.single_ready[i] = a.epoch;
    }
    if (i >= 2 * n + (n_items + n_singles) * W) return;
    const int32_t v = staged[i];
    if (i < n) {
        seg0[i] = v;
    } else if (i < 2 * n) {
        a.paths[i - n] = v;
    } else if (i < 2 * n + n_items * W) {
        items0[i - 2 * n] = v;
        if (prepare) reinterpret_cast<int32_t *>(a.items_q)[i - 2 * n] = v;
    } else {
        singles0[i - 2 * n - n_items * W] = v;
        if (prepare) reinterpret_cast<int32_t *>(a.singles_q)[i - 2 * n - n_items * W] = v;
    }
}

hipError_t launch_set_roots(const SelectArgs &a, int32_t *seg0, Item *items0, Item *singles0, const int32_t *staged,
                            int n, int n_items, int n_singles, int n_hctx0, bool prepare, hipStream_t s) {
    const int64_t words = 2ll * n + (int64_t)(n_items + n_singles) * (int)(sizeof(Item) / 4);
    hipLaunchKernelGGL(k_set_roots, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, s, a, seg0, (int32_t *)items0,
                       (int32_t *)singles0, staged, n, n_items, n_singles, n_hctx0, prepare);
    return hipGetLastError();
}

// Scheduler state, statistics, the work queue seeded with the items of the roots, and the
// single-visitor queue seeded with the traversals that are alone at their root.
__global__ void k_select_reset(SelectArgs a, int n_items0, int n_singles0, int open0, int n_traversals, int n_hctx0) {
    const int gid = blockIdx.x * blockDim.x + threadIdx.x;
    const int step = gridDim.x * blockDim.x;
    if (gid == 0) reset_words(a, n_items0, n_singles0, open0, n_hctx0);
    if (a.stats && gid < 16) a.stats[gid] = 0;
    if (gid < 3) a.times[gid] = 0;
    for (int i = gid; i < n_items0; i += step) {
        a.items_q[i] = a.items0[i];
        a.q_ready[i] = a.epoch;
    }
    for (int i = gid; i < n_singles0; i += step) {
        a.singles_q[i] = a.singles0[i];
        a.single_ready[i] = a.epoch;
    }
    // a traversal that the selection does not finish (the kernel gave up) has an empty path
    for (int i = gid; i < n_traversals; i += step) {
        a.path_len[i] = 0;
        a.leaf[i] = -1;
        a.list_flag[i] = 0;
    }
}

hipError_t launch_select(const ForestDev &f, const SelectArgs &a, int n_items0, int n_singles0, int n_traversals,
                         int most_visitors, int max_fanout, bool rave, int n_cus, int n_hctx0,
                         bool prepared, const LoneOut &out, hipStream_t s) {
    // Every traversal alone at its root (one per tree: leaf-parallel self-play): the single-visitor
    // kernel is the whole select and takes its walkers from the host's list; every walker writes its
    // own leaf and path length, so nothing has to be cleared first (the statistics apart).
    // Otherwise the reset launch.
    const bool alone = n_items0 == 0 && n_singles0 == n_traversals;
    const bool blocks = by_blocks(n_items0, most_visitors, max_fanout);
    if ((!alone && !blocks && !prepared) || a.stats || a.trace) {  // (the statistics and the timeline start at zero)
        int reset_blocks = (n_traversals + 255) / 256;
        hipLaunchKernelGGL(k_select_reset, dim3(reset_blocks), dim3(256), 0, s, a, n_items0, n_singles0,
                           n_traversals - n_singles0, n_traversals, n_hctx0);
    }
    if (blocks) return launch_select_blocks(f, a, n_items0, n_singles0, max_fanout, rave, out, s);
#define OMK_DISPATCH(RM)                                                              \
    return rave ? launch_select_class<RM, true>(f, a, n_items0, most_visitors, n_traversals, n_cus, out, s) \
                : launch_select_class<RM, false>(f, a, n_items0, most_visitors, n_traversals, n_cus, out, s)
    if (max_fanout <= 64) { OMK_DISPATCH(1); }
    if (max_fanout <= 256) { OMK_DISPATCH(4); }
    if (max_fanout <= 384) { OMK_DISPATCH(6); }
    OMK_DISPATCH(16);
#undef OMK_DISPATCH
}

}  // namespace omk
