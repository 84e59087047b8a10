// C ABI of libomk_forest.so: handles, host<->device transfers, structural validation,
// and the launch glue of the selection / backup kernels.  Declarations and the reference
// interfaces they replace: include/omk_forest.h.
#include "../../include/omk_forest.h"

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <vector>

#include "omk_internal.h"
#include "omk_priors.h"
#include "omk_staging.h"

using namespace omk;

static thread_local char g_err[512] = "";

static int fail(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

#define HIP_TRY(expr)                                                                              \
    do {                                                                                           \
        hipError_t e_ = (expr);                                                                    \
        if (e_ != hipSuccess) return fail(OMK_ERR_HIP, "%s: %s", #expr, hipGetErrorString(e_));    \
    } while (0)

// No C++ exception crosses the C boundary: what ends the entry points that hold host vectors.
#define OMK_NO_THROW \
    catch (const std::exception &e_) { return fail(OMK_ERR_INVALID, "out of host memory (%s)", e_.what()); }

struct omk_forest {
    int device = 0;
    int64_t capacity = 0;
    int64_t n_nodes = 0;
    bool has_rave = false;
    bool uploaded = false;
    bool prior_sorted = false;
    // What the last call changed the structure by, if it was an expansion: node made_node[i] has made_count[i] children
    std::vector<int32_t> made_node, made_count;
    int max_fanout = 0;
    // Counts the changes that give node ids a new meaning (a compaction, an upload of a different
    // structure): paths, roots and work items of a batch made before such a change are stale.
    int64_t generation = 0;
    uint64_t structure_sum = 0;  // checksum of the child ranges last uploaded
    bool structure_changed = false;  // the device's child ranges are no longer the uploaded ones (expansion, compaction)
    hipStream_t own_stream = nullptr;
    hipStream_t stream = nullptr;
    // device arrays
    int2 *span = nullptr;
    int32_t *N = nullptr, *VL = nullptr, *rN = nullptr, *action = nullptr;
    float *W = nullptr, *P = nullptr, *rW = nullptr;
    // RAVE blend per node (ForestDev::q2): valid for the RAVE constant blend_k while blend_valid; whatever
    // changes N, W, rN or rW of nodes refreshes it or clears the flag
    float *Q2 = nullptr;
    bool blend_valid = false, blend_k_known = false;
    float blend_k = 0.0f;
    uint32_t *legal = nullptr;
    uint64_t *hash = nullptr;
    bool has_legal = false, has_action = false, has_hash = false;
    // Child slots re-pointed at transpositions (omk_tt_select_redirect): alias[s] >= 0 = the node slot s holds
    // instead of node s.  Allocated by the first such call; `redirected` once a slot has been re-pointed: the
    // forest is then a graph, and what assumes a tree refuses it until the next upload.
    int32_t *alias = nullptr;
    bool redirected = false;
    // The way between the host and the kernels: one block of pinned memory that both sides address (see link_*).
    char *link = nullptr;
    Staging staging;
    int32_t link_seq = 0;         // number of the last call that waited
    int32_t *link_count = nullptr;  // HostSignal::count
    char *scratch = nullptr;  // work space of a compaction, kept for the next (kKeepScratch)
    size_t scratch_bytes = 0;
    // counts the calls that change N or child ranges: what was read of them before is stale after
    int64_t changes = 0;
    int children = 0;       // live batches and tables created on this forest
    bool released = false;  // omk_forest_destroy was called while children were alive

    ForestMut mut() const {
        ForestMut m;
        m.span = span;
        m.N = N;
        m.W = W;
        m.P = P;
        m.VL = VL;
        m.rN = has_rave ? rN : nullptr;
        m.rW = has_rave ? rW : nullptr;
        m.q2 = has_rave ? Q2 : nullptr;
        m.legal = has_legal ? legal : nullptr;
        m.action = has_action ? action : nullptr;
        m.hash = has_hash ? hash : nullptr;
        return m;
    }

    ForestDev dev() const {
        ForestDev d;
        d.span = span;
        d.N = N;
        d.W = W;
        d.P = P;
        d.VL = VL;
        d.rN = has_rave ? rN : nullptr;
        d.rW = has_rave ? rW : nullptr;
        d.q2 = has_rave ? Q2 : nullptr;
        d.legal = has_legal ? legal : nullptr;
        d.action = has_action ? action : nullptr;
        d.hash = has_hash ? hash : nullptr;
        d.n_nodes = n_nodes;
        return d;
    }
};

constexpr int kSchedStep = 1024;  // int32 words between two scheduler words: 4 KiB
// Simulations cut by max_depth: two counters, used in turn (select calls of even / odd number).  Every
// select clears the counter of the next one, so that a select of lone traversals needs no reset launch.
constexpr int kTruncatedWord = 40;
constexpr int kTraceCap = 16384;  // records of the timeline of one select

struct omk_batch {
    omk_forest *f = nullptr;
    int32_t max_traversals = 0;
    int32_t max_depth = 0;
    int32_t stride = 0;
    int32_t n = 0;          // traversals bound by set_roots
    int64_t generation = -1;  // the forest's generation when the roots were set
    bool selected = false;  // paths of a select are on the device
    // What the selection that made them says of the paths.  (What the forest or the roots are
    // like when they are settled says nothing: paths that follow transpositions meet in nodes that several trees
    // hold, and an upload makes the forest a tree again under them.)
    PathsAre paths_are = PathsAre::kAny;
    bool one_root = false;  // of all traversals
    bool stamped = false;  // the last selection has left its time stamps
    int32_t *paths = nullptr, *path_len = nullptr, *leaf = nullptr;
    float *values = nullptr;
    Item *items0 = nullptr, *items_q = nullptr, *singles0 = nullptr, *singles_q = nullptr;
    int32_t n_singles0 = 0;
    int32_t most_visitors = 1;  // of one root
    bool in_order = true;       // the traversals' roots ascend
    int32_t n_hctx0 = 0;  // contexts of heavy roots, handed out when the roots are set
    int32_t *seg0 = nullptr, *seg[2] = {nullptr, nullptr};
    int32_t *sc_child = nullptr, *sc_occ = nullptr;
    // [1..16] work statistics, [17] single-visitor queue length, [32] status of omk_batch_leaf_keys,
    // [40..41] simulations cut by max_depth (kTruncatedWord);
    // the scheduler words of the multi-visitor kernel follow at 4 KiB steps (kSchedStep), so
    // that each lies in a memory channel of its own
    int32_t *counters = nullptr;
    int32_t poll_sleep = 1;
    bool stats_on = false;
    bool trace_on = false;  // the selection records its timeline (omk_batch_set_trace)
    int32_t *q_ready = nullptr;  // per queue slot: number of the select call that published it
    int32_t *single_ready = nullptr;  // the same per entry of the single-visitor queue
    int32_t *hctx = nullptr;     // contexts of heavy nodes
    int32_t *hbound = nullptr;   // boundaries between their slices
    int32_t *list_flag = nullptr;  // per visitor-list start: which depth's list is complete
    int32_t hctx_cap = 0;
    int32_t q_cap = 0;
    int32_t epoch = 0;           // select calls so far
    int32_t prepared = 0;        // number of the call that omk_batch_set_roots has made the reset for (0: none)
    int32_t spin_limit = 1 << 18;  // polls of about a microsecond: a quarter of a second, a selection takes a millisecond
    int32_t n_cus = 0;
    int32_t n_items0 = 0;
    int32_t *out = nullptr;  // the leaf gather in pinned memory (see gather), out_bytes of it
    size_t out_bytes = 0;
    std::unique_ptr<int32_t[]> heads;  // the leaves and their counts of a gather that crossed in pieces
    ExportOut gathered = {};      // its parts
    // which selection it is of (the forest's and the batch's counts when it was made): an expansion takes leaves,
    // child counts and visit counts from it while nothing has changed them
    int64_t select_calls = 0, gathered_call = -1, gathered_changes = -1;
    // The gather that a selection of lone traversals has made itself (lone_rows): its call, the forest's changes
    // before it, its number, and the point of the stream it lies at (Staging::now).  read_call: the selection that
    // was read last.
    int64_t lone_call = -1, lone_changes = -1, read_call = -1;
    int32_t lone_seq = 0;
    uint64_t lone_staged = 0;
    std::vector<int32_t> leaf_table;  // work space of an expansion
    std::vector<int32_t> winners, counts;
    long long *trace = nullptr;  // records of the timeline, kTraceCap of them
    std::vector<int32_t> order, order_tmp;  // work space of omk_batch_set_roots
    std::vector<Item> items_h, singles_h;
};

struct omk_tt {
    omk_forest *f = nullptr;
    int log2_slots = 0;
    TTSlot *slots = nullptr;
    TTMeta *meta = nullptr;
    int *d_status = nullptr;       // 8 counters: zero between calls, read and cleared at the end of one (tt_counts)
    uint32_t clock = 0;            // access_counter_ of the reference: entry i of a call has the time clock + i
    float threshold = 0.1f;        // Config::replacement_threshold
    void *work = nullptr;          // staging of store / traverse calls
    size_t work_bytes = 0;
    int64_t generation = -1;       // the forest's generation the stored node ids belong to (-1: nothing stored yet)
};

// The entries hold node ids.  They are the reference's weak_ptr entries, which die with the tree they
// point into (PHMapTranspositionTable::lookup erases an entry whose node is gone,
// src/mcts/phmap_transposition_table.cpp:100-108): once the forest's node ids have taken a new meaning
// (a compaction, an upload of another tree), every entry stored before is such a dead entry, and the
// table is emptied before anything else is done with it.  The access counter runs on, as the
// reference's does.
static int tt_same_tree(omk_tt *tt) {
    omk_forest *f = tt->f;
    if (tt->generation == f->generation) return OMK_OK;
    if (tt->generation >= 0) HIP_TRY(launch_tt_clear(tt->slots, tt->meta, tt->log2_slots, f->stream));
    tt->generation = f->generation;
    return OMK_OK;
}

static int tt_work(omk_tt *tt, size_t bytes) {
    if (bytes <= tt->work_bytes) return OMK_OK;
    HIP_TRY(hipStreamSynchronize(tt->f->stream));
    if (tt->work) HIP_TRY(hipFree(tt->work));
    tt->work = nullptr;
    tt->work_bytes = 0;
    HIP_TRY(hipMalloc(&tt->work, bytes));
    tt->work_bytes = bytes;
    return OMK_OK;
}

template <typename T>
static hipError_t dalloc(T **p, int64_t count) {
    return hipMalloc((void **)p, (size_t)std::max<int64_t>(count, 1) * sizeof(T));
}

// ---- the host's side of the pinned block ----
//
// A copy of a few hundred bytes between pageable memory and the card costs 12 us (to the card) to 20 us (back)
// on an MI355X, and hipStreamSynchronize 5 us more than a kernel's store into pinned memory that the host polls.
// So a call's inputs are copied into the staging part of this block, which the kernels read through the host
// link, and its results come back into pinned memory, followed by the call's number in the flag word.
// Staging is handed out front to back; once a call has seen its flag everything enqueued before has run, and
// the next one starts at the front again.  It stays as large as it is: a call with more than that sends it in pieces.
constexpr size_t kLinkHead = 4096;         // the flag word, on a page of its own
constexpr size_t kLinkStaging = 4 << 20;   // (30 us to allocate, like 4 KiB)
constexpr size_t kLinkPiece = 1 << 20;     // what does not fit goes in pieces of this, four of them on their way
static hipError_t link_alloc(omk_forest *f) {
    hipError_t e = hipHostMalloc((void **)&f->link, kLinkHead + kLinkStaging, hipHostMallocDefault);
    if (e != hipSuccess) return e;
    f->staging = Staging(kLinkStaging);
    *(int32_t *)f->link = f->link_seq;
    return hipSuccess;
}

// `bytes` (at most kLinkStaging) of staging, aligned to a cache line; valid until the next call that waits for the
// stream.
static int link_stage(omk_forest *f, size_t bytes, void **out) {
    size_t at = f->staging.take(bytes);
    if (at == Staging::kFull) {
        HIP_TRY(hipStreamSynchronize(f->stream));
        f->staging.idle();
        at = f->staging.take(bytes);
        if (at == Staging::kFull) return fail(OMK_ERR_INVALID, "%zu bytes of staging", bytes);
    }
    *out = f->link + kLinkHead + at;
    return OMK_OK;
}

static HostSignal link_signal(omk_forest *f) {
    f->link_seq = (int32_t)((uint32_t)f->link_seq + 1u);
    return HostSignal{f->link_count, (int32_t *)f->link, f->link_seq};
}

// Waits for the kernel that carries the link_signal of number `seq`.  A wait of more than about a millisecond goes
// to the runtime, which does not burn the core and reports an error of the stream.
static int link_wait_for(omk_forest *f, int32_t seq) {
    const int32_t *flag = (const int32_t *)f->link;
    auto reached = [&] { return (int32_t)((uint32_t)__atomic_load_n(flag, __ATOMIC_ACQUIRE) - (uint32_t)seq) >= 0; };
    for (int i = 0; i < 20000; i++) {
        if (reached()) return OMK_OK;
#if defined(__x86_64__)
        __builtin_ia32_pause();
#endif
    }
    HIP_TRY(hipStreamSynchronize(f->stream));
    if (!reached()) return fail(OMK_ERR_HIP, "the kernel that was waited for did not report");
    return OMK_OK;
}

// Waits for the last one: everything enqueued has run, and staging starts at the front again.
static int link_wait(omk_forest *f) {
    if (int rc = link_wait_for(f, f->link_seq)) return rc;
    f->staging.idle();
    return OMK_OK;
}

// Bulk transfers (omk_link.hip): arrays of the host, one per segment, to or from the device.  What fits in the
// staging goes in one piece; more is cut into pieces, kBulkSlots or kBackSlots of them on their way at a time, so
// that the host's copy of one piece runs beside the link's transfer of the next.
struct Bulk {
    Segments g = {};
    char *host[kMaxSegments] = {};
    Bulk() { g.start[0] = 0; }
    void add(void *dev, int step, const void *h, int64_t words) {
        if (!h || words <= 0) return;
        g.dev[g.n] = (uint32_t *)dev;
        g.step[g.n] = step;
        host[g.n] = (char *)const_cast<void *>(h);
        g.n++;
        g.start[g.n] = g.start[g.n - 1] + words;
    }
    int64_t words() const { return g.start[g.n]; }
    // the host's side of words [first, first + count)
    template <class F>
    void each(int64_t first, int64_t count, F &&f) const {
        for (int q = 0; q < g.n; q++) {
            const int64_t lo = std::max(first, g.start[q]), hi = std::min(first + count, g.start[q + 1]);
            if (lo < hi) f(host[q] + (lo - g.start[q]) * 4, (lo - first) * 4, (size_t)(hi - lo) * 4);
        }
    }
};
// Pieces to the card: of 1 MB, what counts is the kernels' reading of the link, which smaller ones slow down (8.4 MB:
// 285 us, in pieces of 512 KB 300).  Pieces back: of 512 KB, what counts is the host's copy out of them, which works
// best on what its cache holds (11.5 MB: 372 us, in pieces of 1 MB 411, of 256 KB 435, without the copy 262).
constexpr int64_t kBulkWords = 1 << 18, kBackWords = 1 << 17;
constexpr int kBulkSlots = 4, kBackSlots = 8;
static_assert(kBulkWords * kBulkSlots * 4 <= (int64_t)kLinkStaging, "the slots are the staging");
static_assert(kBackWords * kBackSlots * 4 <= (int64_t)kLinkStaging, "the slots are the staging");

static int bulk_put(omk_forest *f, const Bulk &b) {
    const int64_t words = b.words();
    const bool whole = words <= kBulkWords * kBulkSlots;
    void *staged = nullptr;
    if (int rc = link_stage(f, (size_t)(whole ? words : kBulkWords * kBulkSlots) * 4, &staged)) return rc;
    char *at = (char *)staged;
    if (whole) {
        b.each(0, words, [&](char *h, int64_t off, size_t n) { memcpy(at + off, h, n); });
        HIP_TRY(launch_put(b.g, (const uint32_t *)at, 0, words, HostSignal{nullptr, nullptr, 0}, f->stream));
        return OMK_OK;
    }
    int32_t seq[kBulkSlots] = {};
    for (int64_t c = 0; c * kBulkWords < words; c++) {
        const int slot = (int)(c % kBulkSlots);
        char *p = at + (size_t)slot * kBulkWords * 4;
        const int64_t first = c * kBulkWords, n = std::min(kBulkWords, words - first);
        if (c >= kBulkSlots)
            if (int rc = link_wait_for(f, seq[slot])) return rc;
        b.each(first, n, [&](char *h, int64_t off, size_t bytes) { memcpy(p + off, h, bytes); });
        const HostSignal sig = link_signal(f);
        seq[slot] = sig.seq;
        HIP_TRY(launch_put(b.g, (const uint32_t *)p, first, n, sig, f->stream));
    }
    return link_wait(f);
}

static int bulk_get(omk_forest *f, const Bulk &b) {
    const int64_t words = b.words(), pieces = (words + kBackWords - 1) / kBackWords;
    if (pieces == 0) return OMK_OK;
    void *staged = nullptr;
    if (int rc = link_stage(f, (size_t)std::min<int64_t>(words, kBackWords * kBackSlots) * 4, &staged)) return rc;
    char *at = (char *)staged;
    int32_t seq[kBackSlots] = {};
    auto ask = [&](int64_t c) {
        const HostSignal sig = link_signal(f);
        seq[c % kBackSlots] = sig.seq;
        return launch_get(b.g, (uint32_t *)(at + (size_t)(c % kBackSlots) * kBackWords * 4), c * kBackWords,
                          std::min(kBackWords, words - c * kBackWords), sig, f->stream);
    };
    for (int64_t c = 0; c < std::min<int64_t>(pieces, kBackSlots); c++) HIP_TRY(ask(c));
    for (int64_t c = 0; c < pieces; c++) {
        if (int rc = link_wait_for(f, seq[c % kBackSlots])) return rc;
        const char *p = at + (size_t)(c % kBackSlots) * kBackWords * 4;
        b.each(c * kBackWords, std::min(kBackWords, words - c * kBackWords),
               [&](char *h, int64_t off, size_t bytes) { memcpy(h, p + off, bytes); });
        if (c + kBackSlots < pieces) HIP_TRY(ask(c + kBackSlots));
    }
    f->staging.idle();
    return OMK_OK;
}

// `words` 32-bit words of device memory (at most kLinkStaging bytes) to the host; waits for the stream: 8 us.
static int link_fetch(omk_forest *f, void *h_dst, const void *d_src, size_t words) {
    void *staged = nullptr;
    if (int rc = link_stage(f, words * 4, &staged)) return rc;
    HIP_TRY(launch_fetch((uint32_t *)staged, (const uint32_t *)d_src, (int64_t)words, link_signal(f), f->stream));
    if (int rc = link_wait(f)) return rc;
    memcpy(h_dst, staged, words * 4);
    return OMK_OK;
}

static int use_device(const omk_forest *f) {
    if (f->released) return fail(OMK_ERR_STATE, "the forest of this handle has been destroyed");
    HIP_TRY(hipSetDevice(f->device));
    (void)hipGetLastError();  // launches are checked with hipGetLastError: start from a clean slate
    return OMK_OK;
}

// Roots, paths and work items of a batch are node ids: stale once the forest was compacted or a
// different structure uploaded.
static int tree_only(const char *who, const omk_forest *f) {
    if (f->redirected)
        return fail(OMK_ERR_UNSUPPORTED,
                    "%s: child slots of this forest have been re-pointed at transpositions (omk_tt_select_redirect): "
                    "it is a graph until the next upload, and this operation needs a tree", who);
    return OMK_OK;
}

static int fresh_batch(const char *who, const omk_batch *b) {
    if (b->generation != b->f->generation)
        return fail(OMK_ERR_STATE, "%s: the forest was compacted or uploaded with another structure since this "
                    "batch's roots were set; call omk_batch_set_roots and select again", who);
    return OMK_OK;
}

extern "C" {

const char *omk_last_error(void) { return g_err; }
int omk_version(void) { return 1; }

int omk_forest_create(const omk_forest_desc *desc, omk_forest **out) {
    if (!desc || !out) return fail(OMK_ERR_INVALID, "omk_forest_create: null argument");
    if (desc->capacity_nodes <= 0 || desc->capacity_nodes > 0x7FFFFFF0ll)
        return fail(OMK_ERR_INVALID, "omk_forest_create: capacity_nodes %lld out of range",
                    (long long)desc->capacity_nodes);
    int count = 0;
    HIP_TRY(hipGetDeviceCount(&count));
    if (desc->device < 0 || desc->device >= count)
        return fail(OMK_ERR_INVALID, "omk_forest_create: device %d of %d", desc->device, count);
    omk_forest *f = new (std::nothrow) omk_forest();
    if (!f) return fail(OMK_ERR_INVALID, "out of host memory");
    f->device = desc->device;
    f->capacity = desc->capacity_nodes;
    f->has_rave = desc->has_rave != 0;
    hipError_t e = hipSetDevice(f->device);
    if (e == hipSuccess) e = hipStreamCreate(&f->own_stream);
    const int64_t n = f->capacity;
    if (e == hipSuccess) e = dalloc(&f->span, n);
    if (e == hipSuccess) e = dalloc(&f->N, n);
    if (e == hipSuccess) e = dalloc(&f->W, n);
    if (e == hipSuccess) e = dalloc(&f->P, n);
    if (e == hipSuccess) e = dalloc(&f->VL, n);
    if (e == hipSuccess && f->has_rave) e = dalloc(&f->rN, n);
    if (e == hipSuccess && f->has_rave) e = dalloc(&f->rW, n);
    if (e == hipSuccess && f->has_rave) e = dalloc(&f->Q2, n);
    if (e == hipSuccess) e = dalloc(&f->link_count, 64);
    if (e == hipSuccess) e = launch_fill_words(f->link_count, 0u, 64, f->own_stream);
    if (e == hipSuccess) e = link_alloc(f);
    if (e != hipSuccess) {
        int rc = fail(OMK_ERR_HIP, "omk_forest_create: %s", hipGetErrorString(e));
        omk_forest_destroy(f);
        return rc;
    }
    f->stream = f->own_stream;
    *out = f;
    return OMK_OK;
}

static void forest_free(omk_forest *f) {
    (void)hipSetDevice(f->device);
    if (f->own_stream) (void)hipStreamSynchronize(f->own_stream);
    void *ptrs[] = {f->span, f->N, f->W, f->P, f->VL, f->rN, f->rW, f->Q2, f->action, f->legal, f->hash, f->alias, f->link_count, f->scratch};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    if (f->link) (void)hipHostFree(f->link);
    if (f->own_stream) (void)hipStreamDestroy(f->own_stream);
    (void)hipGetLastError();
    delete f;
}

// Batches and tables point into their forest: the memory goes when the last of them has.
static void forest_child_gone(omk_forest *f) {
    if (--f->children == 0 && f->released) forest_free(f);
}

int omk_forest_destroy(omk_forest *f) {
    if (!f) return OMK_OK;
    if (f->released) return fail(OMK_ERR_STATE, "omk_forest_destroy: called twice");
    if (f->children > 0) {
        f->released = true;
        return OMK_OK;
    }
    forest_free(f);
    return OMK_OK;
}

int omk_forest_set_stream(omk_forest *f, void *hip_stream) {
    if (!f) return fail(OMK_ERR_INVALID, "omk_forest_set_stream: null forest");
    if (int rc = use_device(f)) return rc;
    HIP_TRY(hipStreamSynchronize(f->stream));
    f->stream = hip_stream ? (hipStream_t)hip_stream : f->own_stream;
    return OMK_OK;
}

int omk_forest_get_stream(omk_forest *f, void **hip_stream_out) {
    if (!f || !hip_stream_out) return fail(OMK_ERR_INVALID, "omk_forest_get_stream: null argument");
    *hip_stream_out = (void *)f->stream;
    return OMK_OK;
}

int omk_sync(omk_forest *f) {
    if (!f) return fail(OMK_ERR_INVALID, "omk_sync: null forest");
    if (int rc = use_device(f)) return rc;
    HIP_TRY(hipStreamSynchronize(f->stream));
    return OMK_OK;
}

// The selection kernels give every node to exactly one wavefront per batch; that is only
// correct when every node is the child of at most one parent, so it is checked here, on
// the host, before anything reaches the device (it also keeps every child range in
// bounds, which is what protects the kernels from wild reads).
static int find_fault(const omk_soa_view *v, int64_t n) {
    std::vector<uint8_t> is_child((size_t)n, 0);
    for (int64_t i = 0; i < n; i++) {
        int32_t cc = v->child_count[i];
        if (cc == 0) continue;
        int32_t cb = v->child_begin[i];
        if (cc < 0) return fail(OMK_ERR_STRUCTURE, "node %lld: child_count %d < 0", (long long)i, cc);
        if (cc > OMK_MAX_FANOUT)
            return fail(OMK_ERR_STRUCTURE, "node %lld: child_count %d exceeds OMK_MAX_FANOUT %d", (long long)i, cc,
                        OMK_MAX_FANOUT);
        if (cb < 0 || (int64_t)cb + cc > n)
            return fail(OMK_ERR_STRUCTURE, "node %lld: children [%d, %d) outside [0, %lld)", (long long)i, cb,
                        cb + cc, (long long)n);
        for (int32_t c = cb; c < cb + cc; c++) {
            if (c == i) return fail(OMK_ERR_STRUCTURE, "node %lld is its own child", (long long)i);
            if (is_child[(size_t)c]) return fail(OMK_ERR_STRUCTURE, "node %d has two parents", c);
            is_child[(size_t)c] = 1;
        }
    }
    return OMK_OK;
}

// Marks the bits [at, at + count) of `bits`; false when one was marked before.
static bool mark_range(uint64_t *bits, int64_t at, int32_t count) {
    uint64_t met = 0;
    for (int64_t w = at >> 6, end = (at + count + 63) >> 6; w < end; w++) {
        uint64_t m = ~0ull;
        if (w == at >> 6) m &= ~0ull << (at & 63);
        if (w == (at + count - 1) >> 6) m &= ~0ull >> (63 - ((at + count - 1) & 63));
        met |= bits[w] & m;
        bits[w] |= m;
    }
    return met == 0;
}

// The same test in one pass over the child counts, eight at a time (most nodes are leaves), and a bit per node for
// "is somebody's child"; a structure that fails it goes through find_fault for the message.  On the way: the widest
// fan-out, whether every node's children are stored by descending prior, and a checksum of the structure.
static int validate(const omk_soa_view *v, int64_t n, int *max_fanout, bool *prior_sorted, uint64_t *structure_sum) {
    std::vector<uint64_t> is_child((size_t)(n + 63) / 64, 0);
    int mf = 0;
    bool sorted = v->legal == nullptr;
    uint64_t h = 0xCBF29CE484222325ull ^ (uint64_t)n;  // of (node, child range) of every expanded node
    const int32_t *count = v->child_count;
    for (int64_t i = 0; i < n; i++) {
        while (i + 8 <= n && !(count[i] | count[i + 1] | count[i + 2] | count[i + 3] | count[i + 4] | count[i + 5] |
                               count[i + 6] | count[i + 7]))
            i += 8;
        if (i >= n) break;
        const int32_t cc = count[i];
        if (cc == 0) continue;
        const int32_t cb = v->child_begin[i];
        if (cc < 0 || cc > OMK_MAX_FANOUT || cb < 0 || (int64_t)cb + cc > n || (i >= cb && i < (int64_t)cb + cc) ||
            !mark_range(is_child.data(), cb, cc))
            return find_fault(v, n);
        if (sorted)
            for (int32_t c = cb + 1; c < cb + cc && sorted; c++) sorted = v->P[c - 1] >= v->P[c];
        mf = std::max(mf, (int)cc);
        h = (h ^ ((uint64_t)i * 0x9E3779B97F4A7C15ull + ((uint64_t)(uint32_t)cb << 32) + (uint32_t)cc)) * 0x100000001B3ull;
    }
    *max_fanout = mf;
    *prior_sorted = sorted;
    *structure_sum = h;
    return OMK_OK;
}

int omk_forest_upload(omk_forest *f, const omk_soa_view *v) try {
    if (!f || !v) return fail(OMK_ERR_INVALID, "omk_forest_upload: null argument");
    const int64_t n = v->n_nodes;
    if (n <= 0 || n > f->capacity)
        return fail(OMK_ERR_CAPACITY, "omk_forest_upload: %lld nodes, capacity %lld", (long long)n,
                    (long long)f->capacity);
    if (!v->N || !v->W || !v->P || !v->VL || !v->child_begin || !v->child_count)
        return fail(OMK_ERR_INVALID, "omk_forest_upload: N, W, P, VL, child_begin, child_count are required");
    if (f->has_rave && (!v->rN || !v->rW))
        return fail(OMK_ERR_INVALID, "omk_forest_upload: the forest was created with RAVE, rN and rW are required");
    int mf = 0;
    bool sorted = false;
    uint64_t ssum = 0;
    if (int rc = validate(v, n, &mf, &sorted, &ssum)) return rc;
    if (int rc = use_device(f)) return rc;

    hipStream_t s = f->stream;
    f->has_action = v->action != nullptr;
    if (f->has_action && !f->action) HIP_TRY(dalloc(&f->action, f->capacity));
    f->has_legal = v->legal != nullptr;
    if (f->has_legal && !f->legal) HIP_TRY(dalloc(&f->legal, (f->capacity + 31) / 32));
    f->has_hash = v->hash != nullptr;
    if (f->has_hash && !f->hash) HIP_TRY(dalloc(&f->hash, f->capacity));
    Bulk up;
    up.add(f->span, 2, v->child_begin, n);
    up.add((int32_t *)f->span + 1, 2, v->child_count, n);
    up.add(f->N, 1, v->N, n);
    up.add(f->W, 1, v->W, n);
    up.add(f->P, 1, v->P, n);
    up.add(f->VL, 1, v->VL, n);
    if (f->has_rave) {
        up.add(f->rN, 1, v->rN, n);
        up.add(f->rW, 1, v->rW, n);
    }
    if (f->has_action) up.add(f->action, 1, v->action, n);
    if (int rc = bulk_put(f, up)) return rc;
    if (f->has_legal || f->has_hash) {
        Bulk more;
        if (f->has_legal) more.add(f->legal, 1, v->legal, (n + 31) / 32);
        if (f->has_hash) more.add(f->hash, 1, v->hash, 2 * n);
        if (int rc = bulk_put(f, more)) return rc;
    }
    f->changes++;
    // the same structure again (statistics put back): node ids keep their meaning
    if (!f->uploaded || f->structure_changed || n != f->n_nodes || ssum != f->structure_sum) f->generation++;
    f->structure_sum = ssum;
    f->structure_changed = false;
    if (f->redirected) {  // an upload brings a tree: every slot holds its own node again
        HIP_TRY(launch_fill_words(f->alias, 0xFFFFFFFFu, f->capacity, f->stream));
        f->redirected = false;
    }
    f->n_nodes = n;
    f->max_fanout = mf;
    f->made_node.clear();
    f->made_count.clear();
    f->prior_sorted = sorted;
    f->uploaded = true;
    // the RAVE blend of every node from the new statistics, for the constant the selections have been using
    // (a first selection, or one with another constant, computes it itself)
    f->blend_valid = false;
    if (f->has_rave && f->blend_k_known) {
        HIP_TRY(launch_blend_all(f->dev(), f->blend_k, s));
        f->blend_valid = true;
    }
    return OMK_OK;
} OMK_NO_THROW

int omk_forest_download(omk_forest *f, omk_soa_view *v) {
    if (!f || !v) return fail(OMK_ERR_INVALID, "omk_forest_download: null argument");
    if (!f->uploaded) return fail(OMK_ERR_STATE, "omk_forest_download: nothing uploaded");
    if (v->n_nodes != f->n_nodes)
        return fail(OMK_ERR_INVALID, "omk_forest_download: view has %lld nodes, forest %lld", (long long)v->n_nodes,
                    (long long)f->n_nodes);
    if (int rc = use_device(f)) return rc;
    const int64_t n = f->n_nodes;
    Bulk down;
    down.add(f->N, 1, v->N, n);
    down.add(f->W, 1, v->W, n);
    down.add(f->P, 1, v->P, n);
    down.add(f->VL, 1, v->VL, n);
    if (f->has_rave) {
        down.add(f->rN, 1, v->rN, n);
        down.add(f->rW, 1, v->rW, n);
    }
    return bulk_get(f, down);
}

static inline bool view_legal(const omk_soa_view *v, int64_t i) {
    return !v->legal || ((v->legal[i >> 5] >> (i & 31)) & 1u);
}

int64_t omk_soa_count_legal(const omk_soa_view *v) {
    if (!v || v->n_nodes < 0) return fail(OMK_ERR_INVALID, "omk_soa_count_legal: null view");
    if (!v->legal) return v->n_nodes;
    int64_t c = 0;
    const int64_t words = v->n_nodes >> 5;
    for (int64_t w = 0; w < words; w++) c += __builtin_popcount(v->legal[w]);
    for (int64_t i = words << 5; i < v->n_nodes; i++) c += view_legal(v, i);
    return c;
}

int omk_soa_compact_legal(const omk_soa_view *v, int64_t count, int32_t *N, float *W, float *P, int32_t *VL,
                          int32_t *rN, float *rW, int32_t *child_begin, int32_t *child_count, int32_t *action,
                          uint64_t *hash, int32_t *old_to_new, int32_t *new_to_old) try {
    if (!v || !N || !W || !P || !VL || !child_begin || !child_count)
        return fail(OMK_ERR_INVALID, "omk_soa_compact_legal: N, W, P, VL, child_begin, child_count are required");
    const int64_t n = v->n_nodes;
    if (n <= 0 || !v->N || !v->W || !v->P || !v->VL || !v->child_begin || !v->child_count)
        return fail(OMK_ERR_INVALID, "omk_soa_compact_legal: the view has no nodes or lacks a required array");
    if ((rN && !v->rN) || (rW && !v->rW) || (hash && !v->hash))
        return fail(OMK_ERR_INVALID, "omk_soa_compact_legal: rN, rW or hash asked for, the view has none");
    // rank[i]: kept nodes before node i
    std::vector<int32_t> rank((size_t)n + 1);
    int64_t c = 0;
    for (int64_t i = 0; i < n; i++) {
        rank[(size_t)i] = (int32_t)c;
        c += view_legal(v, i);
    }
    rank[(size_t)n] = (int32_t)c;
    if (c != count)
        return fail(OMK_ERR_INVALID, "omk_soa_compact_legal: the view keeps %lld nodes, room for %lld was announced",
                    (long long)c, (long long)count);
    if (action && !v->action)
        for (int64_t j = 0; j < c; j++) action[j] = -1;
    for (int64_t i = 0; i < n; i++) {
        if (old_to_new) old_to_new[i] = view_legal(v, i) ? rank[(size_t)i] : -1;
        if (!view_legal(v, i)) continue;
        const int64_t j = rank[(size_t)i];
        N[j] = v->N[i];
        W[j] = v->W[i];
        P[j] = v->P[i];
        VL[j] = v->VL[i];
        if (rN) rN[j] = v->rN[i];
        if (rW) rW[j] = v->rW[i];
        if (hash) hash[j] = v->hash[i];
        if (new_to_old) new_to_old[j] = (int32_t)i;
        const int64_t cb = v->child_begin[i], cc = v->child_count[i];
        if (cc < 0 || cb < 0 || cb + cc > n)
            return fail(OMK_ERR_INVALID, "omk_soa_compact_legal: node %lld has the child range [%lld, +%lld)", (long long)i,
                        (long long)cb, (long long)cc);
        child_count[j] = cc > 0 ? rank[(size_t)(cb + cc)] - rank[(size_t)cb] : 0;
        child_begin[j] = child_count[j] > 0 ? rank[(size_t)cb] : 0;
        if (action) {
            if (v->action) action[j] = v->action[i];
            else
                for (int64_t q = cb; q < cb + cc; q++)
                    if (view_legal(v, q)) action[rank[(size_t)q]] = (int32_t)(q - cb);
        }
    }
    return OMK_OK;
} OMK_NO_THROW

int omk_forest_download_structure(omk_forest *f, int64_t n_nodes, int32_t *h_child_begin, int32_t *h_child_count,
                                  int32_t *h_action) {
    if (!f) return fail(OMK_ERR_INVALID, "omk_forest_download_structure: null forest");
    if (!f->uploaded) return fail(OMK_ERR_STATE, "omk_forest_download_structure: nothing uploaded");
    if (n_nodes != f->n_nodes)
        return fail(OMK_ERR_INVALID, "omk_forest_download_structure: room for %lld nodes, forest has %lld",
                    (long long)n_nodes, (long long)f->n_nodes);
    if (int rc = use_device(f)) return rc;
    Bulk down;
    down.add(f->span, 2, h_child_begin, n_nodes);
    down.add((int32_t *)f->span + 1, 2, h_child_count, n_nodes);
    if (f->has_action) down.add(f->action, 1, h_action, n_nodes);
    if (int rc = bulk_get(f, down)) return rc;
    if (h_action && !f->has_action)
        for (int64_t i = 0; i < n_nodes; i++) h_action[i] = (int32_t)i;
    return OMK_OK;
}

int omk_forest_set_keys(omk_forest *f, const int32_t *h_nodes, const uint64_t *h_keys, int64_t n) {
    if (!f || (n > 0 && (!h_nodes || !h_keys))) return fail(OMK_ERR_INVALID, "omk_forest_set_keys: null argument");
    if (!f->uploaded) return fail(OMK_ERR_STATE, "omk_forest_set_keys: nothing uploaded");
    if (n < 0) return fail(OMK_ERR_INVALID, "omk_forest_set_keys: n = %lld", (long long)n);
    if (int rc = use_device(f)) return rc;
    hipStream_t s = f->stream;
    if (!f->has_hash) {
        // a forest that came without position keys: every node starts with "no key"
        if (!f->hash) HIP_TRY(dalloc(&f->hash, f->capacity));
        HIP_TRY(launch_fill_words(f->hash, 0xFFFFFFFFu, f->capacity * 2, s));
        f->has_hash = true;
    }
    if (n == 0) return OMK_OK;
    int64_t bad = 0;
    for (int64_t i = 0; i < n; i++) bad += h_nodes[i] < 0 || h_nodes[i] >= f->n_nodes;
    const int64_t most = (size_t)n * 12 <= kLinkStaging ? n : (int64_t)kLinkPiece / 12;
    for (int64_t at = 0; at < n; at += most) {
        const int64_t m = std::min(most, n - at);
        void *staged = nullptr;
        if (int rc = link_stage(f, (size_t)m * 12, &staged)) return rc;
        uint64_t *keys = (uint64_t *)staged;
        int32_t *nodes = (int32_t *)(keys + m);
        memcpy(keys, h_keys + at, (size_t)m * 8);
        memcpy(nodes, h_nodes + at, (size_t)m * 4);
        HIP_TRY(launch_set_keys(f->hash, nodes, keys, m, f->n_nodes, s));
    }
    if (bad) return fail(OMK_ERR_INVALID, "omk_forest_set_keys: %lld node ids outside the forest (skipped)", (long long)bad);
    return OMK_OK;
}

}  // extern "C"

// What the host asks about a node's children, in pinned memory until the next call that stages something: one
// kernel and one wait (8 us) where every array was a synchronous copy of its own (42 us a call, and a self-play
// program asks for every game).
struct RootChildren {
    int32_t begin, count;
    const int32_t *visits, *action, *legal;  // visits: of the node the slot holds
};

static int root_children(omk_forest *f, int32_t root, RootChildren *out) {
    void *staged = nullptr;
    if (int rc = link_stage(f, 128 + 12ull * OMK_MAX_FANOUT, &staged)) return rc;
    int32_t *r = (int32_t *)staged;
    HIP_TRY(launch_root_children(f->dev(), f->redirected ? f->alias : nullptr, root, r, r + 32, OMK_MAX_FANOUT,
                                 link_signal(f), f->stream));
    if (int rc = link_wait(f)) return rc;
    out->begin = r[0];
    out->count = r[1];
    out->visits = r + 32;
    out->action = r + 32 + OMK_MAX_FANOUT;
    out->legal = r + 32 + 2 * OMK_MAX_FANOUT;
    return OMK_OK;
}

extern "C" {

int omk_forest_add_root_noise(omk_forest *f, int32_t root, const float *h_gamma, int32_t n_gamma, float epsilon) {
    if (!f || !h_gamma) return fail(OMK_ERR_INVALID, "omk_forest_add_root_noise: null argument");
    if (!f->uploaded) return fail(OMK_ERR_STATE, "omk_forest_add_root_noise: nothing uploaded");
    if (root < 0 || root >= f->n_nodes) return fail(OMK_ERR_INVALID, "omk_forest_add_root_noise: root %d", root);
    if (int rc = tree_only("omk_forest_add_root_noise", f)) return rc;
    if (int rc = use_device(f)) return rc;
    // A root that the expansion before this call gave its children (a self-play program expands its roots and then
    // adds the noise, game by game): their number is known here, and nothing has to be waited for (11 -> 4 us a
    // root).  The list is short for a program's roots; of a long one only the head is searched.
    int32_t known = -1;
    const size_t made = std::min<size_t>(f->made_node.size(), 4096);
    for (size_t i = 0; i < made && known < 0; i++)
        if (f->made_node[i] == root) known = f->made_count[i];
    if (known > 0 && n_gamma != known)
        return fail(OMK_ERR_INVALID, "omk_forest_add_root_noise: %d samples for %d children", n_gamma, known);
    // MCTSEngine::addDirichletNoise from the normalisation on, statement by statement; the mix is the kernel's,
    // child by child in the same arithmetic, and happens only if the samples are as many as the children
    const int32_t given = std::max(0, std::min(n_gamma, (int32_t)OMK_MAX_FANOUT));
    void *staged = nullptr;
    if (int rc = link_stage(f, 128 + (size_t)given * 4, &staged)) return rc;
    int32_t *result = (int32_t *)staged;
    float *noise = (float *)staged + 32;
    float sum = 0.0f;
    for (int32_t j = 0; j < given; j++) sum = sum + h_gamma[j];
    const float uniform_noise = 1.0f / (float)std::max(given, 1);
    for (int32_t j = 0; j < given; j++) noise[j] = sum > 0.0f ? h_gamma[j] / sum : uniform_noise;
    HostSignal sig = {nullptr, nullptr, 0};
    if (known < 0) sig = link_signal(f);
    HIP_TRY(launch_root_noise(f->mut(), root, noise, n_gamma, epsilon, result, sig, f->stream));
    if (known >= 0) return OMK_OK;
    if (int rc = link_wait(f)) return rc;
    const int32_t children = result[0];
    if (children > 0 && n_gamma != children)
        return fail(OMK_ERR_INVALID, "omk_forest_add_root_noise: %d samples for %d children", n_gamma, children);
    return OMK_OK;
}

int omk_forest_action_probabilities(omk_forest *f, int32_t root, float temperature, int32_t action_space,
                                    float *h_probabilities, int32_t *h_children) {
    if (!f || !h_probabilities) return fail(OMK_ERR_INVALID, "omk_forest_action_probabilities: null argument");
    if (!f->uploaded) return fail(OMK_ERR_STATE, "omk_forest_action_probabilities: nothing uploaded");
    if (root < 0 || root >= f->n_nodes || action_space <= 0)
        return fail(OMK_ERR_INVALID, "omk_forest_action_probabilities: root %d, action space %d", root, action_space);
    if (int rc = use_device(f)) return rc;
    RootChildren kids;
    if (int rc = root_children(f, root, &kids)) return rc;
    for (int32_t a = 0; a < action_space; a++) h_probabilities[a] = 0.0f;
    if (h_children) *h_children = 0;
    // the counts are those of the nodes the children vector holds (child->getVisitCount(),
    // mcts_engine_tree.cpp:401-403), the actions those of the slots (root->getActions(), :395)
    const int32_t cc = kids.count, *n = kids.visits, *act = kids.action;
    auto is_child = [&](int32_t i) { return kids.legal[i] != 0; };
    // MCTSEngine::getActionProbabilities, statement by statement
    int32_t children = 0, max_idx = -1;
    float max_count = 0.0f;
    for (int32_t i = 0; i < cc; i++) {
        if (!is_child(i)) continue;
        children++;
        const float c = (float)n[i];
        if (max_idx < 0 || c > max_count) {  // std::max_element: the first of the largest
            max_count = c;
            max_idx = i;
        }
    }
    if (h_children) *h_children = children;
    if (children == 0) return OMK_OK;
    const bool near_zero = temperature < 0.01f;
    float sum = 0.0f, scaled[OMK_MAX_FANOUT];
    if (!near_zero && max_count > 0.0f)
        for (int32_t i = 0; i < cc; i++) {
            if (!is_child(i)) continue;
            const float c = (float)n[i];
            scaled[i] = 0.0f;
            if (c > 0.0f) scaled[i] = powf(c / max_count, 1.0f / temperature);
            sum += scaled[i];
        }
    for (int32_t i = 0; i < cc; i++) {
        if (!is_child(i)) continue;
        float prob;
        if (near_zero) {
            prob = i == max_idx ? 1.0f : 0.0f;
        } else if (max_count <= 0.0f || !(sum > 0.0f)) {
            prob = 1.0f / (float)children;
        } else {
            prob = scaled[i] / sum;
        }
        const int32_t a = act[i];
        if (a >= 0 && a < action_space) h_probabilities[a] = prob;
    }
    return OMK_OK;
}

int omk_forest_reroot_child(omk_forest *f, int32_t root, int32_t last_action, int32_t *h_child) {
    if (!f || !h_child) return fail(OMK_ERR_INVALID, "omk_forest_reroot_child: null argument");
    if (!f->uploaded) return fail(OMK_ERR_STATE, "omk_forest_reroot_child: nothing uploaded");
    if (root < 0 || root >= f->n_nodes) return fail(OMK_ERR_INVALID, "omk_forest_reroot_child: root %d", root);
    *h_child = -1;
    if (last_action < 0) return OMK_OK;
    if (int rc = use_device(f)) return rc;
    RootChildren kids;
    if (int rc = root_children(f, root, &kids)) return rc;
    for (int32_t i = 0; i < kids.count; i++)
        if (kids.legal[i] && kids.action[i] == last_action) {
            *h_child = kids.begin + i;
            break;
        }
    return OMK_OK;
}

}  // extern "C"

// Device memory a compaction works in, beyond the forest's own arrays.
struct CompactScratch {
    int32_t *map = nullptr;       // [n] old id of every new node
    int32_t *begin = nullptr;     // [n] new id of every new node's first child
    uint32_t *tmp = nullptr;      // the arrays pass through here, as many at a time as fit
    int64_t tmp_words = 0;
    int32_t *sums = nullptr;      // [kBfsSums]
    BfsLevel *levels = nullptr;   // [kCompactLevels + 1]
};
constexpr int kBfsLevels = 12;        // levels enqueued before the host looks
constexpr int kCompactLevels = 4104;  // more levels than a path has nodes are walked in turns of this many
constexpr size_t kCompactFixed = 1024 + ((kCompactLevels + 1) * sizeof(BfsLevel) + 255) / 256 * 256;

// The compaction itself, in scratch memory the caller provides (room for the forest's node count).
static int compact_in(omk_forest *f, int32_t new_root, int64_t *h_nodes_after, int32_t *h_old_of_new,
                      const CompactScratch &sc) {
    hipStream_t s = f->stream;
    const int64_t n = f->n_nodes;
    HIP_TRY(launch_bfs_start(sc.map, sc.levels, new_root, s));
    int64_t k = 1;
    for (int level = 0;;) {
        HIP_TRY(launch_bfs(f->span, sc.map, sc.begin, sc.levels, level, kBfsLevels, sc.sums, n, s));
        level += kBfsLevels;
        BfsLevel reached;
        if (int rc = link_fetch(f, &reached, sc.levels + level, sizeof(BfsLevel) / 4)) return rc;
        if (reached.cnt < 0)
            return fail(OMK_ERR_STRUCTURE, "omk_forest_compact: the child ranges do not form a tree");
        k = reached.lo;
        if (reached.cnt == 0) break;
        if (level + kBfsLevels > kCompactLevels) {  // go on from the front of the table
            HIP_TRY(launch_copy_words(sc.levels, sc.levels + level, sizeof(BfsLevel) / 4, s));
            level = 0;
        }
    }
    struct {
        void *array;
        int kind;
    } fields[] = {{f->N, 1}, {f->W, 1}, {f->P, 1}, {f->VL, 1}, {f->has_rave ? f->rN : nullptr, 1},
                  {f->has_rave ? f->rW : nullptr, 1},
                  {f->has_rave ? f->Q2 : nullptr, 1},  // the nodes keep their statistics, hence their RAVE blend
                  {f->has_action ? f->action : nullptr, 1}, {f->has_hash ? f->hash : nullptr, 2}, {f->span, 3}};
    CompactFields g = {};
    int64_t used = 0;
    // (a 64-bit array starts at an even word of tmp: after an odd number of arrays of an odd count, in a pass of its own)
    auto move = [&]() -> int {
        if (g.n) HIP_TRY(launch_compact(g, sc.tmp, sc.map, sc.begin, k, s));
        g.n = 0;
        used = 0;
        return OMK_OK;
    };
    for (const auto &fd : fields) {
        if (!fd.array) continue;
        if (used + compact_words(fd.kind, k) > sc.tmp_words || (fd.kind != 1 && (used & 1)))
            if (int rc = move()) return rc;
        g.array[g.n] = (uint32_t *)fd.array;
        g.kind[g.n++] = fd.kind;
        used += compact_words(fd.kind, k);
    }
    if (int rc = move()) return rc;
    if (f->has_legal) {
        HIP_TRY(launch_gather_legal(sc.tmp, f->legal, sc.map, k, s));
        HIP_TRY(launch_copy_words(f->legal, sc.tmp, (k + 31) / 32, s));
    }
    if (h_old_of_new) {
        Bulk down;
        down.add(sc.map, 1, h_old_of_new, k);
        if (int rc = bulk_get(f, down)) return rc;
    }
    f->n_nodes = k;
    f->made_node.clear();
    f->made_count.clear();
    f->changes++;
    f->generation++;
    f->structure_changed = true;
    if (h_nodes_after) *h_nodes_after = k;
    return OMK_OK;
}

// Scratch of up to this much stays with the forest from one move to the next; more is given back after the call.
constexpr size_t kKeepScratch = 64 << 20;

// Words of CompactScratch::tmp for a forest of n nodes: every array at once (eight of 32-bit words and two of 64-bit
// ones) as long as that stays within kKeepScratch, at least one 64-bit array.  A large tree passes through in more
// rounds of two launches, which its nodes outweigh (12 M nodes: 9.5 ms, with every array at once 9.6), and takes at
// most 24 bytes a node.
constexpr int64_t compact_tmp_words(int64_t n) {
    const int64_t kept = ((int64_t)kKeepScratch - (int64_t)kCompactFixed - 8 * (n + 63)) / 4;
    return std::max(2 * n, std::min(12 * n, kept));
}
constexpr size_t compact_bytes(int64_t n) {
    return kCompactFixed + ((size_t)n + 63) / 64 * 64 * 8 + (size_t)compact_tmp_words(n) * 4;
}
static_assert(compact_tmp_words(1 << 20) == 12 << 20, "a tree of a million nodes moves at once");
static_assert(compact_bytes(1500000) <= kKeepScratch && compact_bytes(4000000) <= kKeepScratch, "kept");
static_assert(compact_bytes(1 << 24) <= 24ull << 24 && compact_bytes(0x7FFFFFF0) <= 24ull * 0x7FFFFFF0, "24 bytes a node");

extern "C" {

int omk_forest_compact(omk_forest *f, int32_t new_root, int64_t *h_nodes_after, int32_t *h_old_of_new) {
    if (!f) return fail(OMK_ERR_INVALID, "omk_forest_compact: null forest");
    if (!f->uploaded) return fail(OMK_ERR_STATE, "omk_forest_compact: nothing uploaded");
    if (new_root < 0 || new_root >= f->n_nodes) return fail(OMK_ERR_INVALID, "omk_forest_compact: root %d", new_root);
    if (int rc = tree_only("omk_forest_compact", f)) return rc;
    if (int rc = use_device(f)) return rc;
    const int64_t n = f->n_nodes;
    CompactScratch sc;
    sc.tmp_words = compact_tmp_words(n);
    const size_t words = ((size_t)n + 63) / 64 * 64, bytes = compact_bytes(n);
    if (bytes > f->scratch_bytes) {
        if (f->scratch) {
            HIP_TRY(hipStreamSynchronize(f->stream));
            HIP_TRY(hipFree(f->scratch));
        }
        f->scratch = nullptr;
        f->scratch_bytes = 0;
        HIP_TRY(hipMalloc((void **)&f->scratch, bytes));
        f->scratch_bytes = bytes;
    }
    sc.sums = (int32_t *)f->scratch;
    sc.levels = (BfsLevel *)(f->scratch + 1024);
    sc.map = (int32_t *)(f->scratch + kCompactFixed);
    sc.begin = sc.map + words;
    sc.tmp = (uint32_t *)(sc.begin + words);
    const int rc = compact_in(f, new_root, h_nodes_after, h_old_of_new, sc);
    if (rc != OMK_OK || f->scratch_bytes > kKeepScratch) {
        (void)hipStreamSynchronize(f->stream);
        (void)hipFree(f->scratch);
        f->scratch = nullptr;
        f->scratch_bytes = 0;
    }
    return rc;
}

// ---- the same compaction for callers that cannot allocate ----
//
// All the scratch memory of a compaction of up to kStaticCompactNodes nodes, laid out in one
// file-scope device array: every GPU the library runs on holds its own copy for the life of the
// process.  In host code the array's name is only a handle for hipGetSymbolAddress; the address the
// kernels get is looked up once per device (static_scratch) and kept.
constexpr int64_t kStaticCompactNodes = 1ll << 20;
constexpr size_t kStaticWords = (size_t)kStaticCompactNodes * 4;
constexpr size_t kStaticOffMap = kCompactFixed;
constexpr size_t kStaticOffBegin = kStaticOffMap + kStaticWords;
constexpr size_t kStaticOffTmp = kStaticOffBegin + kStaticWords;
constexpr size_t kStaticTmpWords = 4 * (size_t)kStaticCompactNodes;  // four arrays of 32-bit words at a time
constexpr size_t kStaticScratchBytes = kStaticOffTmp + kStaticTmpWords * 4;
static_assert(kStaticOffMap % 256 == 0, "parts of the scratch keep its alignment");

static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mutex;
static unsigned char *g_scratch_ptr[kMaxDevices];  // device address of `scratch` on every device, once known

// The device address of the scratch array on the forest's device (which must be current).
static int static_scratch(int device, unsigned char **out) {
    if (device < 0 || device >= kMaxDevices) return fail(OMK_ERR_INVALID, "device %d: at most %d devices", device, kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[device]) {
        void *p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(OMK_ERR_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", device, hipGetErrorString(e));
        g_scratch_ptr[device] = (unsigned char *)p;
    }
    *out = g_scratch_ptr[device];
    return OMK_OK;
}

int omk_forest_compact_static(omk_forest *f, int32_t new_root, int64_t *h_nodes_after, int32_t *h_old_of_new) {
    if (!f) return fail(OMK_ERR_INVALID, "omk_forest_compact_static: null forest");
    if (!f->uploaded) return fail(OMK_ERR_STATE, "omk_forest_compact_static: nothing uploaded");
    if (new_root < 0 || new_root >= f->n_nodes)
        return fail(OMK_ERR_INVALID, "omk_forest_compact_static: root %d", new_root);
    if (int rc = tree_only("omk_forest_compact_static", f)) return rc;
    if (f->n_nodes > kStaticCompactNodes)
        return fail(OMK_ERR_CAPACITY,
                    "omk_forest_compact_static: the forest holds %lld nodes, the static scratch memory serves at most "
                    "%lld; use omk_forest_compact",
                    (long long)f->n_nodes, (long long)kStaticCompactNodes);
    if (int rc = use_device(f)) return rc;
    unsigned char *base = nullptr;
    if (int rc = static_scratch(f->device, &base)) return rc;
    CompactScratch sc;
    // every part is written by this call before it is read (the order map and the levels from the root on, the sums
    // per level, the staging array per pass): nothing has to start at zero
    sc.sums = (int32_t *)base;
    sc.levels = (BfsLevel *)(base + 1024);
    sc.map = (int32_t *)(base + kStaticOffMap);
    sc.begin = (int32_t *)(base + kStaticOffBegin);
    sc.tmp = (uint32_t *)(base + kStaticOffTmp);
    sc.tmp_words = (int64_t)kStaticTmpWords;
    const int rc = compact_in(f, new_root, h_nodes_after, h_old_of_new, sc);
    // (the array is the next call's, perhaps of another forest on another stream: this one's kernels have to be done)
    HIP_TRY(hipStreamSynchronize(f->stream));
    return rc;
}

int omk_forest_node_count(omk_forest *f, int64_t *h_nodes, int64_t *h_capacity) {
    if (!f) return fail(OMK_ERR_INVALID, "omk_forest_node_count: null forest");
    if (h_nodes) *h_nodes = f->n_nodes;
    if (h_capacity) *h_capacity = f->capacity;
    return OMK_OK;
}

// ---------------------------------------------------------------- batch

}  // extern "C"

// 32-bit words of the leaf gather of n traversals: lengths | leaves | their child counts | their visit counts | abort
// words | paths and actions, if they are asked for
static size_t gather_words(size_t n, size_t depth, bool paths, bool actions) {
    return n * (4 + (paths ? depth + 1 : 0) + (actions ? depth : 0)) + 4;
}
static ExportOut gather_layout(int32_t *at, size_t n, size_t depth, bool paths, bool actions) {
    ExportOut o = {};
    o.len = at;
    o.leaf = o.len + n;
    o.children = o.leaf + n;
    o.visits = o.children + n;
    o.abort = o.visits + n;
    int32_t *rows = o.abort + 4;
    if (paths) o.paths = rows;
    if (actions) o.actions = rows + (paths ? n * (depth + 1) : 0);
    return o;
}
// Pinned memory of a batch for its gather, at most: a larger gather crosses in pieces.
// (Allocated with the batch, 20 us: the first step of a batch of 256 took 65 us when its read had to do that, and 43
// so, the later ones 37.)
constexpr size_t kGatherBytes = 16 << 20;

extern "C" {

int omk_batch_create(omk_forest *f, int32_t max_traversals, int32_t max_depth, omk_batch **out) {
    if (!f || !out) return fail(OMK_ERR_INVALID, "omk_batch_create: null argument");
    if (max_traversals <= 0 || max_traversals > (1 << 24))
        return fail(OMK_ERR_INVALID, "omk_batch_create: max_traversals %d out of range", max_traversals);
    if (max_depth <= 0 || max_depth > 4096)
        return fail(OMK_ERR_INVALID, "omk_batch_create: max_depth %d out of range", max_depth);
    if ((int64_t)max_traversals * (max_depth + 1) > (1ll << 28))
        return fail(OMK_ERR_CAPACITY, "omk_batch_create: max_traversals x (max_depth+1) = %lld exceeds 2^28",
                    (long long)max_traversals * (max_depth + 1));
    if (int rc = use_device(f)) return rc;
    omk_batch *b = new (std::nothrow) omk_batch();
    if (!b) return fail(OMK_ERR_INVALID, "out of host memory");
    b->f = f;
    f->children++;
    b->max_traversals = max_traversals;
    b->max_depth = max_depth;
    b->stride = (max_traversals + 63) & ~63;
    const int64_t B = b->stride;
    hipError_t e = dalloc(&b->paths, B * (max_depth + 1));
    if (e == hipSuccess) e = dalloc(&b->path_len, B);
    if (e == hipSuccess) e = dalloc(&b->leaf, B);
    if (e == hipSuccess) e = dalloc(&b->values, B);
    if (e == hipSuccess) e = dalloc(&b->items0, B);
    // a multi-visitor item has at least two visitors, and a level holds each visitor once; a heavy
    // node (kHeavyMin visitors or more) adds at most 63 slice items
    // (and as many parts of its partition, and as many boundaries worked out ahead of time)
    b->q_cap = (int32_t)((B + 64) * (max_depth + 1));
    // (a node whose boundaries are worked out ahead of time, and that is then not cut into slices after all, uses
    // a second context for its partition)
    b->hctx_cap = (int32_t)std::min<int64_t>(4096, 2 * (B / kHeavyMin) * (max_depth + 1));
    if (e == hipSuccess) e = dalloc(&b->hctx, (int64_t)b->hctx_cap * kHeavyCtxInts);
    // (a context says by the number of the select call that its children's contexts are listed: memory that an
    // earlier batch left behind would say so for this batch's first calls, whose numbers start again at 1)
    if (e == hipSuccess)
        e = hipMemset(b->hctx, 0, (size_t)std::max<int64_t>((int64_t)b->hctx_cap * kHeavyCtxInts, 1) * 4);
    if (e == hipSuccess) e = dalloc(&b->hbound, (int64_t)b->hctx_cap * kMaxSlices * kBoundInts);
    if (e == hipSuccess)
        e = hipMemset(b->hbound, 0, (size_t)std::max<int64_t>((int64_t)b->hctx_cap * kMaxSlices * kBoundInts, 1) * 4);
    if (e == hipSuccess) e = dalloc(&b->list_flag, B);
    if (e == hipSuccess) e = dalloc(&b->items_q, b->q_cap);
    if (e == hipSuccess) e = dalloc(&b->q_ready, b->q_cap);
    if (e == hipSuccess) e = hipMemset(b->q_ready, 0, (size_t)std::max(b->q_cap, 1) * 4);
    if (e == hipSuccess) e = dalloc(&b->singles0, B);
    if (e == hipSuccess) e = dalloc(&b->singles_q, B);
    if (e == hipSuccess) e = dalloc(&b->seg0, B);
    if (e == hipSuccess) e = dalloc(&b->seg[0], B);
    if (e == hipSuccess) e = dalloc(&b->seg[1], B);
    if (e == hipSuccess) e = dalloc(&b->sc_child, 2 * B);  // two halves, alternating with the depth
    if (e == hipSuccess) e = dalloc(&b->sc_occ, 2 * B);
    if (e == hipSuccess) e = dalloc(&b->counters, 5 * kSchedStep);
    if (e == hipSuccess) e = hipMemset(b->counters, 0, 5 * kSchedStep * 4);
    if (e == hipSuccess) e = dalloc(&b->single_ready, max_traversals);
    if (e == hipSuccess) e = hipMemset(b->single_ready, 0, (size_t)std::max(max_traversals, 1) * 4);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&b->n_cus, hipDeviceAttributeMultiprocessorCount, f->device);
    if (e == hipSuccess) e = hipMemset(b->values, 0, (size_t)B * 4);
    b->out_bytes = std::min(kGatherBytes, gather_words((size_t)B, (size_t)max_depth, true, true) * 4);
    if (e == hipSuccess) e = hipHostMalloc((void **)&b->out, b->out_bytes, hipHostMallocDefault);
    if (e != hipSuccess) {
        int rc = fail(OMK_ERR_HIP, "omk_batch_create: %s", hipGetErrorString(e));
        omk_batch_destroy(b);
        return rc;
    }
    *out = b;
    return OMK_OK;
}

int omk_batch_destroy(omk_batch *b) {
    if (!b) return OMK_OK;
    (void)hipSetDevice(b->f->device);
    (void)hipStreamSynchronize(b->f->stream);
    void *ptrs[] = {b->paths,  b->path_len, b->leaf,     b->values, b->items0,   b->items_q,  b->seg0,
                    b->seg[0], b->seg[1],   b->sc_child, b->sc_occ, b->counters, b->trace,
                    b->singles0, b->singles_q, b->q_ready, b->hctx, b->hbound, b->list_flag, b->single_ready};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    if (b->out) (void)hipHostFree(b->out);
    (void)hipGetLastError();
    forest_child_gone(b->f);
    delete b;
    return OMK_OK;
}

}  // extern "C"

// A selection whose traversals are all alone at their roots, or few at each, in a batch whose selection before was read:
// its walkers or blocks send their own rows (export_lone, k_select_blocks), and the read finds them there.  (Not in a
// batch that nobody has read yet: its evaluator may be on the card, the selection part of a captured graph; the first
// read makes one launch more.)  Small batches only.  A walker's row crosses the host link in pieces of its own, a kernel's in neighbouring lines, and
// from some number of rows on that costs more than the launch saves; a path that a whole block walks ends with
// wavefronts to spare for it.  A step with a read, us, rows by the walkers and by the kernel:
//   walked by a block (a legal mask, more than 64 slots), 225 slots: 64 traversals 20.9 / 24.2, 256 25.9 / 27.4,
//   350 29.7 / 27.7, 1024 39.8 / 33.6; 362 slots: 256 28.5 / 28.0 (in larger trees 31.0 / 31.6), 1024 54.5 / 38.7;
//   walked by a wavefront, 225 slots re-laid: 64 22.4 / 24.0, 128 25.5 / 24.6, 256 29.2 / 26.7, 1024 50.3 / 33.0;
//   chess-like: 64 23.4 / 25.2, 128 25.7 / 26.2, 200 29.7 / 28.0, 1024 53.4 / 38.5
// A batch of few visitors a root (omk_select_blocks.h) sends a root's rows together.  What costs there is a line of the
// host's memory that blocks on several XCDs write parts of: the rows of 2 to 8 roots whose traversals alternate, and of
// many roots with less than 8 visitors each, are the kernel's.  A read of traversals on 225 slots, us, rows by the
// blocks and by the kernel: 1 root x 64 53 / 53; 2 x 32 with the roots in order 37.2 / 38.8, alternating
// 53.4 / 39.2; 8 x 32 49.6 / 53.1 and 62.6 / 53.4; 16 x 32 55.2 / 59.2 and 53.8 / 58.8; steps of 64 x 16 54.8 / 62.1,
// 64 x 64 107 / 131, of 256 x 4 46.2 / 45.7, 512 x 2 56 / 48, 1024 x 2 92 / 71.
constexpr int kLoneRowsBlock = 256, kLoneRowsWave = 128, kBlockRows = 4096;
constexpr int kBlockRowsRoots = 16, kBlockRowsVisitors = 8;
static int lone_rows(omk_batch *b, LoneOut *out) {
    memset(out, 0, sizeof(*out));
    const int roots = b->n_items0 + b->n_singles0;
    const bool whole_lines = roots == 1 || (b->n >= kBlockRowsVisitors * roots && (b->in_order || roots >= kBlockRowsRoots));
    int most = b->f->has_legal && b->f->max_fanout > 64 ? kLoneRowsBlock : kLoneRowsWave;
    if (b->n_items0 > 0)
        most = by_blocks(b->n_items0, b->most_visitors, b->f->max_fanout) && whole_lines ? kBlockRows : 0;
    if (b->n > most || b->max_depth >= 64 || b->read_call != b->select_calls) return OMK_OK;
    static_assert((kBlockRows * (2 * 63 + 5) + 4) * 4 <= kGatherBytes, "the rows fit the batch's pinned buffer");
    out->rows = gather_layout(b->out, (size_t)b->n, (size_t)b->max_depth, true, true);
    for (int i = 0; i < 4; i++) out->rows.abort[i] = 0;  // (these kernels wait for nobody)
    out->sig = link_signal(b->f);
    b->lone_changes = b->f->changes;
    b->lone_seq = out->sig.seq;
    b->lone_staged = b->f->staging.now();
    return OMK_OK;
}

// What a selection of the batch with call number `epoch` is told, the caller's parameters apart.
static SelectArgs select_args(omk_batch *b, int32_t epoch) {
    SelectArgs a;
    memset(&a, 0, sizeof(a));
    a.items0 = b->items0;
    a.seg0 = b->seg0;
    a.items_q = b->items_q;
    a.seg[0] = b->seg[0];
    a.seg[1] = b->seg[1];
    a.q_ready = b->q_ready;
    a.q_cap = b->q_cap;
    a.epoch = epoch;
    a.spin_limit = b->spin_limit;
    a.truncated = b->counters + kTruncatedWord + (epoch & 1);
    a.truncated_next = b->counters + kTruncatedWord + ((epoch + 1) & 1);
    a.stats = b->stats_on ? b->counters + 1 : nullptr;
    a.n_singles = b->counters + 17;
    a.sched_head = b->counters + 1 * kSchedStep;
    a.sched_tail = b->counters + 2 * kSchedStep;
    a.sched_wait = b->counters + 3 * kSchedStep;
    a.singles_head = b->counters + 4 * kSchedStep;
    a.single_ready = b->single_ready;
    a.n_trav = b->n;
    a.n_team_blocks = 0;
    a.fast_singles = 0;
    // A waiting wavefront sleeps about a microsecond between two polls, so that hundreds of them leave the memory
    // system to those that work.  A small batch has few wavefronts waiting and a short chain of crowded nodes, every
    // hand-over of which pays that sleep: they poll without it (measured on 64 traversals: 0.095 -> 0.092 ms; on
    // 4096, with the sleep off: 0.216 -> 0.221).
    a.poll_sleep = b->n <= 256 ? 0 : b->poll_sleep;
    a.hctx = b->hctx;
    a.hbound = b->hbound;
    a.hctx_n = b->counters + 2 * kSchedStep + 64;
    a.hctx_cap = b->hctx_cap;
    a.list_flag = b->list_flag;
    static_assert(kHeavyCtxInts >= 16 + OMK_MAX_FANOUT, "context too small");
    a.times = b->counters + 26;
    a.trace = b->trace_on ? b->trace : nullptr;
    a.trace_n = b->counters + 24;
    a.trace_cap = kTraceCap;
    a.singles0 = b->singles0;
    a.singles_q = b->singles_q;
    a.sc_child = b->sc_child;
    a.sc_occ = b->sc_occ;
    a.paths = b->paths;
    a.path_len = b->path_len;
    a.leaf = b->leaf;
    a.stride = b->stride;
    a.max_depth = b->max_depth;
    return a;
}

// The traversals in ascending order of their roots, those of one root in ascending order: what a stable sort
// gives.  One root for all, and roots that ascend already (one traversal per tree), are in order as they are; else
// a radix sort, eleven bits a pass, as many passes as the largest root has digits.
// Returns whether they ascend already.
static bool order_by_root(const int32_t *roots, int32_t n, std::vector<int32_t> &order, std::vector<int32_t> &tmp) {
    order.resize((size_t)n);
    bool ascending = true;
    int32_t top = 0;
    for (int32_t t = 0; t < n; t++) {
        order[(size_t)t] = t;
        ascending &= t == 0 || roots[t - 1] <= roots[t];
        top = std::max(top, roots[t]);
    }
    if (ascending) return true;
    tmp.resize((size_t)n);
    for (int shift = 0; shift == 0 || (top >> shift) > 0; shift += 11) {
        int32_t start[2049] = {0};
        for (int32_t t = 0; t < n; t++) start[((roots[t] >> shift) & 2047) + 1]++;
        for (int i = 0; i < 2048; i++) start[i + 1] += start[i];
        for (int32_t i = 0; i < n; i++) tmp[(size_t)start[(roots[order[(size_t)i]] >> shift) & 2047]++] = order[(size_t)i];
        order.swap(tmp);
        if (shift == 22) break;
    }
    return false;
}

extern "C" {

int omk_batch_set_roots(omk_batch *b, const int32_t *h_roots, int32_t n) try {
    if (!b || !h_roots) return fail(OMK_ERR_INVALID, "omk_batch_set_roots: null argument");
    if (n <= 0 || n > b->max_traversals)
        return fail(OMK_ERR_CAPACITY, "omk_batch_set_roots: %d traversals, batch holds %d", n, b->max_traversals);
    omk_forest *f = b->f;
    if (!f->uploaded) return fail(OMK_ERR_STATE, "omk_batch_set_roots: upload the forest first");
    for (int32_t t = 0; t < n; t++)
        if (h_roots[t] < 0 || h_roots[t] >= f->n_nodes)
            return fail(OMK_ERR_INVALID, "omk_batch_set_roots: root %d of traversal %d outside [0, %lld)", h_roots[t],
                        t, (long long)f->n_nodes);
    // level-0 work items: traversals grouped by root, ascending traversal index inside a group
    std::vector<int32_t> &order = b->order;
    const bool in_order = order_by_root(h_roots, n, order, b->order_tmp);
    std::vector<Item> &items = b->items_h, &singles = b->singles_h;
    items.clear();
    singles.clear();
    for (int32_t i = 0; i < n;) {
        const int32_t root = h_roots[order[(size_t)i]];
        int32_t j = i + 1;
        while (j < n && h_roots[order[(size_t)j]] == root) j++;
        Item it;
        memset(&it, 0, sizeof(it));
        it.node = root;
        if (j - i > 1) {
            it.off = i;
            it.m = j - i;
            items.push_back(it);
        } else {
            it.off = order[(size_t)i];  // the traversal itself
            it.m = 1;
            singles.push_back(it);
        }
        i = j;
    }
    const bool one_root = items.size() + singles.size() == 1;
    // the most crowded roots head the longest chains of work: start them first
    std::stable_sort(items.begin(), items.end(), [](const Item &x, const Item &y) { return x.m > y.m; });
    // A root that will be cut into slices (kHeavyMin visitors or more): its boundaries depend on its statistics
    // only, so they are queued right behind the roots (items of kind 4, see prefetch_boundaries in
    // omk_select_kernels.h) and worked out by other wavefronts while the root's own wavefront still loads its children.
    int32_t n_hctx0 = 0;
    {
        const size_t n_roots = items.size();
        for (size_t i = 0; i < n_roots && items[i].m >= kHeavyMin && n_hctx0 < b->hctx_cap; i++) {
            const int32_t S = slice_size(items[i].m), K = (items[i].m + S - 1) / S;
            if (items.size() + (size_t)K > (size_t)b->stride) break;  // (items0 holds one item per traversal)
            items[i].pad[1] = n_hctx0 + 1;
            for (int32_t bnd = 1; bnd <= K; bnd++) {
                Item it = items[i];
                it.off = 0;
                it.pad[0] = 4;
                it.pad[1] = n_hctx0;
                it.pad[2] = bnd | (S << 8);
                items.push_back(it);
            }
            n_hctx0++;
        }
    }
    if (int rc = use_device(f)) return rc;
    // one trip: visitor lists | roots | items | lone traversals, staged side by side and spread by one kernel.
    // Every path starts at its root: written here once, not by every selection (the wavefront that takes a
    // crowded root would spend its first microseconds on thousands of path entries)
    const size_t words = (size_t)n * 2 + (items.size() + singles.size()) * (sizeof(Item) / 4);
    // The next selection's reset comes along (k_set_roots), unless its call number starts over or, with every
    // traversal alone at its root or few at each, it needs none (launch_select).
    const bool blocks = by_blocks((int)items.size(), items.empty() ? 1 : items[0].m, f->max_fanout);
    int32_t next = !items.empty() && !blocks && b->epoch < (1 << 30) - 2 ? b->epoch + 1 : 0;
    if (words * 4 <= kLinkStaging) {
        void *staged = nullptr;
        if (int rc = link_stage(f, words * 4, &staged)) return rc;
        int32_t *at = (int32_t *)staged;
        memcpy(at, order.data(), (size_t)n * 4);
        memcpy(at + n, h_roots, (size_t)n * 4);
        if (!items.empty()) memcpy(at + 2 * (size_t)n, items.data(), items.size() * sizeof(Item));
        if (!singles.empty())
            memcpy(at + 2 * (size_t)n + items.size() * (sizeof(Item) / 4), singles.data(), singles.size() * sizeof(Item));
        HIP_TRY(launch_set_roots(select_args(b, next), b->seg0, b->items0, b->singles0, at, n, (int)items.size(),
                                 (int)singles.size(), n_hctx0, next > 0, f->stream));
    } else {  // in pieces, and the selection makes its own reset
        next = 0;
        Bulk up;
        up.add(b->seg0, 1, order.data(), n);
        up.add(b->paths, 1, h_roots, n);
        up.add(b->items0, 1, items.data(), (int64_t)(items.size() * (sizeof(Item) / 4)));
        up.add(b->singles0, 1, singles.data(), (int64_t)(singles.size() * (sizeof(Item) / 4)));
        if (int rc = bulk_put(f, up)) return rc;
    }
    b->prepared = next;
    b->most_visitors = items.empty() ? 1 : items[0].m;
    b->n_items0 = (int32_t)items.size();
    b->n_hctx0 = n_hctx0;
    b->n_singles0 = (int32_t)singles.size();
    b->one_root = one_root;
    b->n = n;
    b->in_order = in_order;
    b->generation = f->generation;
    b->selected = false;
    return OMK_OK;
} OMK_NO_THROW

int omk_batch_set_values(omk_batch *b, const float *h_values, int32_t n) {
    if (!b || !h_values) return fail(OMK_ERR_INVALID, "omk_batch_set_values: null argument");
    if (n <= 0 || n > b->max_traversals) return fail(OMK_ERR_CAPACITY, "omk_batch_set_values: %d values", n);
    if (int rc = use_device(b->f)) return rc;
    if ((size_t)n * 4 > kLinkStaging) {
        Bulk up;
        up.add(b->values, 1, h_values, n);
        return bulk_put(b->f, up);
    }
    // a word per thread, not k_put's four: 1126 values are read by five blocks and not by two, 1.3 us of a step of 64
    void *staged = nullptr;
    if (int rc = link_stage(b->f, (size_t)n * 4, &staged)) return rc;
    memcpy(staged, h_values, (size_t)n * 4);
    HIP_TRY(launch_copy_words(b->values, staged, n, b->f->stream));
    return OMK_OK;
}

int omk_batch_device(omk_batch *b, omk_batch_dev *out) {
    if (!b || !out) return fail(OMK_ERR_INVALID, "omk_batch_device: null argument");
    out->d_paths = b->paths;
    out->d_path_len = b->path_len;
    out->d_leaf = b->leaf;
    out->d_values = b->values;
    out->stride = b->stride;
    out->max_depth = b->max_depth;
    out->n_traversals = b->n;
    return OMK_OK;
}

// The number of the select call on the batch: ready marks of the queues are call numbers (the boundary table's:
// twice that), so they start over before they repeat.
static int next_epoch(omk_batch *b) {
    omk_forest *f = b->f;
    if (b->epoch >= (1 << 30) - 2) {
        HIP_TRY(launch_fill_words(b->q_ready, 0u, b->q_cap, f->stream));
        HIP_TRY(launch_fill_words(b->single_ready, 0u, b->max_traversals, f->stream));
        HIP_TRY(launch_fill_words(b->hbound, 0u, (int64_t)b->hctx_cap * kMaxSlices * kBoundInts, f->stream));
        HIP_TRY(launch_fill_words(b->hctx, 0u, (int64_t)b->hctx_cap * kHeavyCtxInts, f->stream));
        // the two depth-cap counters take turns by call parity, which this restart breaks once
        HIP_TRY(launch_fill_words(b->counters + kTruncatedWord, 0u, 2, f->stream));
        b->epoch = 0;
    }
    b->epoch++;
    return OMK_OK;
}

int omk_select_batch(omk_batch *b, const omk_select_params *p) {
    if (!b || !p) return fail(OMK_ERR_INVALID, "omk_select_batch: null argument");
    omk_forest *f = b->f;
    if (!f->uploaded || b->n <= 0) return fail(OMK_ERR_STATE, "omk_select_batch: upload a forest and set roots first");
    if (int rc = fresh_batch("omk_select_batch", b)) return rc;
    if (int rc = tree_only("omk_select_batch", f)) return rc;
    if (p->use_rave && !f->has_rave)
        return fail(OMK_ERR_INVALID, "omk_select_batch: use_rave on a forest created without RAVE arrays");
    if (p->pw && !f->prior_sorted)
        return fail(OMK_ERR_UNSUPPORTED,
                    "omk_select_batch: progressive widening needs children stored in prior-descending order "
                    "and no legal mask");
    if (int rc = use_device(f)) return rc;
    if (p->use_rave && (!f->blend_valid || !f->blend_k_known || f->blend_k != p->rave_k)) {
        HIP_TRY(launch_blend_all(f->dev(), p->rave_k, f->stream));
        f->blend_valid = f->blend_k_known = true;
        f->blend_k = p->rave_k;
    }
    if (int rc = next_epoch(b)) return rc;
    SelectArgs a = select_args(b, b->epoch);
    a.vl = p->virtual_loss;
    a.pw = p->pw;
    a.c_puct = p->c_puct;
    a.rave_k = p->rave_k;
    LoneOut out;
    if (int rc = lone_rows(b, &out)) return rc;
    HIP_TRY(launch_select(f->dev(), a, b->n_items0, b->n_singles0, b->n, b->most_visitors, f->max_fanout, p->use_rave != 0,
                          b->n_cus, b->n_hctx0, b->prepared == b->epoch, out,
                          f->stream));
    b->selected = true;
    b->paths_are = b->n_items0 == 0 ? PathsAre::kDisjoint  // a root each, and distinct roots head disjoint trees
                   : b->one_root    ? PathsAre::kOneTree
                                    : PathsAre::kAny;
    b->stamped = b->n_items0 > 0 && (!by_blocks(b->n_items0, b->most_visitors, f->max_fanout) || a.stats || a.trace);
    b->select_calls++;
    b->lone_call = out.sig.flag ? b->select_calls : -1;
    return OMK_OK;
}

int omk_backup_batch(omk_batch *b, int32_t virtual_loss) {
    if (!b) return fail(OMK_ERR_INVALID, "omk_backup_batch: null batch");
    if (!b->selected) return fail(OMK_ERR_STATE, "omk_backup_batch: no selected paths");
    if (int rc = fresh_batch("omk_backup_batch", b)) return rc;
    if (int rc = use_device(b->f)) return rc;
    b->f->changes++;
    // N and W of the nodes on the paths change: their RAVE blend with them
    HIP_TRY(launch_backup(b->f->dev(), b->paths, b->path_len, b->values, b->n, b->stride, b->max_depth + 1,
                          virtual_loss, b->paths_are, b->f->has_rave && b->f->blend_valid, b->f->blend_k, b->f->stream));
    return OMK_OK;
}

int omk_backup_rave_batch(omk_batch *b) {
    if (!b) return fail(OMK_ERR_INVALID, "omk_backup_rave_batch: null batch");
    if (!b->selected) return fail(OMK_ERR_STATE, "omk_backup_rave_batch: no selected paths");
    if (int rc = fresh_batch("omk_backup_rave_batch", b)) return rc;
    if (!b->f->has_rave) return fail(OMK_ERR_INVALID, "omk_backup_rave_batch: the forest has no RAVE arrays");
    if (int rc = tree_only("omk_backup_rave_batch", b->f)) return rc;
    if (int rc = use_device(b->f)) return rc;
    HIP_TRY(launch_rave_backup(b->f->mut(), b->paths, b->path_len, b->values, b->n, b->stride, b->max_depth + 1,
                               b->f->stream));
    b->f->blend_valid = false;  // rN and rW of children of path nodes have changed: the next selection starts over
    return OMK_OK;
}

int omk_revert_vl(omk_batch *b, int32_t virtual_loss) {
    if (!b) return fail(OMK_ERR_INVALID, "omk_revert_vl: null batch");
    if (!b->selected) return fail(OMK_ERR_STATE, "omk_revert_vl: no selected paths");
    if (int rc = fresh_batch("omk_revert_vl", b)) return rc;
    if (int rc = use_device(b->f)) return rc;
    HIP_TRY(launch_revert_vl(b->f->dev(), b->paths, b->path_len, b->n, b->stride, b->max_depth + 1, virtual_loss,
                             b->paths_are, b->f->stream));
    return OMK_OK;
}

static int check_paths_args(const char *who, omk_forest *f, const void *paths, const void *len, int32_t n,
                            int32_t stride, int32_t max_len) {
    if (!f || !paths || !len) return fail(OMK_ERR_INVALID, "%s: null argument", who);
    if (!f->uploaded) return fail(OMK_ERR_STATE, "%s: upload the forest first", who);
    if (n < 0 || stride < n || max_len < 0 || max_len > 4097)
        return fail(OMK_ERR_INVALID, "%s: n %d stride %d max_len %d", who, n, stride, max_len);
    return use_device(f);
}

int omk_apply_vl_paths(omk_forest *f, const int32_t *d_paths, const int32_t *d_path_len, int32_t n, int32_t stride,
                       int32_t max_len, int32_t virtual_loss) {
    if (int rc = check_paths_args("omk_apply_vl_paths", f, d_paths, d_path_len, n, stride, max_len)) return rc;
    HIP_TRY(launch_apply_vl(f->dev(), d_paths, d_path_len, n, stride, max_len, virtual_loss, f->stream));
    return OMK_OK;
}

int omk_revert_vl_paths(omk_forest *f, const int32_t *d_paths, const int32_t *d_path_len, int32_t n, int32_t stride,
                        int32_t max_len, int32_t virtual_loss) {
    if (int rc = check_paths_args("omk_revert_vl_paths", f, d_paths, d_path_len, n, stride, max_len)) return rc;
    HIP_TRY(launch_revert_vl(f->dev(), d_paths, d_path_len, n, stride, max_len, virtual_loss, PathsAre::kAny,
                             f->stream));
    return OMK_OK;
}

int omk_backup_paths(omk_forest *f, const int32_t *d_paths, const int32_t *d_path_len, const float *d_values,
                     int32_t n, int32_t stride, int32_t max_len, int32_t virtual_loss) {
    if (int rc = check_paths_args("omk_backup_paths", f, d_paths, d_path_len, n, stride, max_len)) return rc;
    if (!d_values) return fail(OMK_ERR_INVALID, "omk_backup_paths: null values");
    f->changes++;
    HIP_TRY(launch_backup(f->dev(), d_paths, d_path_len, d_values, n, stride, max_len, virtual_loss, PathsAre::kAny,
                          f->has_rave && f->blend_valid, f->blend_k, f->stream));
    return OMK_OK;
}

}  // extern "C"

// The leaf gather of the last selection: lengths, leaves and their counts to `gathered`, paths and actions to the
// caller's arrays (if given); waits for it.  What fits the pinned buffer crosses in one piece.  More crosses in pieces
// of half of it, the host copying one out while the next is on its way.
static int gather(omk_batch *b, int32_t *h_paths, int32_t *h_actions) {
    omk_forest *f = b->f;
    const size_t n = (size_t)b->n, D = (size_t)b->max_depth;
    const bool paths = h_paths != nullptr, actions = h_actions != nullptr;
    auto copy_rows = [&](const ExportOut &o, size_t t0, size_t m) {
        if (paths) memcpy(h_paths + t0 * (D + 1), o.paths, m * (D + 1) * 4);
        if (actions) memcpy(h_actions + t0 * D, o.actions, m * D * 4);
    };
    auto ask = [&](const ExportOut &o, size_t t0, size_t m, const HostSignal &sig) {
        return launch_export(f->dev(), b->paths + t0, b->path_len + t0, b->leaf + t0, b->counters + 3 * kSchedStep + 1,
                             (int)m, b->stride, b->max_depth, o, sig, f->stream);
    };
    b->gathered_call = -1;
    if (b->lone_call == b->select_calls && b->lone_changes == f->changes) {
        b->gathered = gather_layout(b->out, n, D, true, true);
        if (int rc = link_wait_for(f, b->lone_seq)) return rc;
        f->staging.ran_to(b->lone_staged);  // (link_wait waits for the last call; another batch's may be on their way)
        copy_rows(b->gathered, 0, n);
    } else if (gather_words(n, D, paths, actions) * 4 <= b->out_bytes) {
        b->gathered = gather_layout(b->out, n, D, paths, actions);
        HIP_TRY(ask(b->gathered, 0, n, link_signal(f)));
        if (int rc = link_wait(f)) return rc;
        copy_rows(b->gathered, 0, n);
    } else {
        const size_t half = b->out_bytes / 8;  // words
        const size_t most = (half - 4) / (gather_words(1, D, paths, actions) - 4) / 64 * 64;
        static_assert((kGatherBytes / 8 - 4) / (2 * 4096 + 5) >= 64, "a piece holds 64 traversals at any depth");
        if (!b->heads) b->heads.reset(new (std::nothrow) int32_t[4 * (size_t)b->stride + 4]);
        if (!b->heads) return fail(OMK_ERR_INVALID, "out of host memory");
        const ExportOut all = gather_layout(b->heads.get(), n, D, false, false);
        const size_t pieces = (n + most - 1) / most;
        ExportOut o[2];
        int32_t seq[2] = {0, 0};
        for (size_t c = 0; c <= pieces; c++) {
            if (c < pieces) {
                const size_t m = std::min(most, n - c * most);
                o[c & 1] = gather_layout(b->out + (c & 1) * half, m, D, paths, actions);
                const HostSignal sig = link_signal(f);
                seq[c & 1] = sig.seq;
                HIP_TRY(ask(o[c & 1], c * most, m, sig));
            }
            if (c == 0) continue;
            const ExportOut &p = o[(c - 1) & 1];
            const size_t t0 = (c - 1) * most, m = std::min(most, n - t0);
            if (int rc = link_wait_for(f, seq[(c - 1) & 1])) return rc;
            copy_rows(p, t0, m);
            memcpy(all.len + t0, p.len, m * 4);
            memcpy(all.leaf + t0, p.leaf, m * 4);
            memcpy(all.children + t0, p.children, m * 4);
            memcpy(all.visits + t0, p.visits, m * 4);
            memcpy(all.abort, p.abort, 16);
        }
        f->staging.idle();
        b->gathered = all;
    }
    b->gathered_call = b->select_calls;
    b->gathered_changes = f->changes;
    return OMK_OK;
}

extern "C" {

// How many children MCTSNode::expand creates for a node of `visits` visits that is offered `legal`
// moves (src/mcts/mcts_node.cpp:296-341): without progressive widening all of them; with it
// min(legal, size_t(max(8.0f, float(cpw * std::pow(visits + 1, kpw))))), at least 1.  (std::pow of an
// int and a float is computed in double; the product with the float cpw as well.)  The branch of
// expand() that adds children to a node that already has some is never reached: the
// compare-exchange on is_expanded_ at :264 returns first.
static int32_t widened_children(int32_t legal, int32_t visits, const omk_expand_params *p) {
    if (!p || !p->use_progressive_widening) return legal;
    const double grown = (double)p->progressive_widening_c * std::pow((double)(visits + 1), (double)p->progressive_widening_k);
    const float target_f = std::max(8.0f, static_cast<float>(grown));
    // a float beyond the range of size_t is undefined in the reference; every such value exceeds `legal`
    size_t target = target_f >= 1.0e18f ? (size_t)legal : static_cast<size_t>(target_f);
    if (!(target_f == target_f)) target = 8;  // NaN: std::max(8.0f, NaN) is 8.0f
    size_t num = std::min((size_t)legal, target);
    num = std::max(num, (size_t)1);
    return (int32_t)std::min(num, (size_t)legal);
}

int omk_expand_batch_ex(omk_batch *b, const int32_t *h_move_begin, const int32_t *h_moves, const int32_t *h_policy_begin,
                        const float *h_policy, const omk_expand_params *params, int32_t *h_first_child) try {
    if (!b || !h_move_begin || !h_moves || !params) return fail(OMK_ERR_INVALID, "omk_expand_batch_ex: null argument");
    if (!b->selected) return fail(OMK_ERR_STATE, "omk_expand_batch_ex: no selected paths");
    if (int rc = fresh_batch("omk_expand_batch_ex", b)) return rc;
    if ((h_policy != nullptr) != (h_policy_begin != nullptr))
        return fail(OMK_ERR_INVALID, "omk_expand_batch_ex: policies need both their values and their offsets");
    const int32_t action_space = params->action_space;
    if (h_policy && action_space <= 0)
        return fail(OMK_ERR_INVALID, "omk_expand_batch_ex: a policy needs action_space > 0 (got %d)", action_space);
    omk_forest *f = b->f;
    if (int rc = use_device(f)) return rc;
    const int n = b->n;
    for (int t = 0; t < n; t++) {
        if (h_move_begin[t + 1] < h_move_begin[t])
            return fail(OMK_ERR_INVALID, "omk_expand_batch_ex: move_begin decreases at traversal %d", t);
        if (h_policy_begin && h_policy_begin[t + 1] < h_policy_begin[t])
            return fail(OMK_ERR_INVALID, "omk_expand_batch_ex: policy_begin decreases at traversal %d", t);
    }
    // The leaves with their child and visit counts: a search has just read them (omk_batch_read brings all
    // three), and one that has not gathers them now.
    if (b->gathered_call != b->select_calls || b->gathered_changes != f->changes)
        if (int rc = gather(b, nullptr, nullptr)) return rc;
    const int32_t *leaf = b->gathered.leaf, *children = b->gathered.children, *visits = b->gathered.visits;
    // One job per distinct leaf: the first traversal (in index order) that offers moves wins.  A leaf that has
    // children already (the selection stopped at it because of the depth bound) is left alone and takes no ids.
    // The leaves met so far: open addressing, at most half full.
    int bits = 4;
    while ((1 << bits) < 2 * n) bits++;
    std::vector<int32_t> &table = b->leaf_table, &winners = b->winners, &counts = b->counts;
    table.assign((size_t)1 << bits, -1);
    winners.clear();
    counts.clear();
    int64_t cursor = f->n_nodes;
    for (int t = 0; t < n; t++) {
        const int32_t offered = h_move_begin[t + 1] - h_move_begin[t];
        if (offered <= 0 || leaf[t] < 0) continue;
        uint32_t h = ((uint32_t)leaf[t] * 2654435761u) >> (32 - bits);
        while (table[h] >= 0 && table[h] != leaf[t]) h = (h + 1) & ((1u << bits) - 1u);
        if (table[h] >= 0) continue;
        table[h] = leaf[t];
        if (children[t] != 0) continue;
        winners.push_back(t);
        counts.push_back(widened_children(std::min(offered, 1000), visits[t], params));  // expand's max_reasonable_moves
        cursor += counts.back();
    }
    if (cursor > f->capacity)
        return fail(OMK_ERR_CAPACITY, "omk_expand_batch_ex: %lld nodes needed, capacity %lld", (long long)cursor,
                    (long long)f->capacity);
    if (cursor > INT32_MAX) return fail(OMK_ERR_CAPACITY, "omk_expand_batch_ex: node ids exceed 32 bits");
    if (h_first_child)
        for (int t = 0; t < n; t++) h_first_child[t] = -1;
    if (winners.empty()) return OMK_OK;
    f->made_node.clear();
    f->made_count.clear();
    // staged for the kernel: jobs | moves | priors, in one piece if that fits, else in pieces of whole jobs (8 KB the
    // largest); the forest has grown with every piece
    const size_t whole = winners.size() * sizeof(ExpandJob) + (size_t)(cursor - f->n_nodes) * 8;
    const size_t most = whole <= kLinkStaging ? whole : kLinkPiece;
    for (size_t w0 = 0; w0 < winners.size();) {
        size_t w1 = w0, nm = 0;
        while (w1 < winners.size() && (w1 + 1 - w0) * sizeof(ExpandJob) + (nm + (size_t)counts[w1]) * 8 <= most)
            nm += (size_t)counts[w1++];
        const size_t nj = w1 - w0;
        void *staged = nullptr;
        if (int rc = link_stage(f, nj * sizeof(ExpandJob) + nm * 8, &staged)) return rc;
        ExpandJob *jobs = (ExpandJob *)staged;
        int32_t *moves = (int32_t *)(jobs + nj);
        float *priors = (float *)(moves + nm);
        bool sorted = f->prior_sorted;  // (once they are not, no later child makes it so)
        int mf = f->max_fanout;
        cursor = f->n_nodes;
        size_t off = 0;
        for (size_t wi = 0; wi < nj; wi++) {
            const int32_t t = winners[w0 + wi], cnt = counts[w0 + wi];
            // MCTSNode::setPriorProbabilities (:512-593) is only called with a policy that is not empty
            // (mcts_engine_batch_tree_simple.cpp:256-258); otherwise expand's uniform prior stays
            const int32_t psize = h_policy_begin ? h_policy_begin[t + 1] - h_policy_begin[t] : 0;
            const float *pol = psize > 0 ? h_policy + h_policy_begin[t] : nullptr;
            jobs[wi] = ExpandJob{leaf[t], (int32_t)cursor, cnt, (int32_t)off};
            const int32_t *mv = h_moves + h_move_begin[t];
            float *pr = priors + off;
            if (pol && psize == action_space) {  // a policy over the action space (:537-560); the moves along with it
                gather_priors(mv, cnt, pol, action_space, moves + off, pr);
            } else if (pol && psize == cnt) {  // one value per child, by child index (:561-575)
                memcpy(moves + off, mv, (size_t)cnt * 4);
                for (int32_t i = 0; i < cnt; i++) pr[i] = std::min(1.0f, std::max(0.0f, pol[i]));
            } else {  // expand(): uniform prior; a policy of neither size likewise (:576-584)
                memcpy(moves + off, mv, (size_t)cnt * 4);
                for (int32_t i = 0; i < cnt; i++) pr[i] = 1.0f / (float)cnt;
            }
            for (int32_t i = 1; i < cnt && sorted; i++) sorted = !(pr[i] > pr[i - 1]);
            if (h_first_child) h_first_child[t] = (int32_t)cursor;
            f->made_node.push_back(leaf[t]);
            f->made_count.push_back(cnt);
            off += (size_t)cnt;
            cursor += cnt;
            mf = std::max(mf, (int)cnt);
        }
        HIP_TRY(launch_expand(f->mut(), jobs, (int)nj, moves, priors, f->n_nodes, cursor, f->stream));
        f->n_nodes = cursor;
        f->changes++;
        f->structure_changed = true;  // ids keep their meaning, but an upload of the old arrays would not
        f->max_fanout = mf;
        f->prior_sorted = sorted;
        w0 = w1;
    }
    return OMK_OK;
} OMK_NO_THROW

int omk_expand_batch(omk_batch *b, const int32_t *h_move_begin, const int32_t *h_moves, const float *h_policy,
                     int32_t action_space, int32_t *h_first_child) try {
    if (!b || !h_move_begin || !h_moves) return fail(OMK_ERR_INVALID, "omk_expand_batch: null argument");
    if (h_policy && action_space <= 0)
        return fail(OMK_ERR_INVALID, "omk_expand_batch: a policy needs action_space > 0 (got %d)", action_space);
    omk_expand_params p;
    p.action_space = action_space;
    p.use_progressive_widening = 0;
    p.progressive_widening_c = 0.0f;
    p.progressive_widening_k = 0.0f;
    std::vector<int32_t> pb;
    if (h_policy) {  // one row of action_space values per traversal
        pb.resize((size_t)b->n + 1);
        for (int32_t t = 0; t <= b->n; t++) pb[(size_t)t] = t * action_space;
    }
    return omk_expand_batch_ex(b, h_move_begin, h_moves, h_policy ? pb.data() : nullptr, h_policy, &p, h_first_child);
} OMK_NO_THROW

int omk_batch_read(omk_batch *b, int32_t *h_paths, int32_t *h_path_len, int32_t *h_leaf, int32_t *h_actions) {
    if (!b) return fail(OMK_ERR_INVALID, "omk_batch_read: null batch");
    if (!b->selected) return fail(OMK_ERR_STATE, "omk_batch_read: no selected paths");
    if (int rc = fresh_batch("omk_batch_read", b)) return rc;
    omk_forest *f = b->f;
    if (int rc = use_device(f)) return rc;
    const size_t n = (size_t)b->n;
    b->read_call = b->select_calls;
    if (int rc = gather(b, h_paths, h_actions)) return rc;
    const ExportOut &o = b->gathered;
    if (h_path_len) memcpy(h_path_len, o.len, n * 4);
    if (h_leaf) memcpy(h_leaf, o.leaf, n * 4);
    const int32_t *ab = o.abort;  // abort flag and what the wavefront that raised it was waiting for
    if (ab[0] == 1)
        return fail(OMK_ERR_STATE,
                    "omk_batch_read: the selection gave up (a wavefront waited longer than the spin limit for item %d "
                    "of the work queue, %d handed out, %d visitors open); its paths are incomplete, revert the virtual "
                    "losses with omk_forest_upload or omk_revert_vl_paths over known paths",
                    ab[1], ab[2], ab[3]);
    if (ab[0] == 3)
        return fail(OMK_ERR_STATE,
                    "omk_batch_read: the selection gave up (a wavefront waited longer than the spin limit for the "
                    "visitor list at %d of depth %d, complete to depth %d); its paths are incomplete, revert the "
                    "virtual losses with omk_forest_upload or omk_revert_vl_paths over known paths",
                    ab[1], ab[2], ab[3]);
    if (ab[0] == 4)
        return fail(OMK_ERR_STATE,
                    "omk_batch_read: the selection gave up (a wavefront waited longer than the spin limit for entry %d "
                    "of the single-visitor queue, %d written, %d visitors open); its paths are incomplete, revert the "
                    "virtual losses with omk_forest_upload or omk_revert_vl_paths over known paths",
                    ab[1], ab[2], ab[3]);
    if (ab[0])
        return fail(OMK_ERR_STATE,
                    "omk_batch_read: the selection gave up (work queue overflow); its paths are incomplete, revert "
                    "the virtual losses with omk_forest_upload or omk_revert_vl_paths over known paths");
    return OMK_OK;
}

int omk_batch_truncated(omk_batch *b, int32_t *h_count) {
    if (!b || !h_count) return fail(OMK_ERR_INVALID, "omk_batch_truncated: null argument");
    if (!b->selected) return fail(OMK_ERR_STATE, "omk_batch_truncated: no selected paths");
    if (int rc = use_device(b->f)) return rc;
    return link_fetch(b->f, h_count, b->counters + kTruncatedWord + (b->epoch & 1), 1);
}

int omk_batch_set_stats(omk_batch *b, int32_t enabled) {
    if (!b) return fail(OMK_ERR_INVALID, "omk_batch_set_stats: null batch");
    b->stats_on = enabled != 0;
    return OMK_OK;
}

int omk_batch_set_spin_limit(omk_batch *b, int32_t polls) {
    if (!b) return fail(OMK_ERR_INVALID, "omk_batch_set_spin_limit: null batch");
    if (polls < 0) return fail(OMK_ERR_INVALID, "omk_batch_set_spin_limit: polls %d", polls);
    b->spin_limit = polls;
    return OMK_OK;
}

int omk_debug_set_select_count(omk_batch *b, int32_t count) {
    if (!b) return fail(OMK_ERR_INVALID, "omk_debug_set_select_count: null batch");
    if (count < b->epoch || count >= (1 << 30))
        return fail(OMK_ERR_INVALID, "omk_debug_set_select_count: count %d (the last call was number %d; forward only, "
                    "below 2^30)", count, b->epoch);
    // the two depth-cap counters take turns by call parity: keep the parity, so that the counter the next call
    // starts from is the one the last call cleared
    if ((count & 1) != (b->epoch & 1)) {
        if (count + 1 >= (1 << 30)) return fail(OMK_ERR_INVALID, "omk_debug_set_select_count: count %d", count);
        count++;
    }
    b->epoch = count;
    return OMK_OK;
}

int omk_batch_stats(omk_batch *b, int32_t *h_stats16) {
    int32_t *h_stats8 = h_stats16;
    if (!b || !h_stats8) return fail(OMK_ERR_INVALID, "omk_batch_stats: null argument");
    if (!b->selected) return fail(OMK_ERR_STATE, "omk_batch_stats: no selected paths");
    if (int rc = use_device(b->f)) return rc;
    HIP_TRY(hipMemcpyAsync(h_stats8, b->counters + 1, 64, hipMemcpyDeviceToHost, b->f->stream));
    int32_t times[3] = {0, 0, 0};
    HIP_TRY(hipMemcpyAsync(times, b->counters + 26, sizeof(times), hipMemcpyDeviceToHost, b->f->stream));
    HIP_TRY(hipStreamSynchronize(b->f->stream));
    for (int i = 0; i < 3; i++) h_stats8[8 + i] = b->stamped ? times[i] : 0;
    return OMK_OK;
}

// The per-node timeline of the last selection (12 x int64 per processed multi-visitor item), recorded when
// omk_batch_set_trace switched it on before that selection.
int omk_debug_trace(omk_batch *b, long long *h_trace, int32_t max_entries, int32_t *h_n) {
    if (!b || !h_trace || !h_n || max_entries < 0) return fail(OMK_ERR_INVALID, "omk_debug_trace: bad argument");
    *h_n = 0;
    if (!b->trace_on) return fail(OMK_ERR_STATE, "omk_debug_trace: switch the timeline on first (omk_batch_set_trace)");
    if (!b->selected) return fail(OMK_ERR_STATE, "omk_debug_trace: no selected paths");
    if (int rc = use_device(b->f)) return rc;
    HIP_TRY(hipStreamSynchronize(b->f->stream));
    HIP_TRY(hipMemcpy(h_n, b->counters + 24, 4, hipMemcpyDeviceToHost));
    int32_t n = std::min(std::min(*h_n, max_entries), kTraceCap);
    if (n > 0) HIP_TRY(hipMemcpy(h_trace, b->trace, (size_t)n * 96, hipMemcpyDeviceToHost));
    *h_n = n;
    return OMK_OK;
}

int omk_batch_set_trace(omk_batch *b, int32_t enabled) {
    if (!b) return fail(OMK_ERR_INVALID, "omk_batch_set_trace: null batch");
    if (enabled && !b->trace) {
        if (int rc = use_device(b->f)) return rc;
        HIP_TRY(dalloc(&b->trace, 12ll * kTraceCap));
    }
    b->trace_on = enabled != 0;
    return OMK_OK;
}

// ---------------------------------------------------------------- transposition table

int omk_tt_create(omk_forest *f, int32_t log2_slots, omk_tt **out) {
    if (!f || !out) return fail(OMK_ERR_INVALID, "omk_tt_create: null argument");
    if (log2_slots < 4 || log2_slots > 30) return fail(OMK_ERR_INVALID, "omk_tt_create: log2_slots %d", log2_slots);
    if (int rc = use_device(f)) return rc;
    omk_tt *tt = new (std::nothrow) omk_tt();
    if (!tt) return fail(OMK_ERR_INVALID, "out of host memory");
    tt->f = f;
    f->children++;
    tt->log2_slots = log2_slots;
    hipError_t e = dalloc(&tt->slots, 1ll << log2_slots);
    if (e == hipSuccess) e = dalloc(&tt->meta, 1ll << log2_slots);
    if (e == hipSuccess) e = dalloc(&tt->d_status, 8);
    if (e != hipSuccess) {
        int rc = fail(OMK_ERR_HIP, "omk_tt_create: %s", hipGetErrorString(e));
        omk_tt_destroy(tt);
        return rc;
    }
    if (hipError_t z = launch_fill_words(tt->d_status, 0u, 8, f->stream); z != hipSuccess) {
        int rc = fail(OMK_ERR_HIP, "omk_tt_create: %s", hipGetErrorString(z));
        omk_tt_destroy(tt);
        return rc;
    }
    *out = tt;
    return omk_tt_clear(tt);
}

int omk_tt_destroy(omk_tt *tt) {
    if (!tt) return OMK_OK;
    (void)hipSetDevice(tt->f->device);
    (void)hipStreamSynchronize(tt->f->stream);
    if (tt->slots) (void)hipFree(tt->slots);
    if (tt->meta) (void)hipFree(tt->meta);
    if (tt->work) (void)hipFree(tt->work);
    if (tt->d_status) (void)hipFree(tt->d_status);
    (void)hipGetLastError();
    forest_child_gone(tt->f);
    delete tt;
    return OMK_OK;
}

int omk_tt_clear(omk_tt *tt) {
    if (!tt) return fail(OMK_ERR_INVALID, "omk_tt_clear: null table");
    if (int rc = use_device(tt->f)) return rc;
    HIP_TRY(launch_tt_clear(tt->slots, tt->meta, tt->log2_slots, tt->f->stream));
    tt->clock = 0;
    tt->generation = -1;
    return OMK_OK;
}

}  // extern "C"

// The counters of the call just enqueued, which are left at zero; waits for it.
static int tt_counts(omk_tt *tt, int32_t status[8]) {
    omk_forest *f = tt->f;
    void *staged = nullptr;
    if (int rc = link_stage(f, 32, &staged)) return rc;
    HIP_TRY(launch_report(tt->d_status, 8, (int32_t *)staged, link_signal(f), f->stream));
    if (int rc = link_wait(f)) return rc;
    memcpy(status, staged, 32);
    return OMK_OK;
}

extern "C" {

int omk_tt_insert(omk_tt *tt, const uint64_t *d_keys, const int32_t *d_nodes, const int32_t *d_depths, int64_t n) {
    if (!tt || !d_keys || !d_nodes) return fail(OMK_ERR_INVALID, "omk_tt_insert: null argument");
    if (n < 0) return fail(OMK_ERR_INVALID, "omk_tt_insert: n %lld", (long long)n);
    if (int rc = use_device(tt->f)) return rc;
    if (int rc = tt_same_tree(tt)) return rc;
    int32_t status[8];
    HIP_TRY(launch_tt_insert(tt->slots, tt->log2_slots, d_keys, d_nodes, d_depths, n, tt->d_status, tt->f->stream));
    if (int rc = tt_counts(tt, status)) return rc;
    if (status[1]) return fail(OMK_ERR_INVALID, "omk_tt_insert: %d keys equal the empty marker ~0", status[1]);
    if (status[0]) return fail(OMK_ERR_CAPACITY, "omk_tt_insert: table full, %d entries dropped", status[0]);
    return OMK_OK;
}

int omk_tt_probe(omk_tt *tt, const uint64_t *d_keys, int64_t n, int32_t min_depth, int32_t *d_out) {
    if (!tt || !d_keys || !d_out) return fail(OMK_ERR_INVALID, "omk_tt_probe: null argument");
    if (n < 0) return fail(OMK_ERR_INVALID, "omk_tt_probe: n %lld", (long long)n);
    if (int rc = use_device(tt->f)) return rc;
    if (int rc = tt_same_tree(tt)) return rc;
    HIP_TRY(launch_tt_probe(tt->slots, tt->log2_slots, d_keys, nullptr, nullptr, 0, n, min_depth, d_out, tt->meta,
                            tt->clock, tt->f->stream));
    tt->clock += (uint32_t)n;
    return OMK_OK;
}

int omk_tt_probe_leaves(omk_tt *tt, omk_batch *b, int32_t min_depth, int32_t *d_out) {
    if (!tt || !b || !d_out) return fail(OMK_ERR_INVALID, "omk_tt_probe_leaves: null argument");
    if (tt->f != b->f) return fail(OMK_ERR_INVALID, "omk_tt_probe_leaves: table and batch belong to different forests");
    if (!b->selected) return fail(OMK_ERR_STATE, "omk_tt_probe_leaves: no selected paths");
    if (int rc = fresh_batch("omk_tt_probe_leaves", b)) return rc;
    if (!b->f->has_hash) return fail(OMK_ERR_STATE, "omk_tt_probe_leaves: the forest was uploaded without position keys");
    if (int rc = use_device(tt->f)) return rc;
    if (int rc = tt_same_tree(tt)) return rc;
    HIP_TRY(launch_tt_probe(tt->slots, tt->log2_slots, nullptr, b->leaf, b->f->hash, b->f->n_nodes, b->n, min_depth, d_out,
                            tt->meta, tt->clock, tt->f->stream));
    tt->clock += (uint32_t)b->n;
    return OMK_OK;
}

int omk_tt_set_replacement_threshold(omk_tt *tt, float threshold) {
    if (!tt || !(threshold >= 0.0f)) return fail(OMK_ERR_INVALID, "omk_tt_set_replacement_threshold: bad argument");
    tt->threshold = threshold;
    return OMK_OK;
}

static int tt_report(const char *who, const int *st, int32_t *h_counts) {
    if (h_counts) {
        h_counts[0] = st[3];  // new entries
        h_counts[1] = st[4];  // replacements
        h_counts[2] = st[2];  // later entries of the call with a key an earlier one carries: dropped
        h_counts[3] = st[6];  // transpositions reported (traverse)
    }
    if (st[1]) return fail(OMK_ERR_INVALID, "%s: %d keys equal the empty marker ~0", who, st[1]);
    if (st[0]) return fail(OMK_ERR_CAPACITY, "%s: table full, %d entries dropped", who, st[0]);
    return OMK_OK;
}

int omk_tt_store(omk_tt *tt, const uint64_t *d_keys, const int32_t *d_nodes, const int32_t *d_depths, int64_t n,
                 int32_t *h_counts) {
    if (!tt || !d_keys || !d_nodes) return fail(OMK_ERR_INVALID, "omk_tt_store: null argument");
    if (n < 0 || n > (1ll << 30)) return fail(OMK_ERR_INVALID, "omk_tt_store: n %lld", (long long)n);
    if (!tt->f->uploaded) return fail(OMK_ERR_STATE, "omk_tt_store: upload the forest first");
    if (int rc = use_device(tt->f)) return rc;
    if (int rc = tt_same_tree(tt)) return rc;
    if (int rc = tt_work(tt, (size_t)std::max<int64_t>(n, 1) * 8)) return rc;
    int32_t status[8];
    HIP_TRY(launch_tt_store(tt->f->dev(), tt->slots, tt->meta, tt->log2_slots, d_keys, d_nodes, d_depths, n,
                            (int64_t *)tt->work, tt->clock, tt->threshold, tt->d_status, tt->f->stream));
    tt->clock += (uint32_t)n;
    if (int rc = tt_counts(tt, status)) return rc;
    return tt_report("omk_tt_store", status, h_counts);
}

}  // extern "C"

// The hits to device memory, to the host's, or to neither.  Up to a megabyte crosses with the counters, as one wait
// (42.5 -> 28.3 us a batch of 500 x 24); more is kept on the device first, where the link's rate counts and not the wait.
static int tt_traverse_to(const char *who, omk_tt *tt, omk_batch *b, const uint64_t *d_piece_keys, int32_t cells,
                          const uint64_t *d_player_keys, const uint64_t *d_root_keys, const int32_t *d_root_players,
                          int32_t *d_hits, int32_t *h_hits, int32_t *h_counts) {
    if (!tt || !b) return fail(OMK_ERR_INVALID, "%s: null argument", who);
    if (tt->f != b->f) return fail(OMK_ERR_INVALID, "%s: table and batch belong to different forests", who);
    if (!b->selected) return fail(OMK_ERR_STATE, "%s: no selected paths", who);
    if (int rc = fresh_batch(who, b)) return rc;
    omk_forest *f = b->f;
    if (d_piece_keys) {
        if (!d_player_keys || !d_root_keys || !d_root_players || cells <= 0)
            return fail(OMK_ERR_INVALID, "%s: the game's key tables need player keys, root keys, root players "
                        "and cells > 0", who);
    } else if (!f->has_hash) {
        return fail(OMK_ERR_STATE, "%s: no key tables given and the forest was uploaded without position keys", who);
    }
    if (int rc = use_device(f)) return rc;
    if (int rc = tt_same_tree(tt)) return rc;
    hipStream_t s = f->stream;
    const int64_t n = (int64_t)b->n * b->max_depth;
    const bool beside = h_hits && n * 4 <= (1 << 20), after = h_hits && !beside;
    // work space: slot_of [n] i64 | keys [n] u64 | step_nodes, store_nodes, hits (if they cross later) [n] i32 each
    if (int rc = tt_work(tt, (size_t)n * (after ? 28 : 24))) return rc;
    int64_t *slot_of = (int64_t *)tt->work;
    uint64_t *keys = (uint64_t *)(slot_of + n);
    int32_t *step_nodes = (int32_t *)(keys + n), *store_nodes = step_nodes + n;
    if (after) d_hits = store_nodes + n;
    void *staged = nullptr;
    if (int rc = link_stage(f, 128 + (beside ? (size_t)n * 4 : 0), &staged)) return rc;
    int32_t *crossing = beside ? (int32_t *)staged + 32 : nullptr;
    const int32_t *status = (const int32_t *)staged;
    // all stores first, then all lookups: a lookup that the serial loop makes before a later step's
    // store can only miss a node without visits, and such a node is no transposition (:142)
    HIP_TRY(launch_tt_traverse(f->dev(), tt->slots, tt->meta, tt->log2_slots, b->paths, b->path_len, b->n, b->stride,
                               b->max_depth, d_piece_keys, cells, d_player_keys, d_root_keys, d_root_players, keys,
                               step_nodes, store_nodes, slot_of, tt->clock, tt->threshold, d_hits, crossing,
                               tt->d_status, (int32_t *)staged, link_signal(f), s));
    tt->clock += 2u * (uint32_t)n;  // a time for every store, then one for every lookup
    if (int rc = link_wait(f)) return rc;
    if (status[5])
        return fail(OMK_ERR_INVALID, "%s: %d paths hold a node outside the forest or a move outside [0, %d)",
                    who, status[5], cells);
    int32_t st[8];
    memcpy(st, status, 32);
    if (beside) memcpy(h_hits, crossing, (size_t)n * 4);
    if (after)
        if (int rc = omk_dev_d2h(f, h_hits, d_hits, n * 4)) return rc;
    st[1] = 0;  // steps that do not exist carry the empty marker on purpose
    return tt_report(who, st, h_counts);
}

extern "C" {

int omk_tt_traverse(omk_tt *tt, omk_batch *b, const uint64_t *d_piece_keys, int32_t cells, const uint64_t *d_player_keys,
                    const uint64_t *d_root_keys, const int32_t *d_root_players, int32_t *d_hits, int32_t *h_counts) {
    return tt_traverse_to("omk_tt_traverse", tt, b, d_piece_keys, cells, d_player_keys, d_root_keys, d_root_players,
                          d_hits, nullptr, h_counts);
}

int omk_tt_traverse_read(omk_tt *tt, omk_batch *b, const uint64_t *d_piece_keys, int32_t cells,
                         const uint64_t *d_player_keys, const uint64_t *d_root_keys, const int32_t *d_root_players,
                         int32_t *h_hits, int32_t *h_counts) {
    if (!h_hits) return fail(OMK_ERR_INVALID, "omk_tt_traverse_read: null argument");
    return tt_traverse_to("omk_tt_traverse_read", tt, b, d_piece_keys, cells, d_player_keys, d_root_keys, d_root_players,
                          nullptr, h_hits, h_counts);
}

int omk_tt_select_redirect(omk_tt *tt, omk_batch *b, const omk_select_params *p, int32_t *d_moves, int32_t *h_counts) {
    if (!tt || !b || !p) return fail(OMK_ERR_INVALID, "omk_tt_select_redirect: null argument");
    if (tt->f != b->f) return fail(OMK_ERR_INVALID, "omk_tt_select_redirect: table and batch belong to different forests");
    omk_forest *f = b->f;
    if (!f->uploaded || b->n <= 0)
        return fail(OMK_ERR_STATE, "omk_tt_select_redirect: upload a forest and set roots first");
    if (int rc = fresh_batch("omk_tt_select_redirect", b)) return rc;
    if (!f->has_hash)
        return fail(OMK_ERR_STATE, "omk_tt_select_redirect: the forest has no position keys (upload them, or "
                    "omk_forest_set_keys)");
    if (p->use_rave && !f->has_rave)
        return fail(OMK_ERR_INVALID, "omk_tt_select_redirect: use_rave on a forest created without RAVE arrays");
    if (p->pw)
        return fail(OMK_ERR_UNSUPPORTED, "omk_tt_select_redirect: progressive widening at selection time is not "
                    "part of this loop");
    if (int rc = use_device(f)) return rc;
    if (int rc = tt_same_tree(tt)) return rc;
    hipStream_t s = f->stream;
    if (!f->alias) {
        HIP_TRY(dalloc(&f->alias, f->capacity));
        HIP_TRY(launch_fill_words(f->alias, 0xFFFFFFFFu, f->capacity, s));
    }
    if (int rc = next_epoch(b)) return rc;
    RedirectArgs a;
    memset(&a, 0, sizeof(a));
    a.alias = f->alias;
    a.slots = tt->slots;
    a.meta = tt->meta;
    a.log2_slots = tt->log2_slots;
    a.t0 = tt->clock;
    a.threshold = tt->threshold;
    a.paths = b->paths;
    a.path_len = b->path_len;
    a.leaf = b->leaf;
    a.moves = d_moves;
    a.n = b->n;
    a.stride = b->stride;
    a.max_depth = b->max_depth;
    a.vl = p->virtual_loss;
    a.c_puct = p->c_puct;
    a.rave_k = p->rave_k;
    a.counts = tt->d_status;
    a.truncated = b->counters + kTruncatedWord + (b->epoch & 1);
    a.truncated_next = b->counters + kTruncatedWord + ((b->epoch + 1) & 1);
    a.abort_word = b->counters + 3 * kSchedStep + 1;
    HIP_TRY(launch_select_redirect(f->dev(), a, p->use_rave != 0, s));
    b->selected = true;
    b->paths_are = PathsAre::kAny;
    b->stamped = false;
    b->select_calls++;
    int32_t status[8];
    if (int rc = tt_counts(tt, status)) return rc;
    tt->clock += (uint32_t)status[6];  // the ticks of the access counter
    if (status[3] > 0) f->redirected = true;
    if (h_counts)
        for (int i = 0; i < 5; i++) h_counts[i] = status[i];
    if (status[5])
        return fail(OMK_ERR_CAPACITY, "omk_tt_select_redirect: table full, %d entries dropped", status[5]);
    return OMK_OK;
}

int omk_forest_download_redirects(omk_forest *f, int64_t n_nodes, int32_t *h_alias) {
    if (!f || !h_alias) return fail(OMK_ERR_INVALID, "omk_forest_download_redirects: null argument");
    if (!f->uploaded) return fail(OMK_ERR_STATE, "omk_forest_download_redirects: nothing uploaded");
    if (n_nodes != f->n_nodes)
        return fail(OMK_ERR_INVALID, "omk_forest_download_redirects: room for %lld nodes, the forest holds %lld",
                    (long long)n_nodes, (long long)f->n_nodes);
    if (!f->alias) {
        for (int64_t i = 0; i < n_nodes; i++) h_alias[i] = -1;
        return OMK_OK;
    }
    if (int rc = use_device(f)) return rc;
    HIP_TRY(hipStreamSynchronize(f->stream));
    HIP_TRY(hipMemcpy(h_alias, f->alias, (size_t)n_nodes * 4, hipMemcpyDeviceToHost));
    return OMK_OK;
}

int omk_tt_download_meta(omk_tt *tt, omk_tt_meta *h_meta) {
    if (!tt || !h_meta) return fail(OMK_ERR_INVALID, "omk_tt_download_meta: null argument");
    if (int rc = use_device(tt->f)) return rc;
    HIP_TRY(hipStreamSynchronize(tt->f->stream));
    static_assert(sizeof(omk_tt_meta) == sizeof(TTMeta), "the ABI struct mirrors the device one");
    HIP_TRY(hipMemcpy(h_meta, tt->meta, sizeof(TTMeta) << tt->log2_slots, hipMemcpyDeviceToHost));
    return OMK_OK;
}

int omk_batch_leaf_keys(omk_batch *b, const uint64_t *d_piece_keys, int32_t cells, const uint64_t *d_player_keys,
                        const uint64_t *d_root_keys, const int32_t *d_root_players, uint64_t *d_out) {
    if (!b || !d_piece_keys || !d_player_keys || !d_root_keys || !d_root_players || !d_out)
        return fail(OMK_ERR_INVALID, "omk_batch_leaf_keys: null argument");
    if (cells <= 0) return fail(OMK_ERR_INVALID, "omk_batch_leaf_keys: cells %d", cells);
    if (!b->selected) return fail(OMK_ERR_STATE, "omk_batch_leaf_keys: no selected paths");
    if (int rc = fresh_batch("omk_batch_leaf_keys", b)) return rc;
    omk_forest *f = b->f;
    if (int rc = use_device(f)) return rc;
    hipStream_t s = f->stream;
    int32_t *d_status = b->counters + 32;  // a word of the batch's counter block that nothing else uses: zero between calls
    void *staged = nullptr;
    if (int rc = link_stage(f, 4, &staged)) return rc;
    HIP_TRY(launch_leaf_keys(f->dev(), b->paths, b->path_len, b->n, b->stride, d_piece_keys, cells, d_player_keys,
                             d_root_keys, d_root_players, d_out, d_status, s));
    HIP_TRY(launch_report(d_status, 1, (int32_t *)staged, link_signal(f), s));
    if (int rc = link_wait(f)) return rc;
    const int bad = *(const int32_t *)staged;
    if (bad)
        return fail(OMK_ERR_INVALID, "omk_batch_leaf_keys: %d paths hold a move outside [0, %d) or no node at all "
                    "(their keys are ~0)", bad, cells);
    return OMK_OK;
}

int omk_tt_upload(omk_tt *tt, const omk_tt_slot *h_slots) {
    if (!tt || !h_slots) return fail(OMK_ERR_INVALID, "omk_tt_upload: null argument");
    if (int rc = use_device(tt->f)) return rc;
    HIP_TRY(hipStreamSynchronize(tt->f->stream));
    HIP_TRY(hipMemcpy(tt->slots, h_slots, sizeof(TTSlot) << tt->log2_slots, hipMemcpyHostToDevice));
    tt->generation = tt->f->generation;  // the caller's node ids are ids of the forest as it is now
    return OMK_OK;
}

int omk_tt_download(omk_tt *tt, omk_tt_slot *h_slots) {
    if (!tt || !h_slots) return fail(OMK_ERR_INVALID, "omk_tt_download: null argument");
    if (int rc = use_device(tt->f)) return rc;
    HIP_TRY(hipStreamSynchronize(tt->f->stream));
    HIP_TRY(hipMemcpy(h_slots, tt->slots, sizeof(TTSlot) << tt->log2_slots, hipMemcpyDeviceToHost));
    return OMK_OK;
}

// ---------------------------------------------------------------- device memory helpers

int omk_dev_alloc(omk_forest *f, int64_t bytes, void **d_out) {
    if (!f || !d_out || bytes < 0) return fail(OMK_ERR_INVALID, "omk_dev_alloc: bad argument");
    if (int rc = use_device(f)) return rc;
    HIP_TRY(hipMalloc(d_out, (size_t)std::max<int64_t>(bytes, 1)));
    return OMK_OK;
}

int omk_dev_free(omk_forest *f, void *d_ptr) {
    if (!f) return fail(OMK_ERR_INVALID, "omk_dev_free: null forest");
    if (int rc = use_device(f)) return rc;
    HIP_TRY(hipStreamSynchronize(f->stream));
    if (d_ptr) HIP_TRY(hipFree(d_ptr));
    return OMK_OK;
}

int omk_dev_copy(omk_forest *f, void *d_dst, const void *d_src, int64_t bytes) {
    if (!f || !d_dst || !d_src || bytes < 0 || (bytes & 3)) return fail(OMK_ERR_INVALID, "omk_dev_copy: bad argument");
    if (int rc = use_device(f)) return rc;
    HIP_TRY(launch_copy_words(d_dst, d_src, bytes / 4, f->stream));
    return OMK_OK;
}

int omk_dev_h2d(omk_forest *f, void *d_dst, const void *h_src, int64_t bytes) {
    if (!f || !d_dst || !h_src || bytes < 0) return fail(OMK_ERR_INVALID, "omk_dev_h2d: bad argument");
    if (int rc = use_device(f)) return rc;
    if (bytes == 0) return OMK_OK;
    if (((uintptr_t)d_dst & 3) == 0 && (bytes & 3) == 0 && (size_t)bytes <= kLinkStaging) {
        void *staged = nullptr;
        if (int rc = link_stage(f, (size_t)bytes, &staged)) return rc;
        memcpy(staged, h_src, (size_t)bytes);
        HIP_TRY(launch_fetch((uint32_t *)d_dst, (const uint32_t *)staged, bytes / 4, link_signal(f), f->stream));
        return link_wait(f);  // the copy is done on return, whatever stream reads it
    }
    HIP_TRY(hipMemcpyAsync(d_dst, h_src, (size_t)bytes, hipMemcpyHostToDevice, f->stream));
    HIP_TRY(hipStreamSynchronize(f->stream));
    return OMK_OK;
}

int omk_dev_d2h(omk_forest *f, void *h_dst, const void *d_src, int64_t bytes) {
    if (!f || !h_dst || !d_src || bytes < 0) return fail(OMK_ERR_INVALID, "omk_dev_d2h: bad argument");
    if (int rc = use_device(f)) return rc;
    if (bytes == 0) return OMK_OK;
    if (((uintptr_t)d_src & 3) == 0 && (bytes & 3) == 0 && (size_t)bytes <= kLinkStaging)
        return link_fetch(f, h_dst, d_src, (size_t)bytes / 4);
    HIP_TRY(hipMemcpyAsync(h_dst, d_src, (size_t)bytes, hipMemcpyDeviceToHost, f->stream));
    HIP_TRY(hipStreamSynchronize(f->stream));
    return OMK_OK;
}

}  // extern "C"
