// Host-side context and device-resident graph state.
#pragma once

#include <hip/hip_runtime.h>

#include "vnm_internal.h"

#include <atomic>
#include <map>
#include <memory>
#include <mutex>
#include <set>
#include <string>
#include <vector>

// Kernel timers: events recorded around selected launches on the context's
// stream (the reference's GpuTimer, util/utility.h:267-301), resolved lazily.
struct vnm_timer_pending {
    std::string name;
    hipEvent_t a, b;
};

namespace vnm {

// Idle device memory of one context, for its next calls: packing takes 60
// buffers and a learned reorder 45, and hipMalloc and hipFree (which waits for the
// whole device) were most of such a call's time (packing R-MAT 65,536 took 7.6 ms,
// of it 0.9 in kernels, and 1.27 from the pool; its learned reorder 8.1 ms and 5.8).
// A block given back may still be read by work enqueued on the context's stream;
// the next owner's work is enqueued behind it, on the same stream, so nothing
// waits.  (Host copies into a block go through the stream as well.  Work on
// another stream must have ended before its buffers are released.)  At most
// POOL_IDLE bytes stay idle, until vnm_ctx_trim, an allocation of any context that
// fails without them, or the end of the context and of its objects, which share
// the pool.
constexpr size_t POOL_IDLE = (size_t)2 << 30;
constexpr size_t POOL_GRAIN = 4096;

class DevPool;

// The process's pools.  (Never destroyed: a context may be left to process exit.)
struct PoolList {
    std::mutex mu;
    std::set<DevPool *> pools;
    std::atomic<int> wanted{0};  // allocations that failed and try again: nothing more goes idle
    static PoolList &all() {
        static PoolList *l = new PoolList();
        return *l;
    }
    inline void flush();
};

// hipMalloc; where it fails, every pool's idle blocks are freed first.
inline hipError_t device_alloc(void **p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        PoolList &l = PoolList::all();
        l.wanted++;
        l.flush();
        e = hipMalloc(p, bytes);
        l.wanted--;
        if (e != hipSuccess) (void)hipGetLastError();
    }
    return e;
}

class DevPool {
public:
    DevPool() {
        PoolList &l = PoolList::all();
        std::lock_guard<std::mutex> lk(l.mu);
        l.pools.insert(this);
    }
    ~DevPool() {
        PoolList &l = PoolList::all();
        std::lock_guard<std::mutex> lk(l.mu);
        l.pools.erase(this);
        flush();
    }
    // Free the idle blocks.
    void trim() {
        std::lock_guard<std::mutex> lk(PoolList::all().mu);
        flush();
    }
    DevPool(const DevPool &) = delete;
    DevPool &operator=(const DevPool &) = delete;
    // A block of at least `bytes` (> 0); *cap its size.
    hipError_t take(size_t bytes, void **p, size_t *cap) {
        {
            std::lock_guard<std::mutex> lk(mu);
            auto it = idle.lower_bound(bytes);
            if (it != idle.end() && it->first <= 2 * bytes + POOL_GRAIN) {
                *p = it->second;
                *cap = it->first;
                idle_bytes -= it->first;
                idle.erase(it);
                return hipSuccess;
            }
        }
        // rounded up to an eighth of its size, so that a little growth still fits;
        // just its size where memory is short
        size_t grain = POOL_GRAIN;
        while (grain * 16 <= bytes) grain *= 2;
        *cap = (bytes + grain - 1) / grain * grain;
        hipError_t e = device_alloc(p, *cap);
        if (e != hipSuccess && *cap > bytes) {
            *cap = bytes;
            e = device_alloc(p, bytes);
        }
        return e;
    }
    void give(void *p, size_t cap) noexcept {
        try {
            std::lock_guard<std::mutex> lk(mu);
            if (idle_bytes + cap <= POOL_IDLE && PoolList::all().wanted == 0) {
                idle.emplace(cap, p);
                idle_bytes += cap;
                return;
            }
        } catch (...) {  // no memory for the entry
        }
        (void)hipFree(p);
    }

private:
    friend struct PoolList;
    // Under PoolList::mu, so that an allocation that failed finds these blocks freed
    // when its own turn to flush comes.
    void flush() {
        std::multimap<size_t, void *> blocks;
        {
            std::lock_guard<std::mutex> lk(mu);
            blocks.swap(idle);
            idle_bytes = 0;
        }
        for (auto &b : blocks) (void)hipFree(b.second);  // waits for the device
    }
    std::mutex mu;
    std::multimap<size_t, void *> idle;
    size_t idle_bytes = 0;
};

inline void PoolList::flush() {
    std::lock_guard<std::mutex> lk(mu);
    for (DevPool *p : pools) p->flush();
}

// The pool that this host thread's allocations come from, for the length of a
// scope: each entry point opens one for its context.
inline thread_local std::shared_ptr<DevPool> t_pool;

struct PoolScope {
    std::shared_ptr<DevPool> prev;
    explicit PoolScope(const std::shared_ptr<DevPool> &p) : prev(t_pool) { t_pool = p; }
    ~PoolScope() { t_pool = prev; }
    PoolScope(const PoolScope &) = delete;
    PoolScope &operator=(const PoolScope &) = delete;
};

}  // namespace vnm

struct vnm_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    std::shared_ptr<vnm::DevPool> pool;
    float *noalloc_slots = nullptr;  // device address of the static SpMM slot array on `device`
    int64_t launches = 0;
    bool timing = false;
    std::vector<vnm_timer_pending> pending;
    std::map<std::string, std::pair<double, int64_t>> timers;
};

namespace vnm {

// A device buffer, from the pool of the scope it was allocated in.
template <typename T>
struct DBuf {
    T *p = nullptr;
    size_t n = 0;
    int alloc(size_t count) {
        release();
        if (count == 0) count = 1;
        hipError_t e;
        if (t_pool) e = t_pool->take(count * sizeof(T), (void **)&p, &cap);
        else e = device_alloc((void **)&p, count * sizeof(T));
        if (e != hipSuccess) {
            p = nullptr;
            return set_error(e == hipErrorOutOfMemory ? VNM_E_OOM : VNM_E_HIP,
                             "hipMalloc of %zu bytes failed: %s", count * sizeof(T), hipGetErrorString(e));
        }
        pool = t_pool;
        n = count;
        return VNM_OK;
    }
    void release() {
        if (p) {
            if (pool) pool->give(p, cap);
            else (void)hipFree(p);
        }
        pool.reset();
        p = nullptr;
        n = 0;
    }
    void swap(DBuf &o) {
        std::swap(p, o.p);
        std::swap(n, o.n);
        std::swap(cap, o.cap);
        pool.swap(o.pool);
    }
    DBuf() = default;
    DBuf(const DBuf &) = delete;
    DBuf &operator=(const DBuf &) = delete;
    ~DBuf() { release(); }

private:
    size_t cap = 0;
    std::shared_ptr<DevPool> pool;
};

}  // namespace vnm

// The matrix lives on the device as the reference's COO (mtx/Mtx.h:78-80):
// entries in the reference's COO order (the order at the last load), ids
// current.  Every reorder relabels these arrays in place, as the Reorder
// kernel does (reorder/reorder.h:23-35).
struct vnm_graph {
    vnm_ctx *ctx = nullptr;
    int32_t nrows = 0, ncols = 0, M = 8;
    int64_t nnz = 0;
    vnm::DBuf<int32_t> row, col;
    vnm::DBuf<float> val;
    // composed relabel since creation: original id -> current id
    vnm::DBuf<int32_t> perm_total;
    // scratch reused across calls
    vnm::DBuf<int32_t> cptr, crow;        // CSC of nonzero entries (N:M run)
    vnm::DBuf<int32_t> perm, inv, cnt, nzr, ws;
    vnm::DBuf<uint32_t> tab;              // per-slot row bitmaps (bytes in words)
    vnm::DBuf<uint32_t> rt;               // N:M greedy row records A and B (16 B per row each)
    vnm::DBuf<int32_t> gst;               // N:M greedy device state
    vnm::DBuf<int32_t> queue;             // work counters of the per-segment passes
    // a batch of N:M greedy rounds captured once (its kernels read only the
    // buffers above, which live as long as the graph)
    hipGraph_t nm_graph = nullptr;
    hipGraphExec_t nm_exec = nullptr;
    std::vector<uint8_t> nm_key;          // the arguments nm_exec was captured with
    size_t tab_slots = 0;
    // a relabel of a matrix with fewer columns than rows moved entries past
    // the padded column count (the row permutation also renames columns)
    bool col_overflow = false;
    // bumped whenever the COO is relabelled or re-sorted; caches built from
    // the COO (the proposer's adjacency) are valid for one epoch
    int64_t epoch = 0;
    void *lp_cache = nullptr;
    void (*lp_cache_free)(void *) = nullptr;
    int32_t nseg() const { return (nrows + M - 1) / M; }
    ~vnm_graph() {
        if (lp_cache_free) lp_cache_free(lp_cache);
        if (nm_exec) (void)hipGraphExecDestroy(nm_exec);
        if (nm_graph) (void)hipGraphDestroy(nm_graph);
    }
};

namespace vnm {

int graph_scratch(vnm_graph *g);
int build_csc(vnm_graph *g);
int build_csc_unique(vnm_graph *g);
int locate_all(vnm_graph *g, int N, int32_t *d_cnt, int32_t *d_nzr);
int relabel(vnm_graph *g, const int32_t *d_perm);
int max_ids(vnm_graph *g, const int32_t *row, const int32_t *col, int32_t *max_row, int32_t *max_col);
int nm_reorder(vnm_graph *g, int N, int sched, int maxiter, vnm_nm_stats *st);
int nm_reorder_batch(vnm_graph *const *gs, int count, int N, const int *scheds, int maxiter,
                     vnm_nm_stats *stats);
int nm_reorder_allpairs(vnm_graph *g, int N, int sched, int maxiter, int clean, vnm_nm_stats *stats);
int nm_reorder_ex(vnm_graph *g, int N, int sched, int maxiter, int round_cap, int32_t *d_trace,
                  int64_t trace_cap, int64_t *trace_len, vnm_nm_stats *stats);
int venom_eval(vnm_graph *g, int V, int32_t *inv, int32_t *inv_strict);
int lp_reorder(vnm_graph *g, const vnm_lp_model *m, int N, int mode, int topk, int window, int maxiter,
               uint64_t seed, vnm_lp_stats *stats);
int lp_reorder_batch(vnm_graph *const *gs, int count, const vnm_lp_model *m, int N, int mode, int topk,
                     int window, int maxiter, uint64_t seed, vnm_lp_stats *stats);
int venom_reorder(vnm_graph *g, int V, int maxiter, vnm_venom_stats *st);
int reload_sort(vnm_graph *g, bool quantize);
int graph_clone(vnm_graph *src, vnm_graph **out);
int ensure_tab(vnm_graph *g, size_t slots);
int noalloc_setup(int device, float **out);

// Event pair around one launch when the context's timers are on.
struct KernelTimer {
    vnm_ctx *ctx;
    const char *name;
    hipEvent_t a = nullptr, b = nullptr;
    KernelTimer(vnm_ctx *c, const char *n);
    void stop();
    ~KernelTimer() { stop(); }  // a scope left early still records its end
    KernelTimer(const KernelTimer &) = delete;
    KernelTimer &operator=(const KernelTimer &) = delete;
};

}  // namespace vnm
