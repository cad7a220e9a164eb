// bd_context.hip -- context lifetime, errors, buffers and small queries.
#include <hip/hip_ext.h>
#include <stddef.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <mutex>

#include "bd_internal.h"

namespace bd {

int set_err(bd_ctx *c, int code, const std::string &msg) {
    if (c) c->err = msg;
    return code;
}

int hip_err(bd_ctx *c, hipError_t e, const char *what) {
    std::string m = std::string(what) + ": " + hipGetErrorString(e);
    return set_err(c, e == hipErrorOutOfMemory ? BD_ENOMEM : BD_EHIP, m);
}

// Device memory of a context.  hipFree waits for the device and unmaps, 105 us
// a call, and hipMalloc takes 37; building the graph of 3 M edges makes 34
// pairs of them (4.8 of 6.8 ms).  So freed blocks of up to kPoolBlock are kept
// for the next allocation of about their size, kPoolBytes of them at most,
// until the context is destroyed or an allocation on the device fails, which
// gives back what every context keeps there.  A context's work is on its one
// stream, and a block is kept only once that stream is idle, as hipFree would
// wait too, so any thread may free it.
constexpr size_t kPoolBlock = (size_t)64 << 20;
constexpr size_t kPoolBytes = (size_t)256 << 20;

// The contexts and the lock of their kept blocks; never destroyed, as a program
// may destroy its contexts late.
struct pool_list {
    std::mutex lock;
    std::vector<bd_ctx *> contexts;
};

static pool_list &pools() {
    static pool_list *p = new pool_list;
    return *p;
}

// With the lock held.
static void pool_release(bd_ctx *c) {
    for (auto &b : c->pool) (void)hipFree(b.p);
    c->pool.clear();
    c->pool_bytes = 0;
}

static void pool_join(bd_ctx *c) {
    const std::lock_guard<std::mutex> g(pools().lock);
    pools().contexts.push_back(c);
}

static void pool_leave(bd_ctx *c) {
    const std::lock_guard<std::mutex> g(pools().lock);
    pool_release(c);
    auto &all = pools().contexts;
    all.erase(std::remove(all.begin(), all.end(), c), all.end());
}

// A kept block of the context that holds `size` bytes without wasting a
// quarter, the smallest of them.
static bool pool_take(bd_ctx *c, size_t size, dev_block *out) {
    const std::lock_guard<std::mutex> g(pools().lock);
    size_t best = c->pool.size();
    for (size_t i = 0; i < c->pool.size(); ++i)
        if (c->pool[i].bytes >= size && c->pool[i].bytes <= size + size / 4 + 4096 &&
            (best == c->pool.size() || c->pool[i].bytes < c->pool[best].bytes))
            best = i;
    if (best == c->pool.size()) return false;
    *out = c->pool[best];
    c->pool[best] = c->pool.back();
    c->pool.pop_back();
    c->pool_bytes -= out->bytes;
    return true;
}

// False when the pool is full, or host memory is.
static bool pool_keep(bd_ctx *c, const dev_block &b) {
    const std::lock_guard<std::mutex> g(pools().lock);
    if (c->pool_bytes + b.bytes > kPoolBytes) return false;
    try {
        c->pool.push_back(b);
    } catch (...) {
        return false;
    }
    c->pool_bytes += b.bytes;
    return true;
}

// hipMalloc; when it fails, what every context keeps on this one's device goes
// back first.
static hipError_t device_malloc(bd_ctx *c, void **p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipErrorOutOfMemory) return e;
    const std::lock_guard<std::mutex> g(pools().lock);
    bool any = false;
    for (bd_ctx *o : pools().contexts) {
        if (o->device != c->device || o->pool.empty()) continue;
        pool_release(o);
        any = true;
    }
    if (!any) return e;
    (void)hipGetLastError();
    return hipMalloc(p, bytes);
}

int dev_alloc(bd_ctx *c, void **p, size_t bytes, const char *what) {
    *p = nullptr;
    const size_t unit = bytes < ((size_t)1 << 20) ? 4096 : (size_t)64 << 10;
    dev_block b{nullptr, (std::max<size_t>(bytes, 1) + unit - 1) / unit * unit};
    if (!pool_take(c, b.bytes, &b)) {
        const hipError_t e = device_malloc(c, &b.p, b.bytes);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            char buf[160];
            snprintf(buf, sizeof(buf), "hipMalloc(%s, %zu bytes) failed: %s", what, bytes,
                     hipGetErrorString(e));
            return set_err(c, e == hipErrorOutOfMemory ? BD_ENOMEM : BD_EHIP, buf);
        }
    }
    try {
        c->live[b.p] = b.bytes;
    } catch (...) {
        (void)hipFree(b.p);
        return BD_ENOMEM;
    }
    *p = b.p;
    return BD_OK;
}

void dev_free(bd_ctx *c, void *p) {
    if (!p) return;
    const auto it = c->live.find(p);
    const size_t size = it == c->live.end() ? kPoolBlock + 1 : it->second;
    if (it != c->live.end()) c->live.erase(it);
    if (size <= kPoolBlock) {
        hipError_t e = hipStreamQuery(c->stream);
        if (e == hipErrorNotReady) {
            (void)hipGetLastError();
            e = hipStreamSynchronize(c->stream);
        }
        if (e == hipSuccess && pool_keep(c, {p, size})) return;
        if (e != hipSuccess) (void)hipGetLastError();
    }
    (void)hipFree(p);
}

// (An asynchronous copy on the stream, waited for, takes 10 us longer.)
int copy_sync(bd_ctx *c, void *dst, const void *src, size_t bytes, hipMemcpyKind kind) {
    BD_HIP(c, hipStreamSynchronize(c->stream));
    BD_HIP(c, hipMemcpy(dst, src, bytes, kind));
    return BD_OK;
}

static void free_search(bd_ctx *c) {
    dev_free(c, c->d_depth);
    dev_free(c, c->d_parent);
    dev_free(c, c->d_tree);
    dev_free(c, c->d_out);
    dev_free(c, c->d_marks);
    c->d_tree = nullptr;
    c->d_out = nullptr;
    c->d_marks = nullptr;
    c->depth_valid = false;
    dev_free(c, c->d_cand);
    dev_free(c, c->d_dirty);
    c->d_dirty = nullptr;
    dev_free(c, c->d_comp);
    dev_free(c, c->d_cc_flag);
    dev_free(c, c->d_cc_tasks);
    c->d_comp = nullptr;
    c->d_cc_flag = nullptr;
    c->d_cc_tasks = nullptr;
    c->cc_ntasks = -1;
    c->cc_prep_ms = 0;
    c->cc_prep_bytes = 0;
    c->have_cc = false;
    dev_free(c, c->d_vis);
    dev_free(c, c->d_vis_save);
    for (auto &b : c->d_bm) dev_free(c, b);
    for (auto &q : c->d_q) dev_free(c, q);
    for (auto &t : c->d_tasks) dev_free(c, t);
    ms_free_graph(c);
    for (auto &b : c->d_ms_slices) dev_free(c, b);
    for (auto &b : c->d_ms_slices) b = nullptr;
    c->ms_max_slices = c->ms_seg_cap = 0;
    dev_free(c, c->d_ms_hubs);
    dev_free(c, c->d_ms_hub_slices);
    c->d_ms_hubs = nullptr;
    c->d_ms_hub_slices = nullptr;
    c->ms_nhubs = c->ms_nhub_slices = 0;
    c->ms_hub_order = 0;
    for (auto &b : c->d_ms) dev_free(c, b);
    for (auto &b : c->d_ms_bits) dev_free(c, b);
    dev_free(c, c->d_ms_depth);
    c->d_depth = c->d_parent = c->d_cand = nullptr;
    c->d_vis = c->d_vis_save = nullptr;
    for (auto &b : c->d_bm) b = nullptr;
    for (auto &q : c->d_q) q = nullptr;
    for (auto &t : c->d_tasks) t = nullptr;
    for (auto &b : c->d_ms) b = nullptr;
    for (auto &b : c->d_ms_bits) b = nullptr;
    c->d_ms_depth = nullptr;
    c->ms_depth_rows = 0;
    c->task_cap = 0;
    c->have_result = false;
    c->chunk_hint = 0;
}

void free_graph(bd_ctx *c) {
    free_search(c);
    free_search_layout(c);
    dev_free(c, c->d_off);
    dev_free(c, c->d_cols);
    dev_free(c, c->d_dead);
    dev_free(c, c->d_head);
    dev_free(c, c->d_el);
    c->d_head = nullptr;
    c->max_deg = 0;
    c->d_off = nullptr;
    c->d_cols = nullptr;
    c->d_dead = nullptr;
    c->d_el = nullptr;
    c->el_m = 0;
    c->nv = c->nnz = c->m = c->nwords = 0;
}

// The host watches the flag, which arrives before the launches queued past the
// end have run; those only look at a done flag, and what is queued after them
// is ordered behind them.
int wait_host_flag(bd_ctx *c, const uint32_t *flag, uint32_t value) {
    for (unsigned n = 1;; ++n) {
        if (__atomic_load_n(flag, __ATOMIC_ACQUIRE) == value) return BD_OK;
        if ((n & 255) == 0) {
            const hipError_t e = hipStreamQuery(c->stream);
            if (e == hipSuccess) return BD_OK;
            (void)hipGetLastError();
            if (e != hipErrorNotReady) return hip_err(c, e, "hipStreamQuery");
        }
        __builtin_ia32_pause();
    }
}

int64_t grid_for(const bd_ctx *c, int64_t work_items, int block) {
    int64_t per_cu = c->tune.grid_per_cu > 0 ? c->tune.grid_per_cu : 8;
    int64_t cap = (int64_t)c->cu_count * per_cu;
    int64_t need = (work_items + block - 1) / block;
    return std::max<int64_t>(1, std::min(cap, need));
}

int alloc_search(bd_ctx *c) {
    free_search(c);
    c->cand_clean = false;  // the first search fills the candidate array
    int rc;
    const int64_t nv = c->nv, nw = c->nwords;
    if ((rc = dev_alloc(c, (void **)&c->d_parent, sizeof(int32_t) * nv, "parent"))) return rc;
    if ((rc = dev_alloc(c, (void **)&c->d_cand, sizeof(int32_t) * nv, "candidate parents")))
        return rc;
    if ((rc = dev_alloc(c, (void **)&c->d_dirty, nw, "candidate words"))) return rc;
    if ((rc = dev_alloc(c, (void **)&c->d_vis, sizeof(uint64_t) * nw, "visited"))) return rc;
    if ((rc = dev_alloc(c, (void **)&c->d_vis_save, sizeof(uint64_t) * nw, "visited copy")))
        return rc;
    for (auto &b : c->d_bm)
        if ((rc = dev_alloc(c, (void **)&b, sizeof(uint64_t) * nw, "frontier bitmap"))) return rc;
    // Segmented lists: kSeg segments of twice the even share, then an
    // overflow segment as large as the whole list can be.
    c->qseg_cap = 2 * ((nv + kSeg - 1) / kSeg) + 4096;
    for (auto &q : c->d_q)
        if ((rc = dev_alloc(c, (void **)&q, sizeof(int32_t) * (kSeg * c->qseg_cap + nv),
                            "frontier queue")))
            return rc;
    // Each vertex of degree >= task_threshold yields <= deg/task_edges + 1
    // tasks and appears in at most one frontier, so this bound is exact.
    const int64_t te = std::max(64, c->tune.task_edges);
    const int64_t tt = std::max(16, c->tune.task_threshold);
    c->task_cap = c->nnz / te + c->nnz / tt + 16;
    c->tseg_cap = 2 * ((c->task_cap + kSeg - 1) / kSeg) + 1024;
    for (auto &t : c->d_tasks)
        if ((rc = dev_alloc(c, (void **)&t, sizeof(td_task) * (kSeg * c->tseg_cap + c->task_cap),
                            "tasks")))
            return rc;
    return build_search_layout(c);
}

}  // namespace bd

using namespace bd;

extern "C" int bd_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return n;
}

extern "C" int bd_create(bd_ctx **out, int device) {
    if (!out) return BD_EINVAL;
    *out = nullptr;
    int n = bd_device_count();
    if (n <= 0) return BD_ENOEXT;
    if (device < 0 || device >= n) return BD_EINVAL;
    bd_ctx *c = new bd_ctx();
    c->device = device;
    pool_join(c);
    // launch shape and thresholds: beedrill_amd/autotune.py's best on MI355X
    // (RMAT scale 24, generator seed 1, models/tuning_rmat_s24.json), except
    // bu_cap (its 64 gained 0.8% there and cost an Erdos-Renyi graph 6%) and
    // bu_batch 8 (six rounds per trip, added after that run)
    c->tune.block = 128;
    c->tune.grid_per_cu = 10;
    c->tune.bu_words = 16;
    c->tune.bu_cap = 32;
    c->tune.wave_threshold = 256;
    c->tune.task_threshold = 16;
    c->tune.task_edges = 1536;
    c->tune.level_driver = 1;
    c->tune.time_steps = 2;
    c->tune.bu_head = 1;
    c->tune.step_kernels = 2;
    c->tune.bu_grid_per_cu = 4;
    c->tune.learned_margin_milli = 250;
    c->tune.ms_alpha = 4;
    c->tune.learned_min_skew = 8;
    c->tune.td_split_edges = 1 << 16;
    c->tune.vertex_order = 4;
    c->tune.bu_batch = 8;
    c->tune.learned_near = 4;
    hipError_t e = hipSetDevice(device);
    if (e == hipSuccess) {
        hipDeviceProp_t prop;
        e = hipGetDeviceProperties(&prop, device);
        if (e == hipSuccess) c->cu_count = prop.multiProcessorCount;
    }
    int khz = 0;
    if (e == hipSuccess) e = hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device);
    if (e == hipSuccess && khz > 0) c->wall_khz = khz;
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    // ev[0..1] bracket whole searches; ev[2..3] time single kernels and use
    // a device-scope release, so a kernel's time does not include writing
    // the L2 back for the host (results are read with hipMemcpy, which
    // orders itself)
    for (int i = 0; i < 4 && e == hipSuccess; ++i)
        e = i < 2 ? hipEventCreate(&c->ev[i])
                  : hipEventCreateWithFlags(&c->ev[i], hipEventReleaseToDevice);
    if (e == hipSuccess) e = device_malloc(c, (void **)&c->d_ctl, 2 * sizeof(ctl_block));
    if (e == hipSuccess) e = device_malloc(c, (void **)&c->d_seg, sizeof(seg_counters));
    if (e == hipSuccess)
        e = hipHostMalloc((void **)&c->h_state, sizeof(host_state),
                          hipHostMallocMapped | hipHostMallocCoherent);
    if (e == hipSuccess) {
        memset((void *)c->h_state, 0, offsetof(host_state, log));
        c->h_ctl = c->h_state->ctl;
        c->h_res = &c->h_state->res;
        c->h_flags = c->h_state->flags;
        c->h_cc = c->h_state->cc;
        c->h_log = c->h_state->log;
        c->log_cap = 1 << 16;
    }
    if (e == hipSuccess) {
        e = device_malloc(c, (void **)&c->d_log, sizeof(bd_level_rec) * c->log_cap);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        bd_destroy(c);
        return BD_EHIP;
    }
    if (static_scratch_init(c) != BD_OK) {
        bd_destroy(c);
        return BD_EHIP;
    }
    *out = c;
    return BD_OK;
}

extern "C" int bd_destroy(bd_ctx *c) {
    if (!c) return BD_OK;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    free_graph(c);
    (void)hipFree(c->d_ctl);
    (void)hipFree(c->d_seg);
    (void)hipFree(c->d_log);
    dev_free(c, c->d_script);
    dev_free(c, c->d_mlp);
    dev_free(c, c->d_mlp_ops);
    dev_free(c, c->d_mlp_ws);
    pool_leave(c);
    if (c->h_state) (void)hipHostFree(c->h_state);
    free_ring(c);
    for (auto &e : c->ev)
        if (e) (void)hipEventDestroy(e);
    for (auto &e : c->ev_pool)
        if (e) (void)hipEventDestroy(e);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
    return BD_OK;
}

extern "C" const char *bd_last_error(const bd_ctx *c) { return c ? c->err.c_str() : "null context"; }

extern "C" int bd_graph_info(bd_ctx *c, int64_t *nv, int64_t *nnz, int64_t *m) {
    if (!c) return BD_EINVAL;
    if (nv) *nv = c->nv;
    if (nnz) *nnz = c->nnz;
    if (m) *m = c->m;
    return BD_OK;
}

extern "C" int bd_graph_download(bd_ctx *c, int64_t *off, int32_t *cols) {
    if (!c) return BD_EINVAL;
    if (!c->d_off) return set_err(c, BD_ESTATE, "no graph");
    BD_HIP(c, hipSetDevice(c->device));
    int rc;
    if (off && (rc = carry_copy(c, carry::i64_i64, off, c->d_off, c->nv + 1))) return rc;
    if (cols && (rc = carry_copy(c, carry::i32_i32, cols, c->d_cols, c->nnz))) return rc;
    return BD_OK;
}

// hybrid_bfs_main.cc:136-144: rng() % V from lcg(0) (lcg.h), rejecting
// vertices of degree 0.  Degrees are read from the device CSR on demand.
extern "C" int bd_pick_roots(bd_ctx *c, int64_t n, int64_t *roots) {
    if (!c || n < 0 || (n > 0 && !roots)) return BD_EINVAL;
    if (!c->d_off) return set_err(c, BD_ESTATE, "no graph");
    BD_HIP(c, hipSetDevice(c->device));
    std::vector<int64_t> off(c->nv + 1);
    if (int rc = copy_sync(c, off.data(), c->d_off, sizeof(int64_t) * (c->nv + 1),
                           hipMemcpyDeviceToHost))
        return rc;
    if (off[c->nv] == 0 && n > 0) return set_err(c, BD_ESTATE, "graph has no edges");
    uint64_t st = 1;  // lcg(0): the skip-ahead loop leaves ran = 1
    const uint64_t mul = 6364136223846793005ULL;
    for (int64_t i = 0; i < n; ++i) {
        int64_t s;
        do {
            st = mul * st + 1ULL;
            s = (int64_t)(st % (uint64_t)c->nv);
        } while (off[s + 1] - off[s] == 0);
        roots[i] = s;
    }
    return BD_OK;
}

extern "C" int bd_set_tuning(bd_ctx *c, const bd_tuning *t) {
    if (!c || !t) return BD_EINVAL;
    bd_tuning n = c->tune;
    if (t->block > 0) {
        if (t->block != 128 && t->block != 256 && t->block != 512)
            return set_err(c, BD_EINVAL, "block must be 128, 256 or 512");
        n.block = t->block;
    }
    if (t->bu_words > 0) n.bu_words = std::min(t->bu_words, 32);
    if (t->bu_cap > 0) n.bu_cap = t->bu_cap;
    if (t->grid_per_cu > 0) n.grid_per_cu = std::min(t->grid_per_cu, 64);
    if (t->wave_threshold > 0) n.wave_threshold = t->wave_threshold;
    if (t->task_threshold > 0) n.task_threshold = std::max(t->task_threshold, 16);
    if (t->task_edges > 0) n.task_edges = std::max(t->task_edges, 64);
    if (t->level_driver == 1 || t->level_driver == 2) n.level_driver = t->level_driver;
    if (t->time_steps >= 1 && t->time_steps <= 4) n.time_steps = t->time_steps;
    if (t->bu_head == 1 || t->bu_head == 2) n.bu_head = t->bu_head;
    if (t->step_kernels == 1 || t->step_kernels == 2) n.step_kernels = t->step_kernels;
    if (t->bu_grid_per_cu > 0) n.bu_grid_per_cu = std::min(t->bu_grid_per_cu, 64);
    if (t->learned_margin_milli > 0) n.learned_margin_milli = t->learned_margin_milli;
    if (t->ms_alpha > 0) n.ms_alpha = t->ms_alpha;
    if (t->learned_min_skew > 0) n.learned_min_skew = t->learned_min_skew;
    if (t->td_split_edges > 0) n.td_split_edges = t->td_split_edges;
    if (t->vertex_order > 4) return set_err(c, BD_EINVAL, "vertex_order must be 1 to 4");
    if (t->vertex_order > 0) n.vertex_order = t->vertex_order;
    if (t->bu_batch > 0) n.bu_batch = t->bu_batch >= 8 ? 8 : (t->bu_batch >= 4 ? 4 : 1);
    if (t->learned_near > 0) n.learned_near = std::min(t->learned_near, 1 << 16);
    bool realloc = (n.task_edges != c->tune.task_edges || n.task_threshold != c->tune.task_threshold ||
                    n.vertex_order != c->tune.vertex_order);
    c->tune = n;
    if (realloc && c->d_off) {
        BD_HIP(c, hipSetDevice(c->device));
        return alloc_search(c);  // rebuilds the search layout when its order changed
    }
    return BD_OK;
}

extern "C" int bd_get_tuning(bd_ctx *c, bd_tuning *t) {
    if (!c || !t) return BD_EINVAL;
    *t = c->tune;
    return BD_OK;
}

// ------------------------------------------------------------ measurement

namespace {

// A plain streaming copy (16-byte loads and stores, grid-stride): the
// reference point for the hardware traffic counters and for achievable HBM
// bandwidth.
__global__ __launch_bounds__(256) void k_copy(const uint4 *__restrict__ src,
                                              uint4 *__restrict__ dst, int64_t n) {
    // four independent 16-byte loads in flight per thread
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i + 3 * stride < n; i += 4 * stride) {
        const uint4 a = src[i], b = src[i + stride], c = src[i + 2 * stride],
                    d = src[i + 3 * stride];
        dst[i] = a;
        dst[i + stride] = b;
        dst[i + 2 * stride] = c;
        dst[i + 3 * stride] = d;
    }
    for (; i < n; i += stride) dst[i] = src[i];
}

}  // namespace

extern "C" int bd_copy_bandwidth(bd_ctx *c, int64_t bytes, int reps, double *gbps) {
    if (!c || bytes < 16 || reps < 1) return BD_EINVAL;
    BD_HIP(c, hipSetDevice(c->device));
    const int64_t n = bytes / 16;
    void *src = nullptr, *dst = nullptr;
    int rc = dev_alloc(c, &src, sizeof(uint4) * n, "copy source");
    if (!rc) rc = dev_alloc(c, &dst, sizeof(uint4) * n, "copy target");
    struct guard {
        bd_ctx *c;
        void *a, *b;
        ~guard() {
            dev_free(c, a);
            dev_free(c, b);
        }
    } g{c, src, dst};
    if (rc) return rc;
    BD_HIP(c, hipMemsetAsync(src, 1, sizeof(uint4) * n, c->stream));
    const int64_t grid = (int64_t)c->cu_count * 4;
    float best = 0;
    for (int r = 0; r < reps; ++r) {
        hipExtLaunchKernelGGL(k_copy, dim3(grid), dim3(256), 0, c->stream, c->ev[2], c->ev[3], 0,
                              (const uint4 *)src, (uint4 *)dst, n);
        BD_HIP(c, hipGetLastError());
        BD_HIP(c, hipEventSynchronize(c->ev[3]));
        float ms = 0;
        BD_HIP(c, hipEventElapsedTime(&ms, c->ev[2], c->ev[3]));
        if (r == 0 || ms < best) best = ms;
    }
    if (gbps) *gbps = best > 0 ? 2.0 * 16.0 * (double)n / (best * 1e-3) / 1e9 : 0.0;
    return BD_OK;
}

