// bd_cc.hip -- connected components on gfx950 (components::run,
// components.cc:38-104, and components::check, :152-202).
//
// Labels are int32[V]; every vertex starts as its own component.  An
// iteration is an edge pass and a shortcut pass, as in the reference:
//   edge pass (:56-66): each vertex takes the smallest label among its
//     neighbours when that is smaller than its own.  The CSR is symmetric,
//     so every directed edge (src -> dst) lowers label[src] in src's own
//     pull: a short list's label is written by its vertex's lane alone, with
//     no atomics; long lists are cut into slices merged by atomicMin.
//   shortcut pass (:74-78): label[v] = label[label[v]] until it is a root.
// The run ends after the first edge pass that changes nothing (:70); the
// iteration count includes that pass.  Labels only decrease and stay ids of
// the vertex's own component, so each component ends labelled by its
// smallest vertex id, whatever order the passes read the labels in.
//
// Most vertices end in one component, and most of those carry its label
// after a pass or two.  From the second pass on, the vertices that carry the
// label g of the vertex of largest degree read nothing: every edge between
// them and the rest is read from its other end (the CSR is symmetric), which
// takes g when g is lower than its own label and lowers the label of root g
// itself when its own is lower; an edge between two of them joins nothing.
// So a pass that changes no label still means that every edge's ends agree,
// and a vertex that has taken g needs no more of its list.  At scale 23 the
// passes after the first then cost little more than reading the labels.
//
// Where no component is that large (a union of many, a forest, long paths)
// every pass reads nearly all labels, so passes have to be few: a vertex that
// takes a lower label also lowers the root of the one it carried, and the
// shortcut brings along every vertex that carries that root.  A label
// that meets a lower one is then gone after the pass; those left have only
// higher ones around, at most half of the labels of a component that has more
// than one, so passes grow with the logarithm of its size and not with its
// diameter (100 k paths of 200: 105 passes, 93 ms, without; 6, 6.7 ms, with).
//
// A run is a fixed sequence of launches with no host round trip: an edge
// pass, a shortcut and a one-workgroup launch that closes the pass
// (k_cc_close); launches queued past the last pass return at once.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <vector>

#include "bd_device.h"
#include "bd_internal.h"

namespace bd {
namespace {

// The run's state on the device, and what it leaves for the host.
struct cc_state {
    int32_t done;     // an edge pass changed nothing
    int32_t g;        // label of the vertex of largest degree, before the pass
    int32_t changed;  // a label went down in this pass
    int32_t bad;      // a label out of range
    int64_t iters;    // passes closed
    uint64_t t_start, t_hook, t_passes;  // wall_clock64 stamps; sum over passes
};
struct cc_result {
    int64_t iters, components, labels_read, edge_bytes;
    uint64_t ticks, pass_ticks;
    int32_t bad;
    uint32_t seq;
};

// Every vertex its own component; state and counters cleared.
__global__ void k_cc_init(int32_t *__restrict__ comp, int64_t nv, cc_state *__restrict__ st,
                          unsigned long long *__restrict__ count, int ncount) {
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv;
         v += (int64_t)gridDim.x * blockDim.x)
        comp[v] = (int32_t)v;
    if (blockIdx.x != 0) return;
    for (int i = threadIdx.x; i < ncount; i += blockDim.x) count[i] = 0;
    if (threadIdx.x == 0) {
        *st = cc_state{};
        st->t_start = wall_clock64();
    }
}

// Lists of kCcHeavy edges or more are cut into slices of kCcSlice edges,
// one wave each, merged into the label with atomicMin; shorter lists are
// walked 64 edges at a time by the wave that owns their vertex.
constexpr int kCcHeavy = 256;
constexpr int kCcSlice = 2048;

__device__ __forceinline__ int32_t shfl(int32_t x, int src) {
    return __builtin_amdgcn_ds_bpermute(src << 2, x);
}
__device__ __forceinline__ int64_t shfl(int64_t x, int src) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(src << 2, (int)(uint32_t)(uint64_t)x);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute(src << 2, (int)(uint32_t)((uint64_t)x >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Slices of the heavy lists and the vertex of largest degree (top: (degree
// << 32) | ~vertex, the smallest id among equals); built once per graph.
// *count ends as the number of slices the graph needs, even past cap (then
// only cap are kept).
__global__ __launch_bounds__(256) void k_cc_tasks(const int64_t *__restrict__ off, int64_t nv,
                                                  td_task *__restrict__ tasks,
                                                  unsigned long long *__restrict__ count, int64_t cap,
                                                  unsigned long long *__restrict__ top) {
    unsigned long long best = 0;
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv;
         v += (int64_t)gridDim.x * blockDim.x) {
        const int64_t b = off[v], e = off[v + 1];
        const unsigned long long d = (unsigned long long)(e - b < 0x7fffffff ? e - b : 0x7fffffff);
        const unsigned long long key = (d << 32) | (0xffffffffULL - (unsigned long long)v);
        best = key > best ? key : best;
        if (e - b < kCcHeavy) continue;
        const int64_t n = (e - b + kCcSlice - 1) / kCcSlice;
        const int64_t at = (int64_t)atomicAdd(count, (unsigned long long)n);
        for (int64_t i = 0; i < n && at + i < cap; ++i) {
            td_task t;
            t.beg = b + i * kCcSlice;
            t.end = t.beg + kCcSlice < e ? t.beg + kCcSlice : e;
            t.src = (int32_t)v;
            t.pad = 0;
            tasks[at + i] = t;
        }
    }
    // one atomic per workgroup: all meet on one address
    __shared__ unsigned long long red[4];
    best = wave_max(best);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; ++w) best = red[w] > best ? red[w] : best;
        atomicMax(top, best);
    }
}

// First pass: the lowest neighbour id of each of a wave's 64 light lists (lane
// i's starts at number s of the group's `total` entries, has d, and entry q is
// cols[base_k + q]).  As in the later passes every lane takes an entry whatever
// the degrees, but the owner search and the segmented minimum there are 14
// lane exchanges for 64 entries, and the LDS unit was what bound the pass.
// Here a bitmap marks where lists start, an entry's list is the count of bits
// up to it, and each list has a slot for its minimum: four LDS operations.
// Scale 18: 37 -> 24 us a pass, scale 23: 536 -> 457 (1.0 GB).  With the owner
// search kept, more rounds in flight gained nothing at scale 23.
constexpr int kFirstRounds = 4;  // rounds of 64 entries in flight
struct first_lds {
    uint64_t start[kCcHeavy];  // bit q: a list starts at entry q
    int64_t base[64];          // by rank among the lists that are not empty
    int32_t low[64];
};

__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

__device__ __forceinline__ int32_t first_min(first_lds &f, const int32_t *cols, int32_t d, int32_t s,
                                             int32_t total, int64_t base_k, int32_t mine) {
    const int lane = lane_id();
    const int32_t nwords = (total + 63) >> 6;  // d < kCcHeavy: at most kCcHeavy
    const int rank = __popcll(__ballot(d > 0) & ((1ULL << lane) - 1));
    for (int32_t w = lane; w < nwords; w += 64) f.start[w] = 0;
    wave_lds_order();
    if (d > 0) {
        atomicOr((unsigned long long *)&f.start[s >> 6], 1ULL << (s & 63));
        f.base[rank] = base_k;
        f.low[rank] = mine;
    }
    wave_lds_order();
    const uint64_t upto = (2ULL << lane) - 1;  // this lane's entry and those before
    int before = -1;  // rank of the list that the entry before the round is in
    for (int32_t t = 0; t < total; t += 64 * kFirstRounds) {
        int o[kFirstRounds];
        int32_t c[kFirstRounds];
#pragma unroll
        for (int r = 0; r < kFirstRounds; ++r) {
            const int32_t w = (t >> 6) + r, q = t + 64 * r + lane;
            const uint64_t m = w < nwords ? f.start[w] : 0;
            o[r] = before + __popcll(m & upto);
            before += __popcll(m);
            // past the end: the last entry again
            c[r] = __builtin_nontemporal_load(cols + f.base[o[r]] + (q < total ? q : total - 1));
        }
#pragma unroll
        for (int r = 0; r < kFirstRounds; ++r) atomicMin(&f.low[o[r]], c[r]);
    }
    wave_lds_order();
    const int32_t got = d > 0 ? f.low[rank] : mine;
    wave_lds_order();  // the slots are rewritten by the next group
    return got;
}

// Vertices from which the second pass lowers roots; in smaller graphs the tenth
// is the first to.  Where a pass brings many labels down at once, most of their
// vertices find the root not yet lowered, and the atomics take up to 0.3 ms:
// more than the passes they save on a small graph that needs few.  Erdos-Renyi
// graphs of mean degree 16, a run without and with it from the second pass on:
// 1 M vertices 414 and 656 us, 2 M 773 and 1060, 4 M 1772 and 1729, 8 M 3602 and
// 3320; eight such graphs side by side, 4.2 M vertices in all 3150 and 2752 us,
// 16 M 15.1 and 10.8 ms.  Of mean degree 3, 1 M vertices in nine passes: 374 us,
// and 472 with it from the sixth on.  Graphs that take more have many to come.
constexpr int64_t kRootsDownNv = (int64_t)1 << 22;

// Edge pass.  Units [0, ntasks) are heavy slices; unit ntasks + g is
// the vertex group [64g, 64g + 64), whose light lists are consecutive in
// cols (heavy lists between them are skipped).  The group's light edges are
// numbered q = 0..T-1 (light vertex i owns q in [s_i, s_i + d_i)) and taken
// 64 at a time, one per lane, so every lane loads whatever the degrees (the
// first pass: first_min):
//   owner   o(q) = the last i with s_i <= q   (binary search over lanes)
//   edge    k    = off[base + o] + q - s_o
//   label   l    = comp[cols[k]]
// Owners are non-decreasing across the lanes of a chunk, so a suffix min
// restricted to equal owners leaves the chunk's min for owner i in the
// lane where i's run starts, max(s_i - t, 0), which lane i reads.
// In the first pass the neighbour's id stands in for its label: every label
// is still its vertex's id when the pass starts, and a pass may read a
// neighbour's label from before that neighbour's own update in the same pass,
// so this is one of the pass's own outcomes, with no label gathered.  Later
// passes skip the vertices labelled g and, with lower_roots, lower the roots of
// the labels that go (see the top of the file).
template <bool FIRST>
__global__ __launch_bounds__(256) void k_cc_hook(const int64_t *__restrict__ off,
                                                 const int32_t *__restrict__ cols, int32_t *comp,
                                                 int64_t nv, const td_task *__restrict__ tasks,
                                                 int64_t ntasks, bool lower_roots,
                                                 cc_state *__restrict__ st,
                                                 unsigned long long *__restrict__ labels_read,
                                                 unsigned long long *__restrict__ edge_bytes) {
    if (!FIRST && st->done) return;
    __shared__ first_lds lds[FIRST ? 4 : 1];
    const int lane = threadIdx.x & 63;
    const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
    const int64_t nunits = ntasks + (nv + 63) / 64;
    const int32_t g = FIRST ? -1 : st->g;
    if (blockIdx.x == 0 && threadIdx.x == 0) st->t_hook = wall_clock64();
    bool ch = false;
    int32_t offer = 0x7fffffff;  // lowest label seen beside one labelled g
    // nbytes: algorithmic bytes besides the 8 B (column id + label) of each
    // label read
    unsigned long long nread = 0, nbytes = 0;
    for (int64_t u = wave; u < nunits; u += nwaves) {
        if (u < ntasks) {
            const int64_t beg = tasks[u].beg, end = tasks[u].end;
            const int32_t src = tasks[u].src;
            int32_t mine = 0x7fffffff;
            if (!FIRST) {
                mine = lane_bcast(comp[src], 0);
                if (mine == g) continue;
            }
            uint32_t m = 0xffffffffu;
            bool saw = false;
            for (int64_t k0 = beg; k0 < end; k0 += 4 * 64) {
                int32_t c[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t k = k0 + r * 64 + lane;
                    c[r] = __builtin_nontemporal_load(cols + (k < end ? k : end - 1));
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (k0 + r * 64 + lane >= end) continue;
                    const uint32_t l = FIRST ? (uint32_t)c[r] : (uint32_t)comp[c[r]];
                    m = l < m ? l : m;
                    saw |= !FIRST && (int32_t)l == g;
                    if (FIRST)
                        nbytes += 4;
                    else
                        ++nread;
                }
                // g is lower than its own label: it takes g and reads no more
                if (!FIRST && g < mine && __ballot(saw)) break;
            }
            m = (uint32_t)wave_min(m);
            if (!FIRST && __ballot(saw) && mine < offer) offer = mine;
            // a slice is never empty, so m is a label; checked all the same
            if (lane == 0 && m != 0xffffffffu && (int32_t)m < comp[src]) {
                if ((int32_t)m < atomicMin(comp + src, (int32_t)m)) ch = true;
                if (lower_roots && (int32_t)m < comp[mine]) atomicMin(comp + mine, (int32_t)m);
            }
            continue;
        }
        const int64_t v = (u - ntasks) * 64 + lane;
        int64_t b = 0, e = 0;
        int32_t mine = 0x7fffffff;
        if (v < nv) {
            mine = FIRST ? (int32_t)v : comp[v];
            if (!FIRST) nbytes += 4;
            if (FIRST || mine != g) {
                b = off[v];
                e = off[v + 1];
                nbytes += 8;
            }
        }
        const int32_t d = e - b < kCcHeavy ? (int32_t)(e - b) : 0;
        if (!FIRST && !__ballot(d > 0)) continue;
        const int32_t s_end = wave_incl_scan32(d);
        const int32_t s = s_end - d;
        const int32_t total = __builtin_amdgcn_readlane(s_end, 63);
        const int64_t base_k = b - s;  // k = base_k of the owner + q
        int32_t acc = mine;
        if constexpr (FIRST) {
            if (total > 0) acc = first_min(lds[threadIdx.x >> 6], cols, d, s, total, base_k, mine);
            if (lane == 0) nbytes += 4 * (unsigned long long)total;
            const bool down = acc < mine;
            if (down) comp[v] = acc;
            ch |= down;
            continue;
        }
        for (int32_t t = 0; t < total; t += 64) {
            const int32_t q = t + lane;
            const int32_t qa = q < total ? q : total - 1;
            int o = 0;
#pragma unroll
            for (int step = 32; step; step >>= 1)
                if (shfl(s, o + step) <= qa) o += step;
            const int64_t k = shfl(base_k, o) + qa;
            // one past the owner's last lane in this chunk
            const int32_t run_end = min(shfl(s_end, o) - t, 64);
            const int32_t lo = shfl(acc, o);
            int32_t m = 0x7fffffff;
            if (q < total && lo != g) {  // at g the owner reads no more
                m = comp[__builtin_nontemporal_load(cols + k)];
                ++nread;
                if (m == g && lo < offer) offer = lo;
            }
#pragma unroll
            for (int step = 1; step < 64; step <<= 1) {
                const int32_t other = shfl(m, (lane + step) & 63);
                if (lane + step < run_end && other < m) m = other;
            }
            const bool mine_here = d > 0 && s < t + 64 && s_end > t;
            const int32_t got = shfl(m, mine_here ? (s > t ? s - t : 0) : lane);
            if (mine_here && acc != g && got < acc) acc = got;
        }
        const bool down = acc < mine;
        if (down) {
            comp[v] = acc;
            if (lower_roots && acc < comp[mine]) atomicMin(comp + mine, acc);
        }
        ch |= down;
    }
    if (!FIRST) {
        offer = (int32_t)wave_min((unsigned long long)(uint32_t)offer);
        if (lane == 0 && offer < g && offer < atomicMin(comp + g, offer)) ch = true;
    }
    if (__ballot(ch) && lane == 0) st->changed = 1;
    nbytes = wave_sum(nbytes + 8 * nread);
    nread = wave_sum(nread);
    const int slot = (blockIdx.x % kSlots) * kLine;
    if (lane == 0 && nread) atomicAdd(&labels_read[slot], nread);
    if (lane == 0 && nbytes) atomicAdd(&edge_bytes[slot], nbytes);
}

// Between the first pass and the second: every vertex's label meets that of
// its neighbour of largest degree (the head index, in search ids; perm maps
// them, or they are graph ids).  Labels are roots here, so the higher root
// takes the lower label, which carries every vertex labelled with it at the
// next shortcut.  The first pass leaves RMAT's large component in many trees,
// one per vertex with no lower neighbour, and the second pass then read 62% of
// the labels at scale 23; the heads join nearly all of them for one gather a
// vertex.
__global__ void k_cc_link(const uint64_t *__restrict__ head, const int32_t *__restrict__ perm,
                          int64_t n, int32_t *comp) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int32_t h = (int32_t)(uint32_t)head[i];
        if (h < 0) continue;
        const int32_t a = comp[perm ? perm[i] : (int32_t)i], b = comp[perm ? perm[h] : h];
        if (a == b) continue;
        const int32_t hi = a > b ? a : b, lo = a > b ? b : a;
        if (comp[hi] > lo) atomicMin(comp + hi, lo);
    }
}

// Shortcut (:74-78): each label becomes its root; the roots (label[v] == v,
// the components, one per label, :84-101) are counted on the way.  A label is
// never above its vertex's id, so chains strictly descend to a root; a label
// outside [0, v] stops the chase and sets *bad instead of being followed.
__global__ __launch_bounds__(256) void k_cc_shortcut(int32_t *comp, int64_t nv,
                                                     cc_state *__restrict__ st, int close_pass,
                                                     unsigned long long *__restrict__ roots) {
    if (st->done) return;
    if (close_pass && blockIdx.x == 0 && threadIdx.x == 0)
        st->t_passes += wall_clock64() - st->t_hook;
    unsigned long long n = 0;
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv;
         v += (int64_t)gridDim.x * blockDim.x) {
        const int32_t c0 = comp[v];
        int32_t c = c0;
        bool ok = c >= 0 && c <= v;
        while (ok) {
            const int32_t cc = comp[c];
            if (cc == c) break;
            ok = cc >= 0 && cc < c;
            if (ok) c = cc;
        }
        if (!ok) {
            st->bad = 1;
            c = c0;
        }
        if (c != c0) comp[v] = c;
        n += c == (int32_t)v;
    }
    n = wave_sum(n);
    if (roots && (threadIdx.x & 63) == 0 && n)
        atomicAdd(&roots[(blockIdx.x % kSlots) * kLine], n);
}

// Close a pass (one wave): it was the last when it changed nothing (or met a
// label out of range), and then the result goes to host memory; otherwise the
// next pass's g is set and the root counters are cleared.
__global__ __launch_bounds__(64) void k_cc_close(const int32_t *__restrict__ comp, int32_t hub,
                                                 cc_state *__restrict__ st,
                                                 unsigned long long *__restrict__ roots,
                                                 const unsigned long long *__restrict__ labels_read,
                                                 const unsigned long long *__restrict__ edge_bytes,
                                                 cc_result *__restrict__ res, uint32_t seq) {
    if (st->done) return;
    const int l = lane_id();
    const bool done = !st->changed || st->bad;
    const unsigned long long n = wave_sum(roots[l * kLine]);
    const unsigned long long r = wave_sum(labels_read[l * kLine]);
    const unsigned long long e = wave_sum(edge_bytes[l * kLine]);
    roots[l * kLine] = 0;
    if (l != 0) return;
    st->iters += 1;
    st->changed = 0;
    st->g = comp[hub];
    st->done = done;
    if (!done) return;
    res->iters = st->iters;
    res->components = (int64_t)n;
    res->labels_read = (int64_t)r;
    res->edge_bytes = (int64_t)e;
    res->ticks = wall_clock64() - st->t_start;
    res->pass_ticks = st->t_passes;
    res->bad = st->bad;
    __threadfence_system();
    __hip_atomic_store(&res->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace
}  // namespace bd

using namespace bd;

extern "C" int bd_cc_run(bd_ctx *c, bd_cc_stats *out) {
    if (!c) return BD_EINVAL;
    if (!c->d_off) return set_err(c, BD_ESTATE, "no graph loaded");
    BD_HIP(c, hipSetDevice(c->device));
    const int64_t nv = c->nv, nw = (nv + 63) / 64;
    int rc;
    if (!c->d_comp && (rc = dev_alloc(c, (void **)&c->d_comp, sizeof(int32_t) * (nv + 1), "labels")))
        return rc;
    // the state, then three kSlots x kLine counter blocks: components, labels
    // read, algorithmic bytes of the edge passes
    constexpr int kBlockWords = kSlots * kLine;
    static_assert(sizeof(cc_state) <= sizeof(unsigned long long) * kLine, "state line");
    static_assert(sizeof(cc_result) <= sizeof(host_state::cc), "result's place");
    if (!c->d_cc_flag &&
        (rc = dev_alloc(c, (void **)&c->d_cc_flag,
                        sizeof(unsigned long long) * (kLine + 3 * kBlockWords), "label flags")))
        return rc;
    c->have_cc = false;
    cc_state *st = (cc_state *)c->d_cc_flag;
    unsigned long long *count = (unsigned long long *)c->d_cc_flag + kLine;
    unsigned long long *nread = count + kBlockWords;
    unsigned long long *ebytes = nread + kBlockWords;
    cc_result *res = (cc_result *)c->h_cc;
    const dim3 grid(grid_for(c, nv, 256)), block(256);
    if (c->cc_ntasks < 0) {
        // slices of the long lists, once per graph (like the graph's own
        // indexes, outside the timed run; its time and memory are reported)
        BD_HIP(c, hipEventRecord(c->ev[0], c->stream));
        const int64_t cap = c->nnz / kCcSlice + c->nnz / kCcHeavy + 1;
        dev_free(c, c->d_cc_tasks);  // left by a build that failed part-way
        c->d_cc_tasks = nullptr;
        if ((rc = dev_alloc(c, (void **)&c->d_cc_tasks, sizeof(td_task) * cap, "component slices")))
            return rc;
        BD_HIP(c, hipMemsetAsync(count, 0, 2 * sizeof(unsigned long long), c->stream));
        hipLaunchKernelGGL(k_cc_tasks, dim3(std::min<int64_t>(grid.x, c->cu_count)), block, 0,
                           c->stream, c->d_off, nv, c->d_cc_tasks, count, cap, count + 1);
        BD_HIP(c, hipGetLastError());
        unsigned long long h[2] = {0, 0};
        BD_HIP(c, hipMemcpyAsync(h, count, sizeof(h), hipMemcpyDeviceToHost, c->stream));
        BD_HIP(c, hipEventRecord(c->ev[1], c->stream));
        BD_HIP(c, hipStreamSynchronize(c->stream));
        if ((int64_t)h[0] > cap) return set_err(c, BD_EHIP, "component slices overflow");
        float pms = 0;
        BD_HIP(c, hipEventElapsedTime(&pms, c->ev[0], c->ev[1]));
        c->cc_prep_ms = pms;
        c->cc_prep_bytes = (int64_t)(sizeof(td_task) * cap);
        c->cc_hub = (int32_t)(0xffffffffULL - (h[1] & 0xffffffffULL));
        c->cc_ntasks = (int64_t)h[0];
    }
    const dim3 hook_grid(grid_for(c, (c->cc_ntasks + nw) * 64, 256));
    const auto host_start = std::chrono::steady_clock::now();
    const uint32_t seq = res->seq + 1;
    hipLaunchKernelGGL(k_cc_init, grid, block, 0, c->stream, c->d_comp, nv, st, count,
                       3 * kBlockWords);
    // passes queued at a time: three (most graphs take two to four, and one that
    // is not needed returns at once), then two
    int64_t queued = 0;
    for (int chunk = 3;; chunk = 2) {
        if (queued > nv + 4) return set_err(c, BD_EHIP, "components did not converge");
        for (int k = 0; k < chunk; ++k, ++queued) {
            const bool lower_roots = queued >= (nv < kRootsDownNv ? 9 : 1);
            hipLaunchKernelGGL((queued == 0 ? k_cc_hook<true> : k_cc_hook<false>), hook_grid, block,
                               0, c->stream, (const int64_t *)c->d_off, (const int32_t *)c->d_cols,
                               c->d_comp, nv, (const td_task *)c->d_cc_tasks, c->cc_ntasks,
                               lower_roots, st, nread, ebytes);
            if (queued == 0 && c->d_head) {
                hipLaunchKernelGGL(k_cc_shortcut, grid, block, 0, c->stream, c->d_comp, nv, st, 1,
                                   (unsigned long long *)nullptr);
                hipLaunchKernelGGL(k_cc_link, grid, block, 0, c->stream,
                                   (const uint64_t *)c->d_head, (const int32_t *)c->d_perm,
                                   c->d_perm ? c->nv_active : nv, c->d_comp);
            }
            hipLaunchKernelGGL(k_cc_shortcut, grid, block, 0, c->stream, c->d_comp, nv, st,
                               queued == 0 && c->d_head ? 0 : 1, count);
            hipLaunchKernelGGL(k_cc_close, dim3(1), dim3(64), 0, c->stream,
                               (const int32_t *)c->d_comp, c->cc_hub, st, count,
                               (const unsigned long long *)nread,
                               (const unsigned long long *)ebytes, res, seq);
        }
        BD_HIP(c, hipGetLastError());
        if ((rc = wait_host_flag(c, &res->seq, seq))) return rc;
        if (__atomic_load_n(&res->seq, __ATOMIC_ACQUIRE) == seq) break;
    }
    if (res->bad) return set_err(c, BD_EHIP, "component label out of range");
    const double host_ms = std::chrono::duration<double, std::milli>(
                               std::chrono::steady_clock::now() - host_start)
                               .count();
    c->have_cc = true;
    if (out) {
        const double ms = (double)res->ticks / (double)c->wall_khz;
        out->num_components = res->components;
        out->num_iters = res->iters;
        out->ms = ms > 0 ? ms : host_ms;
        out->pass_ms = std::min(out->ms, (double)res->pass_ticks / (double)c->wall_khz);
        out->labels_read = res->labels_read;
        out->edge_bytes = res->edge_bytes;
        out->pass_launches = res->iters;
        out->prep_ms = c->cc_prep_ms;
        out->prep_bytes = c->cc_prep_bytes;
    }
    return BD_OK;
}

extern "C" int bd_cc_fetch(bd_ctx *c, int64_t *labels) {
    if (!c || !labels) return BD_EINVAL;
    if (!c->have_cc) return set_err(c, BD_ESTATE, "components have not run");
    BD_HIP(c, hipSetDevice(c->device));
    return carry_copy(c, carry::i32_i64, labels, c->d_comp, c->nv);
}

// components::check (components.cc:152-202) on the host, from downloaded
// copies: one source per label (the last vertex carrying it); a BFS from it
// must meet only that label, and every vertex must be reached.
extern "C" int bd_cc_check(bd_ctx *c, int *ok) {
    if (!c || !ok) return BD_EINVAL;
    if (!c->have_cc) return set_err(c, BD_ESTATE, "components have not run");
    const int64_t nv = c->nv;
    std::vector<int64_t> off(nv + 1), label(nv);
    std::vector<int32_t> cols(c->nnz);
    int rc = bd_graph_download(c, off.data(), cols.data());
    if (!rc) rc = bd_cc_fetch(c, label.data());
    if (rc) return rc;
    std::vector<int64_t> source(nv, -1), queue;
    std::vector<char> visited(nv, 0);
    bool good = true;
    for (int64_t v = 0; v < nv && good; ++v) {
        if (label[v] < 0 || label[v] >= nv)
            good = false;
        else
            source[label[v]] = v;
    }
    queue.reserve(nv);
    for (int64_t l = 0; l < nv && good; ++l) {
        if (source[l] < 0) continue;
        queue.clear();
        visited[source[l]] = 1;
        queue.push_back(source[l]);
        for (size_t h = 0; h < queue.size() && good; ++h) {
            const int64_t u = queue[h];
            for (int64_t e = off[u]; e < off[u + 1]; ++e) {
                const int64_t w = cols[e];
                if (label[w] != l) {
                    good = false;
                    break;
                }
                if (!visited[w]) {
                    visited[w] = 1;
                    queue.push_back(w);
                }
            }
        }
    }
    for (int64_t v = 0; v < nv && good; ++v)
        if (!visited[v]) good = false;
    *ok = good ? 1 : 0;
    return BD_OK;
}
