// bd_readout.hip -- results carried to the caller's memory.
//
// A caller's array is ordinary memory, mostly fresh: its pages are mapped as
// they are first written, at 4 to 8 GB/s with the one thread of a plain copy
// (64 MB: 7.3 ms, of which the transfer is 1.2), and int64 ids and int32
// depths move two to four times the bytes that they hold.  So kernels write a
// result in its narrow form (a byte a depth, 4 bytes an id) into a ring of
// pinned chunks, and a few host threads widen chunks into the caller's pages
// while later ones are on their way.
#include <string.h>

#include <algorithm>
#include <atomic>
#include <new>
#include <thread>
#include <vector>

#include "bd_cpus.h"
#include "bd_internal.h"

namespace bd {

namespace {

constexpr int64_t kChunkBytes = 1 << 20;  // of the narrow form
constexpr int kUnits = 4;                 // pieces of a chunk, each widened by one thread
// Outputs under this are widened by the caller's thread alone: starting a
// thread takes about 15 us, as long as writing 100 KB of fresh pages.
constexpr int64_t kThreadBytes = 2 << 20;
// Helpers: 64 MB of fresh pages take 4.6 ms on one thread, 2.4 on two, 1.3 on
// four, 0.8 to 1.1 on eight and no less on twelve.
constexpr int kMaxHelpers = 7;

// n 4-byte words to host memory, 16 bytes a lane (src and out lie on 16 bytes:
// allocations, from multiples of a chunk).
__global__ __launch_bounds__(256) void k_to_host(const uint32_t *__restrict__ src, int64_t n,
                                                 uint32_t *__restrict__ out) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = t; i < n / 4; i += stride) ((uint4 *)out)[i] = ((const uint4 *)src)[i];
    if (t < n % 4) out[n - 1 - t] = src[n - 1 - t];
}

// n 4-byte words from host memory.
__global__ __launch_bounds__(256) void k_from_host(const uint32_t *__restrict__ src, int64_t n,
                                                   uint32_t *__restrict__ dst) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

size_t narrow_size(carry k) { return k == carry::u8_i32 ? 1 : k == carry::i64_i64 ? 8 : 4; }
size_t wide_size(carry k) { return k == carry::u8_i32 || k == carry::i32_i32 ? 4 : 8; }

// n elements of the narrow form, widened.  A byte of 255 is -1.
void widen(carry k, const void *src, void *dst, int64_t n) {
    if (k == carry::u8_i32) {
        const uint8_t *s = (const uint8_t *)src;
        int32_t *d = (int32_t *)dst;
        for (int64_t i = 0; i < n; ++i) d[i] = s[i] == 255 ? -1 : (int32_t)s[i];
    } else if (k == carry::i32_i64) {
        const int32_t *s = (const int32_t *)src;
        int64_t *d = (int64_t *)dst;
        for (int64_t i = 0; i < n; ++i) d[i] = s[i];
    } else {
        memcpy(dst, src, n * wide_size(k));
    }
}

// Helpers spin while their chunk is on its way, so they may be half of the CPUs
// that the process has the use of.  Those that its quota leaves are read once a
// context (7 to 23 us).
int helper_threads(bd_ctx *c) {
    if (c->cpus == 0) c->cpus = usable_cpus();
    return std::min(kMaxHelpers, std::min(c->cpus, affinity_cpus()) / 2);
}

// The pinned ring, at least `bytes` and at most kRing chunks, and its events.
// BD_ENOMEM when it cannot be pinned: results then go the plain way.
int ensure_ring(bd_ctx *c, int64_t bytes) {
    if (c->ring_bytes < bytes) {
        // what a small graph needs is pinned in no time; a whole ring takes about 2 ms
        int64_t want = 64 << 10;
        while (want < bytes) want *= 2;
        want = std::min<int64_t>(want, kRing * kChunkBytes);
        if (c->h_ring) (void)hipHostFree(c->h_ring);
        c->h_ring = nullptr;
        c->ring_bytes = 0;
        const hipError_t e = hipHostMalloc(&c->h_ring, want, hipHostMallocMapped | hipHostMallocCoherent);
        if (e != hipSuccess) {
            c->h_ring = nullptr;
            (void)hipGetLastError();
            return BD_ENOMEM;
        }
        c->ring_bytes = want;
    }
    if (bytes > kChunkBytes)
        for (auto &ev : c->ring_ev)
            if (!ev) BD_HIP(c, hipEventCreateWithFlags(&ev, hipEventDisableTiming));
    return BD_OK;
}

// Without the ring: a chunk at a time through device memory and a plain copy.
int carry_plain(bd_ctx *c, carry kind, void *dst, int64_t n, const carry_part &part) {
    const int64_t ns = (int64_t)narrow_size(kind), ws = (int64_t)wide_size(kind);
    const int64_t per = std::min<int64_t>(n, kChunkBytes / ns);
    struct buffers {
        bd_ctx *c;
        void *dev = nullptr;
        char *host = nullptr;
        ~buffers() {
            dev_free(c, dev);
            delete[] host;
        }
    } b{c};
    int rc;
    if ((rc = dev_alloc(c, &b.dev, per * ns, "result chunk"))) return rc;
    if (ns != ws && !(b.host = new (std::nothrow) char[per * ns]))
        return set_err(c, BD_ENOMEM, "result chunk");
    for (int64_t first = 0; first < n; first += per) {
        const int64_t cnt = std::min(per, n - first);
        char *to = (char *)dst + first * ws;
        if ((rc = part(first, cnt, b.dev)) ||
            (rc = copy_sync(c, b.host ? b.host : to, b.dev, cnt * ns, hipMemcpyDeviceToHost)))
            return rc;
        if (b.host) widen(kind, b.host, to, cnt);
    }
    return BD_OK;
}

}  // namespace

int carry_out(bd_ctx *c, carry kind, void *dst, int64_t n, const carry_part &part) {
    if (n <= 0) return BD_OK;
    const int64_t ns = (int64_t)narrow_size(kind), ws = (int64_t)wide_size(kind);
    const int64_t per = kChunkBytes / ns, chunks = (n + per - 1) / per;
    int rc;
    if ((rc = ensure_ring(c, std::min<int64_t>(n * ns, kRing * kChunkBytes))))
        return rc == BD_ENOMEM ? carry_plain(c, kind, dst, n, part) : rc;
    char *ring = (char *)c->h_ring;
    if (chunks == 1) {
        if ((rc = part(0, n, ring))) return rc;
        BD_HIP(c, hipStreamSynchronize(c->stream));
        if (n * ws < kThreadBytes) {
            widen(kind, ring, dst, n);
            return BD_OK;
        }
    }
    // unit u is piece u % kUnits of chunk u / kUnits; chunk k lies in slot
    // k % kRing, which it may take once the units of chunk k - kRing are done
    const int64_t nunits = chunks * kUnits, up = per / kUnits;
    std::atomic<int64_t> next{0}, ready{chunks == 1 ? 1 : 0};
    std::atomic<bool> stop{false};
    std::vector<std::atomic<int>> left(chunks);
    for (auto &x : left) x.store(kUnits, std::memory_order_relaxed);
    auto do_unit = [&](int64_t u) {
        const int64_t k = u / kUnits, at = (u - k * kUnits) * up;
        const int64_t cnt = std::min(up, std::min(per, n - k * per) - at);
        if (cnt > 0)
            widen(kind, ring + (k % kRing) * kChunkBytes + at * ns, (char *)dst + (k * per + at) * ws, cnt);
        left[k].fetch_sub(1, std::memory_order_release);
    };
    auto help = [&]() {
        for (;;) {
            const int64_t u = next.fetch_add(1, std::memory_order_relaxed);
            if (u >= nunits) return;
            for (unsigned spin = 0; ready.load(std::memory_order_acquire) <= u / kUnits; ++spin) {
                if (stop.load(std::memory_order_relaxed)) return;
                if (spin < 64)
                    __builtin_ia32_pause();
                else
                    std::this_thread::yield();
            }
            do_unit(u);
        }
    };
    int64_t issued = chunks == 1 ? 1 : 0;
    auto issue = [&]() -> int {
        const int64_t k = issued;
        const int r = part(k * per, std::min(per, n - k * per), ring + (k % kRing) * kChunkBytes);
        if (r) return r;
        BD_HIP(c, hipEventRecord(c->ring_ev[k % kRing], c->stream));
        ++issued;
        return BD_OK;
    };
    std::vector<std::thread> helpers;
    while (!rc && issued < std::min<int64_t>(chunks, kRing)) rc = issue();
    if (!rc && n * ws >= kThreadBytes) {
        const int64_t nh = std::min<int64_t>(helper_threads(c), nunits - 1);
        try {
            helpers.reserve(nh);
            for (int64_t i = 0; i < nh; ++i) helpers.emplace_back(help);
        } catch (...) {
            // no more threads to be had: those there are, and this one, do it all
        }
    }
    int64_t held = -1;  // a unit this thread took before its chunk was ready
    while (!rc) {
        const int64_t rd = ready.load(std::memory_order_relaxed);
        if (rd < issued) {
            const hipError_t e = hipEventQuery(c->ring_ev[rd % kRing]);
            if (e == hipSuccess) {
                ready.store(rd + 1, std::memory_order_release);
                continue;
            }
            (void)hipGetLastError();
            if (e != hipErrorNotReady) rc = hip_err(c, e, "hipEventQuery");
        }
        if (!rc && issued < chunks &&
            left[issued - kRing].load(std::memory_order_acquire) == 0) {
            rc = issue();
            continue;
        }
        if (held < 0 && next.load(std::memory_order_relaxed) < std::min(nunits, rd * kUnits)) {
            held = next.fetch_add(1, std::memory_order_relaxed);
            if (held >= nunits) held = -1;
        }
        if (held >= 0 && held / kUnits < rd) {
            do_unit(held);
            held = -1;
            continue;
        }
        if (held < 0 && rd == chunks && next.load(std::memory_order_relaxed) >= nunits) break;
        __builtin_ia32_pause();
    }
    if (rc) stop.store(true);
    for (auto &t : helpers) t.join();
    if (rc) (void)hipStreamSynchronize(c->stream);  // nothing writes the ring any more
    return rc;
}

int carry_copy(bd_ctx *c, carry kind, void *dst, const void *src, int64_t n) {
    const int64_t ns = (int64_t)narrow_size(kind);
    return carry_out(c, kind, dst, n, [&](int64_t first, int64_t count, void *out) -> int {
        return queue_to_host(c, (const char *)src + first * ns, count * ns / 4, out);
    });
}

int queue_to_host(bd_ctx *c, const void *src, int64_t words, void *out) {
    hipLaunchKernelGGL(k_to_host, dim3(grid_for(c, (words + 3) / 4, 256)), dim3(256), 0, c->stream,
                       (const uint32_t *)src, words, (uint32_t *)out);
    BD_HIP(c, hipGetLastError());
    return BD_OK;
}

int host_ring(bd_ctx *c, int64_t bytes, void **p) {
    const int rc = ensure_ring(c, bytes);
    *p = c->h_ring;
    return rc;
}

int stage_in(bd_ctx *c, void *dst, std::initializer_list<host_piece> pieces) {
    size_t total = 0;
    for (const host_piece &x : pieces) total += x.bytes;
    int rc = BD_ENOMEM;
    void *ring;
    if (total <= (size_t)kChunkBytes) {
        // what a call that failed half-way queued may still read the ring
        BD_HIP(c, hipStreamSynchronize(c->stream));
        if ((rc = host_ring(c, (int64_t)total, &ring)) && rc != BD_ENOMEM) return rc;
    }
    if (rc) {  // too large, or nothing to be pinned
        char *at = (char *)dst;
        for (const host_piece &x : pieces) {
            if (x.bytes)
                BD_HIP(c, hipMemcpyAsync(at, x.p, x.bytes, hipMemcpyHostToDevice, c->stream));
            at += x.bytes;
        }
        return BD_OK;
    }
    char *at = (char *)ring;
    for (const host_piece &x : pieces) {
        if (x.bytes) memcpy(at, x.p, x.bytes);
        at += x.bytes;
    }
    hipLaunchKernelGGL(k_from_host, dim3(grid_for(c, (int64_t)total / 4, 256)), dim3(256), 0,
                       c->stream, (const uint32_t *)ring, (int64_t)total / 4, (uint32_t *)dst);
    BD_HIP(c, hipGetLastError());
    return BD_OK;
}

void free_ring(bd_ctx *c) {
    if (c->h_ring) (void)hipHostFree(c->h_ring);
    c->h_ring = nullptr;
    c->ring_bytes = 0;
    for (auto &ev : c->ring_ev) {
        if (ev) (void)hipEventDestroy(ev);
        ev = nullptr;
    }
}

}  // namespace bd
