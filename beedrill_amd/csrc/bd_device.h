// bd_device.h -- wavefront helpers shared by the search kernels (64-lane
// waves of CDNA).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bd {

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

// Wave-wide scans and reductions with DPP lane moves (no LDS round trips):
// row_shr 1, 2, 4, 8 scan each 16-lane row, then row_bcast 15 and 31 carry
// the row totals into the rows above.  Lanes a move cannot reach read 0.
// Every lane of the wave must be active; results are inclusive (lane i
// holds the combination of lanes 0..i), reductions read lane 63.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint64_t dpp_move64(uint64_t x) {
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)x, CTRL, ROW_MASK, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(x >> 32), CTRL, ROW_MASK, 0xf, true);
    return ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo;
}

template <typename Op>
__device__ __forceinline__ uint64_t wave_scan64(uint64_t x, Op op) {
    x = op(x, dpp_move64<0x111, 0xf>(x));  // row_shr:1
    x = op(x, dpp_move64<0x112, 0xf>(x));  // row_shr:2
    x = op(x, dpp_move64<0x114, 0xf>(x));  // row_shr:4
    x = op(x, dpp_move64<0x118, 0xf>(x));  // row_shr:8
    x = op(x, dpp_move64<0x142, 0xa>(x));  // row_bcast:15 into rows 1, 3
    x = op(x, dpp_move64<0x143, 0xc>(x));  // row_bcast:31 into rows 2, 3
    return x;
}

__device__ __forceinline__ uint64_t lane63(uint64_t x) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, 63);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), 63);
    return ((uint64_t)hi << 32) | lo;
}

// x from lane `src`, which must be the same in every lane (a scalar read,
// no LDS round trip).
__device__ __forceinline__ int32_t lane_bcast(int32_t x, int src) {
    return __builtin_amdgcn_readlane(x, src);
}
__device__ __forceinline__ int64_t lane_bcast(int64_t x, int src) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(uint64_t)x, src);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)((uint64_t)x >> 32), src);
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

__device__ __forceinline__ int32_t wave_incl_scan32(int32_t x) {
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, true);
    return x;
}

__device__ __forceinline__ long long wave_incl_scan(long long x) {
    return (long long)wave_scan64((uint64_t)x, [](uint64_t p, uint64_t q) { return p + q; });
}

__device__ __forceinline__ unsigned long long wave_sum(unsigned long long x) {
    return lane63(wave_scan64(x, [](uint64_t p, uint64_t q) { return p + q; }));
}

__device__ __forceinline__ unsigned long long wave_max(unsigned long long x) {
    return lane63(wave_scan64(x, [](uint64_t p, uint64_t q) { return p > q ? p : q; }));
}

__device__ __forceinline__ uint32_t wave_max32(uint32_t x) {
    const auto up = [](uint32_t p, uint32_t q) { return p > q ? p : q; };
    x = up(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, true));
    x = up(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, true));
    x = up(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, true));
    x = up(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, true));
    x = up(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, true));
    x = up(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, true));
    return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}

__device__ __forceinline__ unsigned long long wave_min(unsigned long long x) {
    return lane63(wave_scan64(x, [](uint64_t p, uint64_t q) { return p < q ? p : q; }));
}

__device__ __forceinline__ unsigned long long wave_or(unsigned long long x) {
    return lane63(wave_scan64(x, [](uint64_t p, uint64_t q) { return p | q; }));
}

// Position of the k-th set bit (k from 0) of x.
__device__ __forceinline__ int select_bit(uint64_t x, int k) {
    int pos = 0;
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        const uint64_t low = x & ((1ULL << s) - 1);
        const int c = __popcll(low);
        if (k >= c) {
            k -= c;
            x >>= s;
            pos += s;
        }
    }
    return pos;
}

// The last vertex of [lo, nv) whose list starts at or before position k
// (k < nnz, so that list is not empty).
__device__ __forceinline__ int64_t owner_of(const int64_t *off, int64_t lo, int64_t nv, int64_t k) {
    int64_t hi = nv;
    while (hi - lo > 1) {
        const int64_t mid = (lo + hi) >> 1;
        if (off[mid] <= k)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// Walk the list entries [c0, end) on one wave, whatever the degrees: 64
// vertices at a time, their entries one per lane and kRangeRounds rounds in
// flight.  open(v, b, e) starts a window (lane i: vertex v = first + i, list
// [b, e), empty past nv); visit(o, q, live) takes kRangeRounds entries a lane:
// position q, owner lane o; close(v, b, e) ends the window.  Wave-collective.
constexpr int kRangeRounds = 4;
template <typename Open, typename Visit, typename Close>
__device__ __forceinline__ void walk_range(const int64_t *off, int64_t nv, int64_t nnz, int64_t c0,
                                           int64_t end, Open open, Visit visit, Close close) {
    const int lane = lane_id();
    int64_t v0 = owner_of(off, 0, nv, c0);
    for (int64_t k = c0; k < end;) {
        const int64_t v = v0 + lane;
        const int64_t b = v < nv ? off[v] : nnz, e = v < nv ? off[v + 1] : nnz;
        const int64_t last = lane_bcast(e, 63);
        const int64_t stop = last < end ? last : end;
        if (stop <= k) {  // 64 empty lists
            v0 = owner_of(off, v0, nv, k);
            continue;
        }
        open(v, b, e);
        for (int64_t q0 = k; q0 < stop; q0 += kRangeRounds * 64) {
            int o[kRangeRounds];
            int64_t q[kRangeRounds];
            bool live[kRangeRounds];
#pragma unroll
            for (int j = 0; j < kRangeRounds; ++j) {
                q[j] = q0 + 64 * j + lane;
                live[j] = q[j] < stop;
                if (!live[j]) q[j] = stop - 1;
                o[j] = 0;
#pragma unroll
                for (int st = 32; st > 0; st >>= 1) {
                    const int mid = o[j] + st;
                    if (__shfl(b, mid) <= q[j]) o[j] = mid;
                }
            }
            visit(o, q, live);
        }
        close(v, b, e);
        k = stop;
        v0 += 64;
    }
}

}  // namespace bd
