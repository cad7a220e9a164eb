// bd_mlp.hip -- training and inference kernels of the learned direction
// policy (no reference counterpart; it replaces the predicates at
// hybrid_bfs.cc:167 and :178-179).
//
//   k_mlp_infer_f32   one wave per 32 samples, fp32 MFMA (the numerics reference)
//   k_mlp_infer_mfma  one wave per 16 samples, bf16 MFMA, fp32 accumulate
//   k_mlp_train       Adam's step for the pass before, then loss and gradients
//                     with fp32 MFMA, one partial gradient per workgroup
//   k_mlp_sum         sum of the partial gradients
#include <math.h>
#include <string.h>

#include <algorithm>
#include <type_traits>
#include <vector>

#include "bd_internal.h"
#include "bd_mlp.h"

namespace bd {

namespace {

constexpr int kMaxParams = 32 * 8 + 32 + 32 * 32 + 32 + 2 * 32 + 2;


// The fp32 network on the matrix cores: v_mfma_f32_32x32x2f32 keeps fp32
// operands and sums, and every product of the network (forward, input
// gradients, weight gradients) is a 32-wide contraction, so one wave takes
// 32 samples at a time.  Lane l of a wave holds of a 32x32 result column
// l%32, rows mrow(r, l) = 8 (r/4) + 4 (l/32) + r%4 of registers r = 0..15.
// Layers are computed with samples as columns (Y = W X^T), and the k pair
// of step r is taken as rows mrow(r, 0) and mrow(r, 32): then a layer's
// result registers are the next layer's B operand as they are.
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kTrainWaves = 4;               // waves per workgroup, each with its own samples
constexpr int kTrainBlock = 64 * kTrainWaves;
constexpr int kTrainParams = kMaxParams / kTrainBlock + 1;  // a thread's (and the loss)
constexpr int kTrainMaxGrid = 64;            // workgroups, i.e. partial gradients, of one pass
constexpr int kPartStride = kMaxParams + 2;  // a workgroup's gradients, then its loss
constexpr int kRow = 33;                     // LDS row stride: rows land on different banks

__device__ __forceinline__ int mrow(int r, int l) { return 8 * (r >> 2) + 4 * (l >> 5) + (r & 3); }

__device__ __forceinline__ f32x16 mfma32(float a, float b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// Parameters in LDS, padded to 32 hidden units with zeros (a padded unit's
// activation and gradient are 0).
struct mlp_lds {
    float w1[32 * 9];
    float w2[32 * kRow];
    float w3[2 * 32];
    float b1[32], b2[32], b3[2];
    __device__ __forceinline__ void clear(int tid, int nthreads) {
        float *p = w1;
        for (int i = tid; i < (int)(sizeof(mlp_lds) / sizeof(float)); i += nthreads) p[i] = 0.f;
    }
    // parameter i of the flat layout
    __device__ __forceinline__ void put(int i, int h1, int h2, float v) {
        if (i < h1 * kMlpIn) {
            w1[(i >> 3) * 9 + (i & 7)] = v;
            return;
        }
        i -= h1 * kMlpIn;
        if (i < h1) {
            b1[i] = v;
            return;
        }
        i -= h1;
        if (i < h2 * h1) {
            const int k = i / h1;
            w2[k * kRow + (i - k * h1)] = v;
            return;
        }
        i -= h2 * h1;
        if (i < h2) {
            b2[i] = v;
            return;
        }
        i -= h2;
        if (i < kMlpOut * h2) {
            const int o = i >= h2;
            w3[o * 32 + (i - o * h2)] = v;
            return;
        }
        b3[i - kMlpOut * h2] = v;
    }
};

// A lane's operands of the forward pass.
struct mlp_fwd_regs {
    float w1[4], w2[16], w3[16], b1[16], b2[16], b3[2];
    __device__ __forceinline__ void load(const mlp_lds &s) {
        const int l = threadIdx.x & 63, i = l & 31, q = l >> 5;
#pragma unroll
        for (int k = 0; k < 4; ++k) w1[k] = s.w1[i * 9 + 2 * k + q];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int k = mrow(r, l);
            w2[r] = s.w2[i * kRow + k];
            w3[r] = i < kMlpOut ? s.w3[i * 32 + k] : 0.f;
            b1[r] = s.b1[k];
            b2[r] = s.b2[k];
        }
        b3[0] = s.b3[0];
        b3[1] = s.b3[1];
    }
};

// Forward pass of the wave's 32 samples: lane l holds inputs 2k + l/32 of
// sample l%32 in x[k].  y[] is valid in lanes 0..31.
__device__ __forceinline__ void mlp_fwd32(const mlp_fwd_regs &w, const float (&x)[4], f32x16 &a1,
                                          f32x16 &a2, float (&y)[2]) {
    const f32x16 z = {};
    a1 = z;
#pragma unroll
    for (int k = 0; k < 4; ++k) a1 = mfma32(w.w1[k], x[k], a1);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float v = a1[r] + w.b1[r];
        a1[r] = v > 0.f ? v : 0.f;
    }
    a2 = z;
#pragma unroll
    for (int r = 0; r < 16; ++r) a2 = mfma32(w.w2[r], a1[r], a2);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float v = a2[r] + w.b2[r];
        a2[r] = v > 0.f ? v : 0.f;
    }
    f32x16 o = z;
#pragma unroll
    for (int r = 0; r < 16; ++r) o = mfma32(w.w3[r], a2[r], o);
    y[0] = o[0] + w.b3[0];
    y[1] = o[1] + w.b3[1];
}

// fp32 inference, 32 samples per wave (3038 samples: 105 us with a thread per
// sample and its activations in scratch memory).
__global__ __launch_bounds__(64) void k_mlp_infer_f32(const float *__restrict__ p, int h1, int h2,
                                                      const float *__restrict__ x, int64_t n,
                                                      float *__restrict__ y) {
    __shared__ mlp_lds s;
    const int l = threadIdx.x;
    const int np = (int)mlp_nparams(h1, h2);
    s.clear(l, 64);
    __syncthreads();
    for (int i = l; i < np; i += 64) s.put(i, h1, h2, p[i]);
    __syncthreads();
    mlp_fwd_regs w;
    w.load(s);
    for (int64_t base = (int64_t)blockIdx.x * 32; base < n; base += (int64_t)gridDim.x * 32) {
        const int64_t at = base + (l & 31);
        float xs[4], out[2];
#pragma unroll
        for (int k = 0; k < 4; ++k) xs[k] = at < n ? x[at * kMlpIn + 2 * k + (l >> 5)] : 0.f;
        f32x16 a1, a2;
        mlp_fwd32(w, xs, a1, a2, out);
        if (l < 32 && at < n) {
            y[at * 2] = out[0];
            y[at * 2 + 1] = out[1];
        }
    }
}

__global__ __launch_bounds__(64) void k_mlp_infer_mfma(const float *__restrict__ p, int h1, int h2,
                                                       const float *__restrict__ x, int64_t n,
                                                       float *__restrict__ y) {
    __shared__ float X[16][32];
    __shared__ float H[16][32];
    __shared__ float Y[16][32];
    const int l = threadIdx.x;
    for (int64_t base = (int64_t)blockIdx.x * 16; base < n; base += (int64_t)gridDim.x * 16) {
        for (int i = l; i < 16 * 32; i += 64) {
            const int r = i / 32, cidx = i % 32;
            const int64_t s = base + r;
            X[r][cidx] = (s < n && cidx < kMlpIn) ? x[s * kMlpIn + cidx] : 0.f;
        }
        wave_lds_sync();
        mlp_forward_rows_mfma(p, h1, h2, X, H, Y);
        if (l < 32) {
            const int r = l >> 1, o = l & 1;
            if (base + r < n) y[(base + r) * 2 + o] = Y[r][o];
        }
        wave_lds_sync();
    }
}

// One training pass.  First every workgroup brings the parameters up to date:
// the partial gradients of the pass before are summed and Adam applied, by
// every workgroup alike (workgroup 0 publishes the new state), so an epoch is
// one launch.  Then each wave takes tiles of 32 samples, keeps its weight
// gradients in accumulators, and the workgroup writes one partial gradient.
// State and partials alternate between two copies, since workgroups of a
// pass still read the old ones while others write.
struct train_args {
    const float *x, *t, *mask;
    int64_t n;
    int h1, h2;
    float inv_count;
    const float *part_in;  // partials of the pass before (step > 0)
    int nparts;
    float *part_out;
    const float *st_in;    // parameters, then (step > 0) Adam's two moments, kMaxParams each
    float *st_out;         // null: not kept
    float *p_out;          // also receives the parameters when not null
    int step;              // Adam steps made before this pass; 0: st_in as it is
    float lr, c1, c2;
};

// Measured, 3038 samples: 1750 us a pass with a thread per sample and an LDS
// atomic per sample and parameter (all lanes of a wave on one address); now
// a launch's latency, the parameter update and ~110 MFMAs per wave, 16.0 us
// (27.4 with one parameter's partials loaded after another's and the waves'
// gradients added up in turn).  All of a thread's parameters are loaded
// together, up to 16 partials of each, and the first tile's samples before
// them (32 epochs of 300 to 20000 samples: 8 partials at a time 0 to 2% longer,
// 24 the same, 32 from 1% longer at 3000 to 3% less at 8000, 48 longer).  The
// update is still 6 us of it; twice the threads for it alone leave the others
// half the registers, which spilled (21 us).
__global__ __launch_bounds__(kTrainBlock) void k_mlp_train(train_args a) {
    __shared__ mlp_lds s;
    // per wave: activations and gradients of its samples, [sample][unit]
    __shared__ float A1[kTrainWaves][32 * kRow], A2[kTrainWaves][32 * kRow];
    __shared__ float D1[kTrainWaves][32 * kRow], D2[kTrainWaves][32 * kRow];
    __shared__ float X[kTrainWaves][32 * kMlpIn], DY[kTrainWaves][32 * 2];
    const int tid = threadIdx.x, l = tid & 63, wid = tid >> 6;
    const int i = l & 31, q = l >> 5;
    const int np = (int)mlp_nparams(a.h1, a.h2);
    s.clear(tid, kTrainBlock);
    __syncthreads();
    const int64_t ntiles = (a.n + 31) / 32;
    const int64_t tile0 = (int64_t)blockIdx.x * kTrainWaves + wid;
    float xn[4], tn = 0.f, mn = 0.f;  // the next tile's inputs, target and mask
    const auto fetch = [&](int64_t tile) {
        const int64_t at = tile * 32 + i;
        const bool valid = at < a.n;
#pragma unroll
        for (int k = 0; k < 4; ++k) xn[k] = valid ? a.x[at * kMlpIn + 2 * k + q] : 0.f;
        tn = valid ? a.t[at * 2 + q] : 0.f;
        mn = valid ? (a.mask ? a.mask[at * 2 + q] : 1.f) : 0.f;
    };
    fetch(tile0);
    {
        float p[kTrainParams], mo[kTrainParams], ve[kTrainParams], g[kTrainParams];
#pragma unroll
        for (int r = 0; r < kTrainParams; ++r) {
            const int k = tid + r * kTrainBlock;
            p[r] = k < np ? a.st_in[k] : 0.f;
            mo[r] = k < np && a.step > 1 ? a.st_in[kMaxParams + k] : 0.f;
            ve[r] = k < np && a.step > 1 ? a.st_in[2 * kMaxParams + k] : 0.f;
            g[r] = 0.f;
        }
        if (a.step > 0) {
            int b = 0;
            const auto add = [&](auto count) {
                constexpr int N = decltype(count)::value;
                float v[kTrainParams][N];
#pragma unroll
                for (int r = 0; r < kTrainParams; ++r) {
                    const int k = tid + r * kTrainBlock < np ? tid + r * kTrainBlock : 0;
#pragma unroll
                    for (int j = 0; j < N; ++j) v[r][j] = a.part_in[(b + j) * kPartStride + k];
                }
#pragma unroll
                for (int r = 0; r < kTrainParams; ++r) {
                    if (N == 1) g[r] += v[r][0];
#pragma unroll
                    for (int j = 0; j + 8 <= N; j += 8)
                        g[r] += ((v[r][j] + v[r][j + 1]) + (v[r][j + 2] + v[r][j + 3])) +
                                ((v[r][j + 4] + v[r][j + 5]) + (v[r][j + 6] + v[r][j + 7]));
                }
                b += N;
            };
            while (b + 16 <= a.nparts) add(std::integral_constant<int, 16>{});
            while (b + 8 <= a.nparts) add(std::integral_constant<int, 8>{});
            while (b < a.nparts) add(std::integral_constant<int, 1>{});
        }
#pragma unroll
        for (int r = 0; r < kTrainParams; ++r) {
            const int k = tid + r * kTrainBlock;
            if (k >= np) continue;
            if (a.step > 0) {
                const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
                mo[r] = fmaf(1.f - b1, g[r], b1 * mo[r]);
                ve[r] = fmaf((1.f - b2) * g[r], g[r], b2 * ve[r]);
                const float mh = mo[r] / a.c1, vh = ve[r] / a.c2;
                p[r] -= a.lr * mh / (sqrtf(vh) + eps);
            }
            s.put(k, a.h1, a.h2, p[r]);
            if (blockIdx.x == 0) {
                if (a.st_out) {
                    a.st_out[k] = p[r];
                    a.st_out[kMaxParams + k] = mo[r];
                    a.st_out[2 * kMaxParams + k] = ve[r];
                }
                if (a.p_out) a.p_out[k] = p[r];
            }
        }
    }
    __syncthreads();
    mlp_fwd_regs w;
    w.load(s);
    float w2t[16];  // W2 transposed: row i, k = mrow(r)
#pragma unroll
    for (int r = 0; r < 16; ++r) w2t[r] = s.w2[mrow(r, l) * kRow + i];
    const float w3t = s.w3[q * 32 + i];
    float *a1s = A1[wid], *a2s = A2[wid], *d1s = D1[wid], *d2s = D2[wid], *xs = X[wid],
          *dys = DY[wid];
    const f32x16 z = {};
    f32x16 g1 = z, g2 = z, g3 = z;  // rows: unit of the layer's output, columns: of its input
    float gb1 = 0.f, gb2 = 0.f, gb3 = 0.f, loss = 0.f;
    for (int64_t tile = tile0; tile < ntiles; tile += (int64_t)gridDim.x * kTrainWaves) {
        const bool valid = tile * 32 + i < a.n;
        const float tv = tn, mk = mn;
        float x[4], y[2];
        float odd = 0.f;  // NaN: an infinity or NaN among the inputs or activations
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            x[k] = xn[k];
            odd = fmaf(x[k], 0.f, odd);
            xs[i * kMlpIn + 2 * k + q] = x[k];
        }
        fetch(tile + (int64_t)gridDim.x * kTrainWaves);
        f32x16 a1, a2;
        mlp_fwd32(w, x, a1, a2, y);
        float dyv = 0.f;
        {
            // lane half o takes output o of its sample
            const float yo = __shfl(y[1], i);
            const float yv = q ? yo : y[0];
            if (valid) {
                const float e = yv - tv;
                loss += mk * e * e;
                dyv = 2.f * mk * e * a.inv_count;
            }
            dys[i * 2 + q] = dyv;
        }
        f32x16 d2 = mfma32(w3t, dyv, z);  // k = output
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            d2[r] = valid && a2[r] > 0.f ? d2[r] : 0.f;
            odd = fmaf(a1[r], 0.f, odd);
            a1s[i * kRow + mrow(r, l)] = valid ? a1[r] : 0.f;
            a2s[i * kRow + mrow(r, l)] = valid ? a2[r] : 0.f;
            d2s[i * kRow + mrow(r, l)] = d2[r];
        }
        f32x16 d1 = z;
#pragma unroll
        for (int r = 0; r < 16; ++r) d1 = mfma32(w2t[r], d2[r], d1);
#pragma unroll
        for (int r = 0; r < 16; ++r) d1s[i * kRow + mrow(r, l)] = valid && a1[r] > 0.f ? d1[r] : 0.f;
        wave_lds_sync();
        // weight gradients: contractions over the samples, two per step
        if (!__ballot(odd != 0.f)) {
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const int sm = 2 * k + q;
                const float d1v = d1s[sm * kRow + i], d2v = d2s[sm * kRow + i];
                g1 = mfma32(d1v, i < kMlpIn ? xs[sm * kMlpIn + i] : 0.f, g1);
                g2 = mfma32(d2v, a1s[sm * kRow + i], g2);
                gb1 += d1v;
                gb2 += d2v;
            }
        } else {
            // a unit whose gradient is 0 adds nothing, whatever it is
            // multiplied with (0 times infinity would be NaN)
            for (int sm = 0; sm < 32; ++sm) {
                const float xv = i < kMlpIn ? xs[sm * kMlpIn + i] : 0.f, av = a1s[sm * kRow + i];
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float d1v = d1s[sm * kRow + mrow(r, l)];
                    const float d2v = d2s[sm * kRow + mrow(r, l)];
                    if (d1v != 0.f) g1[r] += d1v * xv;
                    if (d2v != 0.f) g2[r] += d2v * av;
                }
                if ((sm & 1) == q) {
                    gb1 += d1s[sm * kRow + i];
                    gb2 += d2s[sm * kRow + i];
                }
            }
        }
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const int sm = 2 * k + q;
            const float dv = i < kMlpOut ? dys[sm * 2 + i] : 0.f;
            g3 = mfma32(dv, a2s[sm * kRow + i], g3);
            gb3 += dv;
        }
        wave_lds_sync();  // the arrays are rewritten by the next tile
    }
    gb1 += __shfl_xor(gb1, 32);
    gb2 += __shfl_xor(gb2, 32);
    gb3 += __shfl_xor(gb3, 32);
#pragma unroll
    for (int d = 32; d; d >>= 1) loss += __shfl_xor(loss, d);
    // The waves' gradients go to their own arrays, which no sample needs any
    // more, and every thread adds up some parameters' in the waves' order.
    // (Waves adding theirs to one array in turn took 14.5 k of 45 k cycles.)
    enum { kG3 = 32 * kMlpIn, kB1 = kG3 + 64, kB2 = kB1 + 32, kB3 = kB2 + 32, kLoss = kB3 + 2 };
    static_assert(kLoss < 32 * kRow, "fits a sample array");
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int k = mrow(r, l);
        a1s[k * kRow + i] = g2[r];
        if (i < kMlpIn) a2s[k * kMlpIn + i] = g1[r];
        if (k < kMlpOut) a2s[kG3 + k * 32 + i] = g3[r];
    }
    if (l < 32) {
        a2s[kB1 + l] = gb1;
        a2s[kB2 + l] = gb2;
    }
    if (l < kMlpOut) a2s[kB3 + l] = gb3;
    if (l == 0) a2s[kLoss] = loss;
    __syncthreads();
    const int o_b1 = a.h1 * kMlpIn, o_w2 = o_b1 + a.h1, o_b2 = o_w2 + a.h2 * a.h1,
              o_w3 = o_b2 + a.h2, o_b3 = o_w3 + kMlpOut * a.h2;
#pragma unroll
    for (int r = 0; r < kTrainParams; ++r) {
        const int k = tid + r * kTrainBlock;  // np < kTrainParams * kTrainBlock
        if (k > np) continue;
        const bool in_w2 = k >= o_w2 && k < o_b2;
        int at;
        if (in_w2) {
            const int row = (k - o_w2) / a.h1;
            at = row * kRow + (k - o_w2 - row * a.h1);
        } else if (k < o_b1) {
            at = k;
        } else if (k < o_w2) {
            at = kB1 + k - o_b1;
        } else if (k < o_w3) {
            at = kB2 + k - o_b2;
        } else if (k < o_b3) {
            const int o = k - o_w3 >= a.h2;
            at = kG3 + o * 32 + (k - o_w3 - o * a.h2);
        } else {
            at = kB3 + k - o_b3;  // b3, then the loss
        }
        const float *from = (in_w2 ? &A1[0][0] : &A2[0][0]) + at;
        float sum = 0.f;
#pragma unroll
        for (int wv = 0; wv < kTrainWaves; ++wv) sum += from[wv * 32 * kRow];
        a.part_out[(int64_t)blockIdx.x * kPartStride + k] = sum;
    }
}

// The sum of a pass's partial gradients; entry np is the loss.
__global__ void k_mlp_sum(const float *__restrict__ part, int nparts, int np, float inv_count,
                          float *__restrict__ out) {
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k <= np; k += gridDim.x * blockDim.x) {
        float g = 0.f;
        for (int b = 0; b < nparts; ++b) g += part[b * kPartStride + k];
        out[k] = k == np ? g * inv_count : g;
    }
}

int check_mlp(bd_ctx *c) {
    if (!c->has_mlp) return set_err(c, BD_ESTATE, "no network loaded");
    return BD_OK;
}

// Workspace of a training or inference call, kept by the context up to 16 MB
// (a training run of 100 k samples) so that repeated calls allocate nothing.
int mlp_ws(bd_ctx *c, size_t bytes, float **p) {
    if (c->mlp_ws_bytes < bytes) {
        dev_free(c, c->d_mlp_ws);
        c->d_mlp_ws = nullptr;
        c->mlp_ws_bytes = 0;
        int rc = dev_alloc(c, (void **)&c->d_mlp_ws, bytes, "network workspace");
        if (rc) return rc;
        c->mlp_ws_bytes = bytes;
    }
    *p = c->d_mlp_ws;
    return BD_OK;
}

struct mlp_ws_guard {
    bd_ctx *c;
    ~mlp_ws_guard() {
        if (c->mlp_ws_bytes <= ((size_t)16 << 20)) return;
        dev_free(c, c->d_mlp_ws);
        c->d_mlp_ws = nullptr;
        c->mlp_ws_bytes = 0;
    }
};

// Buffers of a training call: samples, two copies of the parameters with
// their moments and of the partial gradients, and the summed gradient.
struct train_bufs {
    float *x, *t, *mask, *st[2], *part[2], *sum;
    int grid;
};

int train_setup(bd_ctx *c, const float *x, const float *t, const float *mask, int64_t n,
                train_bufs *b) {
    const int64_t tiles = (n + 31) / 32;
    b->grid = (int)std::min<int64_t>((tiles + kTrainWaves - 1) / kTrainWaves, kTrainMaxGrid);
    const int64_t part = (int64_t)b->grid * kPartStride, st = 3 * kMaxParams;
    const int64_t words = n * (kMlpIn + 2 * kMlpOut) + 2 * (part + st) + kPartStride;
    float *w = nullptr;
    int rc = mlp_ws(c, sizeof(float) * words, &w);
    if (rc) return rc;
    b->x = w;
    b->t = b->x + n * kMlpIn;
    b->mask = b->t + n * kMlpOut;
    float *at = b->mask + n * kMlpOut;
    for (int k = 0; k < 2; ++k, at += part) b->part[k] = at;
    for (int k = 0; k < 2; ++k, at += st) b->st[k] = at;
    b->sum = at;
    const size_t out = sizeof(float) * kMlpOut * n;  // x, t and mask lie one behind the other
    rc = stage_in(c, b->x, {{x, sizeof(float) * kMlpIn * n}, {t, out}, {mask, mask ? out : 0}});
    if (!mask) b->mask = nullptr;
    return rc;
}

double mask_count(const float *mask, int64_t n) {
    if (!mask) return 2.0 * (double)n;
    double s = 0;
    for (int64_t i = 0; i < 2 * n; ++i) s += mask[i];
    return s;
}

}  // namespace

}  // namespace bd

using namespace bd;

// The step kernels' operand table of the current network (one wave).
__global__ __launch_bounds__(64) void k_mlp_ops(const float *p, int h1, int h2, uint4 *ops) {
    mlp_ops_rec u;
    mlp_prefetch(p, h1, h2, u.r);
#pragma unroll
    for (int i = 0; i < kMlpOpsQuads; ++i) ops[threadIdx.x * kMlpOpsQuads + i] = u.q[i];
}

namespace bd {
// Rebuild the operand table after the parameters change.
int refresh_mlp_ops(bd_ctx *c) {
    if (!c->d_mlp_ops) {
        int rc = dev_alloc(c, (void **)&c->d_mlp_ops, sizeof(uint4) * 64 * kMlpOpsQuads,
                           "mlp operands");
        if (rc) return rc;
    }
    hipLaunchKernelGGL(k_mlp_ops, dim3(1), dim3(64), 0, c->stream, c->d_mlp, c->mlp_h1, c->mlp_h2,
                       c->d_mlp_ops);
    BD_HIP(c, hipGetLastError());
    BD_HIP(c, hipStreamSynchronize(c->stream));
    return BD_OK;
}
}  // namespace bd

extern "C" int bd_mlp_set(bd_ctx *c, const float *params, int h1, int h2) {
    if (!c || !params) return BD_EINVAL;
    if (h1 < 1 || h2 < 1 || h1 > kMlpMaxHidden || h2 > kMlpMaxHidden)
        return set_err(c, BD_EINVAL, "hidden sizes must be in [1, 32]");
    BD_HIP(c, hipSetDevice(c->device));
    const int64_t np = mlp_nparams(h1, h2);
    c->has_mlp = false;
    int rc;
    if (!c->d_mlp &&  // one size fits every network
        (rc = dev_alloc(c, (void **)&c->d_mlp, sizeof(float) * kMaxParams, "mlp")))
        return rc;
    BD_HIP(c, hipMemcpyAsync(c->d_mlp, params, sizeof(float) * np, hipMemcpyHostToDevice, c->stream));
    c->mlp_h1 = h1;
    c->mlp_h2 = h2;
    c->h_mlp.assign(params, params + np);
    if ((rc = refresh_mlp_ops(c))) {  // which waits for the stream
        (void)hipStreamSynchronize(c->stream);
        return rc;
    }
    c->has_mlp = true;
    return BD_OK;
}

extern "C" int bd_mlp_get(bd_ctx *c, float *params, int64_t cap, int *h1, int *h2) {
    if (!c) return BD_EINVAL;
    int rc = check_mlp(c);
    if (rc) return rc;
    const int64_t np = mlp_nparams(c->mlp_h1, c->mlp_h2);
    if (h1) *h1 = c->mlp_h1;
    if (h2) *h2 = c->mlp_h2;
    if (params) {
        if (cap < np) return set_err(c, BD_EINVAL, "buffer too small");
        BD_HIP(c, hipSetDevice(c->device));
        if ((rc = copy_sync(c, params, c->d_mlp, sizeof(float) * np, hipMemcpyDeviceToHost)))
            return rc;
    }
    return BD_OK;
}

extern "C" int bd_mlp_features(const bd_level_rec *r, int64_t nv, int64_t m, int64_t prev_dir,
                               float *x8) {
    if (!r || !x8 || nv <= 0) return BD_EINVAL;
    mlp_features_dev(r->frontier, r->frontier_deg, r->max_frontier_deg, r->unvisited,
                     r->unvisited_deg, r->level, nv, m, prev_dir, x8);
    return BD_OK;
}

extern "C" int bd_mlp_infer(bd_ctx *c, const float *x, int64_t n, float *y, int use_mfma) {
    if (!c || n < 0 || (n > 0 && (!x || !y))) return BD_EINVAL;
    int rc = check_mlp(c);
    if (rc || n == 0) return rc;
    BD_HIP(c, hipSetDevice(c->device));
    float *dx = nullptr;
    mlp_ws_guard g{c};
    if ((rc = mlp_ws(c, sizeof(float) * (kMlpIn + kMlpOut) * n, &dx))) return rc;
    float *dy = dx + kMlpIn * n;
    if ((rc = stage_in(c, dx, {{x, sizeof(float) * kMlpIn * n}}))) return rc;
    const int rows = use_mfma ? 16 : 32;  // samples per wave and round
    const int64_t grid =
        std::max<int64_t>(1, std::min<int64_t>((n + rows - 1) / rows, c->cu_count * 8));
    if (use_mfma)
        hipLaunchKernelGGL(k_mlp_infer_mfma, dim3(grid), dim3(64), 0, c->stream, c->d_mlp,
                           c->mlp_h1, c->mlp_h2, (const float *)dx, n, dy);
    else
        hipLaunchKernelGGL(k_mlp_infer_f32, dim3(grid), dim3(64), 0, c->stream, c->d_mlp,
                           c->mlp_h1, c->mlp_h2, (const float *)dx, n, dy);
    BD_HIP(c, hipGetLastError());
    // the inputs have been read when the outputs take their place in the ring
    return carry_copy(c, carry::i32_i32, y, dy, 2 * n);
}

extern "C" int bd_mlp_loss_grad(bd_ctx *c, const float *x, const float *t, const float *mask,
                                int64_t n, float *grad, float *loss) {
    if (!c || n <= 0 || !x || !t) return BD_EINVAL;
    int rc = check_mlp(c);
    if (rc) return rc;
    BD_HIP(c, hipSetDevice(c->device));
    const int np = (int)mlp_nparams(c->mlp_h1, c->mlp_h2);
    train_bufs b;
    mlp_ws_guard g{c};
    if ((rc = train_setup(c, x, t, mask, n, &b))) return rc;
    const double count = mask_count(mask, n);
    train_args a{};
    a.x = b.x;
    a.t = b.t;
    a.mask = b.mask;
    a.n = n;
    a.h1 = c->mlp_h1;
    a.h2 = c->mlp_h2;
    a.inv_count = count > 0 ? (float)(1.0 / count) : 0.f;
    a.part_out = b.part[0];
    a.st_in = c->d_mlp;
    hipLaunchKernelGGL(k_mlp_train, dim3(b.grid), dim3(kTrainBlock), 0, c->stream, a);
    hipLaunchKernelGGL(k_mlp_sum, dim3((np + 256) / 256), dim3(256), 0, c->stream,
                       (const float *)b.part[0], b.grid, np, a.inv_count, b.sum);
    BD_HIP(c, hipGetLastError());
    std::vector<float> h(np + 1);
    BD_HIP(c, hipMemcpyAsync(h.data(), b.sum, sizeof(float) * (np + 1), hipMemcpyDeviceToHost,
                             c->stream));
    BD_HIP(c, hipStreamSynchronize(c->stream));
    if (grad) std::copy(h.begin(), h.begin() + np, grad);
    if (loss) *loss = h[np];
    return BD_OK;
}

// Full-batch Adam on the device.  When no network is loaded one is created
// (h1 = h2 = 32) with seeded He-uniform weights.
extern "C" int bd_mlp_train(bd_ctx *c, const float *x, const float *t, const float *mask,
                            int64_t n, int epochs, float lr, uint32_t seed, float *loss) {
    if (!c || n <= 0 || !x || !t || epochs < 0) return BD_EINVAL;
    int rc;
    if (!c->has_mlp) {
        const int h1 = 32, h2 = 32;
        std::vector<float> p(mlp_nparams(h1, h2), 0.f);
        uint64_t st = 0x9E3779B97F4A7C15ULL ^ seed;
        auto unif = [&]() {
            st ^= st << 13;
            st ^= st >> 7;
            st ^= st << 17;
            return (float)((st >> 11) * (1.0 / 9007199254740992.0)) * 2.f - 1.f;
        };
        float *w1 = p.data(), *w2 = w1 + h1 * kMlpIn + h1, *w3 = w2 + h2 * h1 + h2;
        for (int i = 0; i < h1 * kMlpIn; ++i) w1[i] = unif() * sqrtf(6.f / kMlpIn);
        for (int i = 0; i < h2 * h1; ++i) w2[i] = unif() * sqrtf(6.f / h1);
        for (int i = 0; i < 2 * h2; ++i) w3[i] = unif() * sqrtf(6.f / h2);
        if ((rc = bd_mlp_set(c, p.data(), h1, h2))) return rc;
    }
    BD_HIP(c, hipSetDevice(c->device));
    const int np = (int)mlp_nparams(c->mlp_h1, c->mlp_h2);
    train_bufs b;
    mlp_ws_guard g{c};
    if ((rc = train_setup(c, x, t, mask, n, &b))) return rc;
    const double count = mask_count(mask, n);
    train_args a{};
    a.x = b.x;
    a.t = b.t;
    a.mask = b.mask;
    a.n = n;
    a.h1 = c->mlp_h1;
    a.h2 = c->mlp_h2;
    a.inv_count = count > 0 ? (float)(1.0 / count) : 0.f;
    a.nparts = b.grid;
    a.lr = lr;
    // pass k applies Adam's step k to the gradients of pass k - 1; the last
    // one leaves the loss at the trained parameters
    for (int k = 0; k <= epochs; ++k) {
        a.step = k;
        a.c1 = 1.f - powf(0.9f, (float)k);
        a.c2 = 1.f - powf(0.999f, (float)k);
        a.part_in = b.part[(k + 1) & 1];
        a.part_out = b.part[k & 1];
        a.st_in = k == 0 ? c->d_mlp : b.st[(k + 1) & 1];
        a.st_out = b.st[k & 1];
        a.p_out = k == epochs && k > 0 ? c->d_mlp : nullptr;
        hipLaunchKernelGGL(k_mlp_train, dim3(b.grid), dim3(kTrainBlock), 0, c->stream, a);
    }
    hipLaunchKernelGGL(k_mlp_sum, dim3((np + 256) / 256), dim3(256), 0, c->stream,
                       (const float *)b.part[epochs & 1], b.grid, np, a.inv_count, b.sum);
    BD_HIP(c, hipGetLastError());
    // the summed gradient with the loss at its end, and the parameters
    void *ring;
    BD_HIP(c, hipStreamSynchronize(c->stream));  // the samples have left the ring
    float own[2 * kPartStride], *h = own;
    if ((rc = host_ring(c, sizeof(own), &ring)) == BD_OK) {
        h = (float *)ring;
        if ((rc = queue_to_host(c, b.sum, np + 1, h)) ||
            (rc = queue_to_host(c, c->d_mlp, np, h + kPartStride)))
            return rc;
    } else if (rc != BD_ENOMEM ||
               (rc = copy_sync(c, h, b.sum, sizeof(float) * (np + 1), hipMemcpyDeviceToHost)) ||
               (rc = copy_sync(c, h + kPartStride, c->d_mlp, sizeof(float) * np,
                               hipMemcpyDeviceToHost))) {
        return rc;
    }
    if ((rc = refresh_mlp_ops(c))) return rc;
    if (loss) *loss = h[np];
    std::copy(h + kPartStride, h + kPartStride + np, c->h_mlp.begin());
    return BD_OK;
}
