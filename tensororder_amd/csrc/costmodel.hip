// Training and inference kernels of the plan-cost MLP (include/tensororder_costmodel.h).
//
// The network is tiny (5378 parameters) and a training step has a few thousand rows, so a step
// is three launches: the forward pass with the activation gradients, a wave per few rows and
// the weights in LDS, all weight gradients (a fixed-order reduction over the rows), Adam.
#include <hip/hip_runtime.h>

#include <stdint.h>
#include <stdio.h>

#include "tensororder_costmodel.h"

#define TO_OK 0
#define TO_ERR_INVALID 2
#define TO_ERR_HIP 3

namespace {

constexpr int kBlock = 256;
constexpr int OFF_W1 = 0;
constexpr int OFF_B1 = OFF_W1 + TO_MLP_H1 * TO_MLP_IN;
constexpr int OFF_W2 = OFF_B1 + TO_MLP_H1;
constexpr int OFF_B2 = OFF_W2 + TO_MLP_H2 * TO_MLP_H1;
constexpr int OFF_W3 = OFF_B2 + TO_MLP_H2;
constexpr int OFF_B3 = OFF_W3 + TO_MLP_OUT * TO_MLP_H2;
static_assert(OFF_B3 + TO_MLP_OUT == TO_MLP_NPARAMS, "parameter layout");

// rows per wave: 2048 rows are a block for every CU, and a training step takes 44.9 us (46.7 with 4
// rows, half the CUs idle; the same from 4096 rows on)
constexpr int kRows = 2;
constexpr int kRowsPerBlock = kRows * (kBlock / 64);

// h[l] of every lane's value, as a scalar
__device__ __forceinline__ float lane_value(float v, int l) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane(__float_as_int(v), l));
}

__device__ __forceinline__ float wave_sum(float v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// The whole forward pass of kRows rows per wave: lane j owns unit j of both hidden layers, the
// previous layer's units are read back with v_readlane, the weights come transposed from LDS
// (pitch 65: no bank conflicts either way).  Bound by latency at the batch sizes of training:
// one launch of 6 us where one thread per activation took three of 38 us together at 2048 rows.
// TRAIN: the gradients of the activations too (as k_backward_rows), from the values at hand and
// the same copy of W2, read along its rows: 14 us where the two launches took 18 (2048 rows).
template <bool TRAIN>
__global__ __launch_bounds__(kBlock) void k_forward(const float* __restrict__ params, const float* __restrict__ x,
                                                    int64_t n, float* __restrict__ h1, float* __restrict__ h2,
                                                    float* __restrict__ y, const float* __restrict__ t,
                                                    float* __restrict__ dy, float* __restrict__ dh2,
                                                    float* __restrict__ dh1, float scale) {
    __shared__ float w1[TO_MLP_IN * 65], w2[TO_MLP_H1 * 65];
    for (int i = threadIdx.x; i < TO_MLP_H1 * TO_MLP_IN; i += kBlock)
        w1[(i % TO_MLP_IN) * 65 + i / TO_MLP_IN] = params[OFF_W1 + i];
    for (int i = threadIdx.x; i < TO_MLP_H2 * TO_MLP_H1; i += kBlock)
        w2[(i % TO_MLP_H1) * 65 + i / TO_MLP_H1] = params[OFF_W2 + i];
    const int lane = threadIdx.x & 63;
    const float b1 = params[OFF_B1 + lane], b2 = params[OFF_B2 + lane];
    const float w30 = params[OFF_W3 + lane], w31 = params[OFF_W3 + TO_MLP_H2 + lane];
    const float b30 = params[OFF_B3], b31 = params[OFF_B3 + 1];
    __syncthreads();
    const int64_t r0 = (int64_t)blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6) * kRows;
    float in[kRows], a[kRows], b[kRows], t0[kRows], t1[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        if constexpr (TRAIN) {
            const int64_t i = r0 + r < n ? r0 + r : n - 1;
            t0[r] = t[i * TO_MLP_OUT];
            t1[r] = t[i * TO_MLP_OUT + 1];
        }
        in[r] = lane < TO_MLP_IN && r0 + r < n ? x[(r0 + r) * TO_MLP_IN + lane] : 0.0f;
        a[r] = b1;
        b[r] = b2;
    }
#pragma unroll
    for (int k = 0; k < TO_MLP_IN; ++k) {
        const float w = w1[k * 65 + lane];
#pragma unroll
        for (int r = 0; r < kRows; ++r) a[r] += lane_value(in[r], k) * w;
    }
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        a[r] = fmaxf(a[r], 0.0f);
        if (r0 + r < n) h1[(r0 + r) * TO_MLP_H1 + lane] = a[r];
    }
#pragma unroll 16
    for (int k = 0; k < TO_MLP_H1; ++k) {
        const float w = w2[k * 65 + lane];
#pragma unroll
        for (int r = 0; r < kRows; ++r) b[r] += lane_value(a[r], k) * w;
    }
    float g[kRows], d[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        b[r] = fmaxf(b[r], 0.0f);
        const float s0 = wave_sum(b[r] * w30) + b30, s1 = wave_sum(b[r] * w31) + b31;
        if (r0 + r < n) {
            h2[(r0 + r) * TO_MLP_H2 + lane] = b[r];
            if (lane < TO_MLP_OUT) y[(r0 + r) * TO_MLP_OUT + lane] = lane == 0 ? s0 : s1;
        }
        if constexpr (TRAIN) {
            const float d0 = scale * (s0 - t0[r]), d1 = scale * (s1 - t1[r]);
            g[r] = b[r] > 0.0f ? d0 * w30 + d1 * w31 : 0.0f;
            d[r] = 0.0f;
            if (r0 + r < n) {
                dh2[(r0 + r) * TO_MLP_H2 + lane] = g[r];
                if (lane < TO_MLP_OUT) dy[(r0 + r) * TO_MLP_OUT + lane] = lane == 0 ? d0 : d1;
            }
        }
    }
    if constexpr (TRAIN) {
#pragma unroll 16
        for (int o = 0; o < TO_MLP_H2; ++o) {
            const float w = w2[lane * 65 + o];
#pragma unroll
            for (int r = 0; r < kRows; ++r) d[r] += lane_value(g[r], o) * w;
        }
#pragma unroll
        for (int r = 0; r < kRows; ++r)
            if (r0 + r < n) dh1[(r0 + r) * TO_MLP_H1 + lane] = a[r] > 0.0f ? d[r] : 0.0f;
    }
}

// The gradients of the activations, laid out as in k_forward:
// dy = 2 (y - target) / (n * OUT), dh2 = (dy W3) * (h2 > 0), dh1 = (dh2 W2) * (h1 > 0)
__global__ __launch_bounds__(kBlock) void k_backward_rows(const float* __restrict__ params, const float* __restrict__ h1,
                                                          const float* __restrict__ h2, const float* __restrict__ y,
                                                          const float* __restrict__ t, int64_t n,
                                                          float* __restrict__ dy, float* __restrict__ dh2,
                                                          float* __restrict__ dh1, float scale) {
    __shared__ float w2[TO_MLP_H2 * TO_MLP_H1];
    for (int i = threadIdx.x; i < TO_MLP_H2 * TO_MLP_H1; i += kBlock) w2[i] = params[OFF_W2 + i];
    const int lane = threadIdx.x & 63;
    const float w30 = params[OFF_W3 + lane], w31 = params[OFF_W3 + TO_MLP_H2 + lane];
    __syncthreads();
    const int64_t r0 = (int64_t)blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6) * kRows;
    float g[kRows], a[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        const int64_t i = r0 + r < n ? r0 + r : n - 1;
        const float d0 = scale * (y[i * TO_MLP_OUT] - t[i * TO_MLP_OUT]);
        const float d1 = scale * (y[i * TO_MLP_OUT + 1] - t[i * TO_MLP_OUT + 1]);
        g[r] = h2[i * TO_MLP_H2 + lane] > 0.0f ? d0 * w30 + d1 * w31 : 0.0f;
        a[r] = 0.0f;
        if (r0 + r < n) {
            dh2[i * TO_MLP_H2 + lane] = g[r];
            if (lane < TO_MLP_OUT) dy[i * TO_MLP_OUT + lane] = lane == 0 ? d0 : d1;
        }
    }
#pragma unroll 16
    for (int o = 0; o < TO_MLP_H2; ++o) {
        const float w = w2[o * TO_MLP_H1 + lane];
#pragma unroll
        for (int r = 0; r < kRows; ++r) a[r] += lane_value(g[r], o) * w;
    }
#pragma unroll
    for (int r = 0; r < kRows; ++r)
        if (r0 + r < n) dh1[(r0 + r) * TO_MLP_H1 + lane] = h1[(r0 + r) * TO_MLP_H1 + lane] > 0.0f ? a[r] : 0.0f;
}

// Every weight gradient dW[j][k] = sum_i g[i][j] in[i][k], bias gradient db[j] = sum_i g[i][j]
// and the loss in one launch: a block owns an 8 x 8 tile (2 x 8 of the output layer), its 1024
// threads are 128 row groups of 8 columns, each summing its rows in double, then the groups are
// added in a fixed order.  64 + 16 + 8 tiles and one block for the loss.  Rows are read whole
// (32 bytes of g, 32 of in per group of 8 lanes), four in flight per thread; bound by the
// latency of those reads.  One block per parameter, which read them 4 bytes apart, took 83 us
// of a 192 us step at 2048 rows; one row in flight 36 us.  wide: g rows are 16-byte aligned.
constexpr int kGradThreads = 1024;
constexpr int kTiles2 = 64, kTiles1 = 16, kTiles3 = 8;

__global__ __launch_bounds__(kGradThreads) void k_weight_grads(
    const float* __restrict__ x, const float* __restrict__ h1, const float* __restrict__ h2,
    const float* __restrict__ dy, const float* __restrict__ dh2, const float* __restrict__ dh1,
    const float* __restrict__ y, const float* __restrict__ t, int64_t n, float* __restrict__ grad,
    float* __restrict__ loss, bool wide) {
    __shared__ double red[kGradThreads / 64][9][8];
    const int tid = threadIdx.x, wave = tid >> 6;
    int b = blockIdx.x;
    if (b == kTiles2 + kTiles1 + kTiles3) {  // the loss
        double acc = 0.0;
        for (int64_t i = tid; i < n * TO_MLP_OUT; i += kGradThreads) {
            const float e = y[i] - t[i];
            acc += (double)e * (double)e;
        }
        for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
        if ((tid & 63) == 0) red[wave][0][0] = acc;
        __syncthreads();
        if (tid == 0 && loss) {
            acc = 0.0;
            for (int w = 0; w < kGradThreads / 64; ++w) acc += red[w][0][0];
            loss[0] = (float)(acc / (double)(n * TO_MLP_OUT));
            __threadfence_system();  // it may lie in host memory
        }
        return;
    }
    const float *g, *in;
    float *dW, *db;
    int dout, din;
    if (b < kTiles2) {
        g = dh2, in = h1, dW = grad + OFF_W2, db = grad + OFF_B2, dout = TO_MLP_H2, din = TO_MLP_H1;
    } else if (b < kTiles2 + kTiles1) {
        b -= kTiles2;
        g = dh1, in = x, dW = grad + OFF_W1, db = grad + OFF_B1, dout = TO_MLP_H1, din = TO_MLP_IN;
    } else {
        b -= kTiles2 + kTiles1;
        g = dy, in = h2, dW = grad + OFF_W3, db = grad + OFF_B3, dout = TO_MLP_OUT, din = TO_MLP_H2;
    }
    const int kt = din / 8;
    const int j0 = (b / kt) * 8, k0 = (b % kt) * 8;
    const int nj = dout < 8 ? dout : 8;
    const int c = tid & 7, group = tid >> 3;
    double acc[8], bias = 0.0;
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = 0.0;
    // four rows in flight per thread: a row's loads take a trip to L2, its sums next to nothing
    typedef float F4 __attribute__((ext_vector_type(4)));
    constexpr int kStep = kGradThreads / 8;
    for (int64_t i = group; i < n; i += 4 * kStep) {
        float v[4], gv[4][8], gc[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const bool row = i + u * kStep < n;
            const int64_t r = row ? i + u * kStep : 0;
            v[u] = in[r * din + k0 + c];
            if (nj == 8 && wide) {
                const F4 lo = *reinterpret_cast<const F4*>(g + r * dout + j0), hi = *reinterpret_cast<const F4*>(g + r * dout + j0 + 4);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    gv[u][j] = lo[j];
                    gv[u][4 + j] = hi[j];
                }
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) gv[u][j] = j < nj ? g[r * dout + j0 + j] : 0.0f;
            }
            gc[u] = k0 == 0 && c < nj ? g[r * dout + j0 + c] : 0.0f;
            if (!row) {  // (row 0 in its place may hold what times 0 is no 0)
                v[u] = gc[u] = 0.0f;
#pragma unroll
                for (int j = 0; j < 8; ++j) gv[u][j] = 0.0f;
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[j] = fma((double)gv[u][j], (double)v[u], acc[j]);
            bias += (double)gc[u];
        }
    }
    // lanes 8 apart are the wave's row groups
#pragma unroll
    for (int j = 0; j < 8; ++j)
        for (int off = 8; off < 64; off <<= 1) acc[j] += __shfl_xor(acc[j], off, 64);
    for (int off = 8; off < 64; off <<= 1) bias += __shfl_xor(bias, off, 64);
    if ((tid & 63) < 8) {
#pragma unroll
        for (int j = 0; j < 8; ++j) red[wave][j][c] = acc[j];
        red[wave][8][c] = bias;
    }
    __syncthreads();
    if (tid < 72) {
        const int j = tid >> 3;
        double s = 0.0;
        for (int w = 0; w < kGradThreads / 64; ++w) s += red[w][j][c];
        if (j < nj) dW[(j0 + j) * din + k0 + c] = (float)s;
        else if (j == 8 && k0 == 0 && c < nj) db[j0 + c] = (float)s;
    }
}

__global__ __launch_bounds__(kBlock) void k_adam(float* __restrict__ p, const float* __restrict__ g,
                                                 float* __restrict__ m, float* __restrict__ v, int64_t count,
                                                 float lr, float b1, float b2, float eps, float c1, float c2) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < count; i += (int64_t)gridDim.x * kBlock) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.0f - b1) * gi;
        const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    }
}

int grid_for(int64_t work) {
    const int64_t g = (work + kBlock - 1) / kBlock;
    return (int)(g < 1 ? 1 : (g > 65535 ? 65535 : g));
}

int status(const char*) {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? TO_OK : TO_ERR_HIP;
}

void launch_weight_grads(const float* x, const float* h1, const float* h2, const float* y, const float* target, int64_t n,
                         const float* dy, const float* dh2, const float* dh1, float* grad, float* loss, hipStream_t st) {
    hipLaunchKernelGGL(k_weight_grads, dim3(kTiles2 + kTiles1 + kTiles3 + 1), dim3(kGradThreads), 0, st, x, h1, h2, dy,
                       dh2, dh1, y, target, n, grad, loss,
                       ((reinterpret_cast<uintptr_t>(dh2) | reinterpret_cast<uintptr_t>(dh1)) & 15) == 0);
}

// The rows in launches of at most 2^26 (the threads of a launch are counted in 32 bits, 32 a row)
template <typename F>
void launch_rows(int64_t n, F launch) {
    constexpr int64_t kMost = 1ll << 26;
    for (int64_t r = 0; r < n; r += kMost) {
        const int64_t m = n - r < kMost ? n - r : kMost;
        launch(r, m, dim3((unsigned)((m + kRowsPerBlock - 1) / kRowsPerBlock)));
    }
}

// dy = scale (y - target)
float out_scale(int64_t n) { return 2.0f / (float)(n * TO_MLP_OUT); }

}  // namespace

extern "C" {

int to_mlp_forward(const float* params, const float* x, int64_t n, float* h1, float* h2, float* y, void* stream) {
    if (!params || !x || !h1 || !h2 || !y || n <= 0) return TO_ERR_INVALID;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    launch_rows(n, [&](int64_t r, int64_t m, dim3 grid) {
        hipLaunchKernelGGL(k_forward<false>, grid, dim3(kBlock), 0, st, params, x + r * TO_MLP_IN, m, h1 + r * TO_MLP_H1,
                           h2 + r * TO_MLP_H2, y + r * TO_MLP_OUT, nullptr, nullptr, nullptr, nullptr, 0.0f);
    });
    return status("to_mlp_forward");
}

int to_mlp_backward(const float* params, const float* x, const float* h1, const float* h2, const float* y,
                    const float* target, int64_t n, float* dy, float* dh2, float* dh1, float* grad, float* loss,
                    void* stream) {
    if (!params || !x || !h1 || !h2 || !y || !target || !dy || !dh2 || !dh1 || !grad || n <= 0)
        return TO_ERR_INVALID;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    launch_rows(n, [&](int64_t r, int64_t m, dim3 grid) {
        hipLaunchKernelGGL(k_backward_rows, grid, dim3(kBlock), 0, st, params, h1 + r * TO_MLP_H1, h2 + r * TO_MLP_H2,
                           y + r * TO_MLP_OUT, target + r * TO_MLP_OUT, m, dy + r * TO_MLP_OUT, dh2 + r * TO_MLP_H2,
                           dh1 + r * TO_MLP_H1, out_scale(n));
    });
    launch_weight_grads(x, h1, h2, y, target, n, dy, dh2, dh1, grad, loss, st);
    return status("to_mlp_backward");
}

int to_mlp_gradient(const float* params, const float* x, const float* target, int64_t n, float* h1, float* h2, float* y,
                    float* dy, float* dh2, float* dh1, float* grad, float* loss, void* stream) {
    if (!params || !x || !target || !h1 || !h2 || !y || !dy || !dh2 || !dh1 || !grad || n <= 0) return TO_ERR_INVALID;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    launch_rows(n, [&](int64_t r, int64_t m, dim3 grid) {
        hipLaunchKernelGGL(k_forward<true>, grid, dim3(kBlock), 0, st, params, x + r * TO_MLP_IN, m, h1 + r * TO_MLP_H1,
                           h2 + r * TO_MLP_H2, y + r * TO_MLP_OUT, target + r * TO_MLP_OUT, dy + r * TO_MLP_OUT,
                           dh2 + r * TO_MLP_H2, dh1 + r * TO_MLP_H1, out_scale(n));
    });
    launch_weight_grads(x, h1, h2, y, target, n, dy, dh2, dh1, grad, loss, st);
    return status("to_mlp_gradient");
}

int to_mlp_adam(float* params, const float* grad, float* m, float* v, int64_t count, float lr, float beta1,
                float beta2, float eps, int64_t step, void* stream) {
    if (!params || !grad || !m || !v || count <= 0 || step < 1) return TO_ERR_INVALID;
    const float c1 = 1.0f - powf(beta1, (float)step);
    const float c2 = 1.0f - powf(beta2, (float)step);
    hipLaunchKernelGGL(k_adam, dim3(grid_for(count)), dim3(kBlock), 0, reinterpret_cast<hipStream_t>(stream),
                       params, grad, m, v, count, lr, beta1, beta2, eps, c1, c2);
    return status("to_mlp_adam");
}

}  // extern "C"
