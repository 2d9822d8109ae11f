// Elementwise and reduction passes of the screening module around its GEMMs
// and recurrences (src/rwkv7m/model/nnx_model.py:1015-1160): unit norms of
// the queries, the gated residual, and the usage EMA with the statistics.  As
// single torch operations these were about half of the module's 190 launches
// per training step, each over a few MB, with a host cost per launch above
// its device time; every pass here reads its inputs once.  At the 0.185B preset (4096
// rows of 768, bf16) a pass takes 4-11 us (the residual's forward moves its 25
// MB in 8.2 us, 3.1 TB/s; the final statistics, one block, 19 us), and the
// read phase's training step goes from 190 launches and 2.37 ms to 109 and
// 1.87 ms, the write phase's (fp32) from 193 and 2.97 ms to 106 and 2.64 ms.
//
// Row passes take a wave per row, lanes over columns; passes that also sum
// over rows take 64 columns by groups of rows and leave one partial row per
// group, added by the caller in an order fixed by the shape.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "wkv7_common.h"
#include "wkv7_launch.h"

namespace rwkv7m {
namespace {

__device__ __forceinline__ float wave_total(float x) {
    return add_swap<32>(add_swap<16>(group_sum<16>(x)));
}

__device__ __forceinline__ float sigmoid(float x) {
    return 1.f / (1.f + expf(-x));
}

// The larger, a NaN if either is one (as torch.maximum).
__device__ __forceinline__ float larger(float a, float b) {
    return a > b || a != a ? a : b;
}

struct RowLane {
    int64_t row;
    int lane;
};
__device__ __forceinline__ RowLane row_lane() {
    return {int64_t(blockIdx.x) * 4 + threadIdx.x / 64,
            int(threadIdx.x % 64)};
}

// 64 columns by the rows blockIdx.y * 4 + wave, + 4 * gridDim.y, ...: `f`
// gives a row's two values, summed over the rows into part[blockIdx.y][2][C].
template <typename F>
__device__ __forceinline__ void column_sums(int64_t rows, int64_t C,
                                            float* part, F f) {
    __shared__ float sum[2][4][64];
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    const int64_t c = int64_t(blockIdx.x) * 64 + lane;
    float a = 0.f, b = 0.f;
    if (c < C)
        for (int64_t r = int64_t(blockIdx.y) * 4 + wave; r < rows;
             r += 4 * int64_t(gridDim.y))
            f(r, c, a, b);
    sum[0][wave][lane] = a;
    sum[1][wave][lane] = b;
    __syncthreads();
    if (wave < 2 && c < C)
        part[(int64_t(blockIdx.y) * 2 + wave) * C + c] =
            (sum[wave][0][lane] + sum[wave][1][lane]) +
            (sum[wave][2][lane] + sum[wave][3][lane]);
}

template <typename X>
__global__ __launch_bounds__(256) void unit_fwd_kernel(ScreenUnitArgs A) {
    const RowLane p = row_lane();
    if (p.row >= A.rows) return;
    const X* x = static_cast<const X*>(A.x) + p.row * A.n;
    float s = 0.f;
    for (int64_t c = p.lane; c < A.n; c += 64) s += load_f(x + c) * load_f(x + c);
    const float norm = sqrtf(wave_total(s) + A.eps * A.eps);
    for (int64_t c = p.lane; c < A.n; c += 64)
        A.out[p.row * A.n + c] = load_f(x + c) / norm;
}

template <typename X>
__global__ __launch_bounds__(256) void unit_bwd_kernel(ScreenUnitArgs A) {
    const RowLane p = row_lane();
    if (p.row >= A.rows) return;
    const X* x = static_cast<const X*>(A.x) + p.row * A.n;
    const float* g = A.dout + p.row * A.n;
    float s = 0.f, d = 0.f;
    for (int64_t c = p.lane; c < A.n; c += 64) {
        const float v = load_f(x + c);
        s += v * v;
        d += v * g[c];
    }
    const float norm = sqrtf(wave_total(s) + A.eps * A.eps);
    d = wave_total(d) / norm;
    for (int64_t c = p.lane; c < A.n; c += 64)
        store_f(static_cast<X*>(A.dx) + p.row * A.n + c,
                (g[c] - load_f(x + c) / norm * d) / norm);
}

// h = h_base + lam sigmoid(pre + bias) read
template <typename E, typename H>
__global__ __launch_bounds__(256) void residual_fwd_kernel(
    ScreenResidualArgs A) {
    const int64_t c = int64_t(blockIdx.x) * 64 + threadIdx.x % 64;
    if (c >= A.C) return;
    const float lam = *A.lam, bias = A.bias[c];
    for (int64_t r = int64_t(blockIdx.y) * 4 + threadIdx.x / 64; r < A.rows;
         r += 4 * int64_t(gridDim.y)) {
        const int64_t i = r * A.C + c;
        const float g = sigmoid(load_f(static_cast<const E*>(A.pre) + i) + bias);
        store_f(static_cast<H*>(A.h) + i,
                load_f(static_cast<const H*>(A.h_base) + i) +
                    lam * g * load_f(static_cast<const H*>(A.read) + i));
    }
}

template <typename E, typename H>
__global__ __launch_bounds__(256) void residual_bwd_kernel(
    ScreenResidualArgs A) {
    const float lam = *A.lam;
    column_sums(A.rows, A.C, A.part,
                [&](int64_t r, int64_t c, float& db, float& dl) {
                    const int64_t i = r * A.C + c;
                    const float g = sigmoid(
                        load_f(static_cast<const E*>(A.pre) + i) + A.bias[c]);
                    const float rd = load_f(static_cast<const H*>(A.read) + i);
                    const float dh = load_f(static_cast<const H*>(A.dh) + i);
                    const float dp = dh * lam * rd * (g * (1.f - g));
                    store_f(static_cast<E*>(A.d_pre) + i, dp);
                    store_f(static_cast<H*>(A.d_read) + i, dh * lam * g);
                    db += dp;
                    dl += dh * g * rd;
                });
}

// One block per step: sums over (b, m) into part[t][8]: rel, max rel, count
// of rel > 1e-3, rel_w, max(rel_w, floor), activity, update norm; and z, u.
constexpr int kStatCols = 9;

template <typename F>
__device__ __forceinline__ float block_reduce(float x, float (&s)[4], F f) {
    for (int m = 32; m >= 1; m >>= 1) x = f(x, __shfl_xor(x, m));
    __syncthreads();
    if (threadIdx.x % 64 == 0) s[threadIdx.x / 64] = x;
    __syncthreads();
    return f(f(s[0], s[1]), f(s[2], s[3]));
}

__global__ __launch_bounds__(256) void stats_step_kernel(ScreenStatsArgs A) {
    __shared__ float s[4];
    const int64_t t = blockIdx.x, n = A.B * A.M;
    float v[kStatCols] = {};
    v[1] = -__builtin_inff();
    for (int64_t i = threadIdx.x; i < n; i += 256) {
        const int64_t at = (i / A.M * A.T + t) * A.M + i % A.M;
        const float r = A.rel[at];
        const float w = A.rel_w ? A.rel_w[at] : 0.f;
        v[0] += r;
        v[1] = larger(r, v[1]);
        v[2] += r > 1e-3f ? 1.f : 0.f;
        v[3] += w;
        v[4] += A.rel_w ? larger(w, A.floor) : 0.f;
        v[5] += A.rel_w ? larger(r, w) : r;
        float u = 0.f;
        for (int64_t j = 0; j < A.ndw; ++j) u += A.upd2[at * A.ndw + j];
        v[6] += sqrtf(u);
    }
    for (int64_t b = threadIdx.x; b < A.B; b += 256) {
        v[7] += A.z_norm[b * A.T + t];
        v[8] += A.u_norm[b * A.T + t];
    }
    for (int k = 0; k < kStatCols; ++k) {
        const float x =
            k == 1 ? block_reduce(v[k], s, larger)
                   : block_reduce(v[k], s,
                                  [](float a, float b) { return a + b; });
        if (threadIdx.x == 0) A.part[t * kStatCols + k] = x;
    }
}

// Block 0: the statistics, in float64 over the steps; the others, one per
// batch row: usage_T = d^T usage_0 + (1 - d) sum_t d^(T-1-t) activity_t.
__global__ __launch_bounds__(256) void stats_final_kernel(ScreenStatsArgs A) {
    __shared__ double s[256];
    const double T = double(A.T), n = double(A.B) * double(A.M);
    if (blockIdx.x == 0) {
        for (int k = 0; k <= kStatCols; ++k) {
            // the last one: the time mean of the EMA, from the activities
            double x = 0.0;
            for (int64_t t = threadIdx.x; t < A.T; t += 256)
                x += k < kStatCols
                         ? double(A.part[t * kStatCols + k])
                         : double(A.part[t * kStatCols + 5]) / n *
                               (1.0 - pow(A.decay, double(A.T - t)));
            if (k == kStatCols) {
                double u0 = 0.0;
                for (int64_t i = threadIdx.x; i < A.B * A.M; i += 256)
                    u0 += double(A.usage0[i]);
                const double d = A.decay;
                x += u0 / n * (d == 1.0 ? T : d * (1.0 - pow(d, T)) / (1.0 - d));
            }
            __syncthreads();
            s[threadIdx.x] = x;
            __syncthreads();
            for (int m = 128; m >= 1; m >>= 1) {
                if (int(threadIdx.x) < m)
                    s[threadIdx.x] += s[threadIdx.x + m];
                __syncthreads();
            }
            if (threadIdx.x == 0) {
                const double per = k == 1 || k == 9 ? T
                                   : k == 2         ? T * double(A.B)
                                   : k >= 7         ? T * double(A.B)
                                                    : T * n;
                A.stats[k] = float(s[0] / per);
            }
        }
        return;
    }
    // M columns by 256 / M runs of steps (or one run, M columns at a time)
    const int64_t b = blockIdx.x - 1;
    const int runs = A.M < 256 ? int(256 / A.M) : 1;
    for (int64_t m0 = 0; m0 < A.M; m0 += 256) {
        const int cols = int(A.M - m0 < 256 ? A.M - m0 : 256);
        const int run = threadIdx.x / cols;
        const int64_t m = m0 + threadIdx.x % cols;
        double x = 0.0;
        if (run < runs)
            for (int64_t t = run; t < A.T; t += runs) {
                const int64_t at = (b * A.T + t) * A.M + m;
                const float r = A.rel[at];
                const float a = A.rel_w ? larger(r, A.rel_w[at]) : r;
                x += double(a) * pow(A.decay, double(A.T - 1 - t));
            }
        __syncthreads();
        s[threadIdx.x] = x;
        __syncthreads();
        if (int(threadIdx.x) < cols) {
            double sum = 0.0;
            for (int k = 0; k < runs; ++k) sum += s[k * cols + threadIdx.x];
            A.usage_T[b * A.M + m] =
                float((1.0 - A.decay) * sum +
                      pow(A.decay, T) * double(A.usage0[b * A.M + m]));
        }
    }
}

dim3 row_grid(int64_t rows) { return dim3(unsigned((rows + 3) / 4)); }
dim3 col_grid(int64_t C, int64_t groups) {
    return dim3(unsigned((C + 63) / 64), unsigned(groups));
}

template <typename E, typename H>
void residual(bool backward, const ScreenResidualArgs& A, hipStream_t s) {
    const dim3 grid = col_grid(A.C, screen_row_groups(A.rows));
    if (backward)
        hipLaunchKernelGGL((residual_bwd_kernel<E, H>), grid, dim3(256), 0, s,
                           A);
    else
        hipLaunchKernelGGL((residual_fwd_kernel<E, H>), grid, dim3(256), 0, s,
                           A);
}

}  // namespace

// Row groups of the column sums: 16 rows each, at most 256 groups (with the
// presets' 12 column tiles 3072 blocks; more groups only lengthen the final
// addition).
int64_t screen_row_groups(int64_t rows) {
    const int64_t g = (rows + 15) / 16;
    return g < 1 ? 1 : g > 256 ? 256 : g;
}

hipError_t launch_screen_unit(bool bf16, bool backward,
                              const ScreenUnitArgs& A, hipStream_t s) {
    const dim3 grid = row_grid(A.rows);
    if (backward) {
        if (bf16)
            hipLaunchKernelGGL(unit_bwd_kernel<bf16_t>, grid, dim3(256), 0, s, A);
        else
            hipLaunchKernelGGL(unit_bwd_kernel<float>, grid, dim3(256), 0, s, A);
    } else {
        if (bf16)
            hipLaunchKernelGGL(unit_fwd_kernel<bf16_t>, grid, dim3(256), 0, s, A);
        else
            hipLaunchKernelGGL(unit_fwd_kernel<float>, grid, dim3(256), 0, s, A);
    }
    return hipGetLastError();
}

hipError_t launch_screen_residual(bool pre_bf16, bool h_bf16, bool backward,
                                  const ScreenResidualArgs& A, hipStream_t s) {
    if (pre_bf16)
        h_bf16 ? residual<bf16_t, bf16_t>(backward, A, s)
               : residual<bf16_t, float>(backward, A, s);
    else
        h_bf16 ? residual<float, bf16_t>(backward, A, s)
               : residual<float, float>(backward, A, s);
    return hipGetLastError();
}

hipError_t launch_screen_stats(const ScreenStatsArgs& A, hipStream_t s) {
    hipLaunchKernelGGL(stats_step_kernel, dim3(unsigned(A.T)), dim3(256), 0, s,
                       A);
    hipLaunchKernelGGL(stats_final_kernel, dim3(unsigned(A.B + 1)), dim3(256),
                       0, s, A);
    return hipGetLastError();
}

}  // namespace rwkv7m
