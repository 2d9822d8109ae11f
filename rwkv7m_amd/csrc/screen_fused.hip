// Elementwise and reduction passes of the screening module around its GEMMs
// and recurrences (src/rwkv7m/model/nnx_model.py:1015-1160): the gated
// residual, and the usage EMA with the statistics.  As single torch operations
// these were about fifty launches of a few MB each in a training step, with a
// host cost per launch above its device time; every pass here reads its inputs
// once.  At the 0.185B preset (4096 rows of 768) a training step issued op by
// op goes from 2.35 to 1.89 ms in the read phase (bf16).

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "wkv7_common.h"
#include "wkv7_launch.h"

namespace rwkv7m {
namespace {

__device__ __forceinline__ float sigmoid(float x) {
    return 1.f / (1.f + expf(-x));
}

// The larger, a NaN if either is one (as torch.maximum).
__device__ __forceinline__ float larger(float a, float b) {
    return a > b || a != a ? a : b;
}

// h = h_base + lam sigmoid(pre) read, element by element, each operation
// rounded as torch's separate ones are (no contraction), so that the results
// and the gradients are theirs bit for bit: in bf16 a coarser or finer sum
// turns roundings that move some gradients by 1e-3.  The sums over the
// gradients' elements (of the gate's bias and of lam) are the caller's.
// Bound by memory: see the file's header for the rate.
template <typename E, typename H>
__global__ __launch_bounds__(256) void residual_fwd_kernel(
    ScreenResidualArgs A) {
#pragma clang fp contract(off)
    const float lam = *A.lam;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < A.n;
         i += 256 * int64_t(gridDim.x)) {
        const float g = sigmoid(load_f(static_cast<const E*>(A.pre) + i));
        const float u = lam * g * load_f(static_cast<const H*>(A.read) + i);
        store_f(static_cast<H*>(A.h) + i,
                load_f(static_cast<const H*>(A.h_base) + i) + u);
    }
}

template <typename E, typename H>
__global__ __launch_bounds__(256) void residual_bwd_kernel(
    ScreenResidualArgs A) {
#pragma clang fp contract(off)
    const float lam = *A.lam;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < A.n;
         i += 256 * int64_t(gridDim.x)) {
        const float g = sigmoid(load_f(static_cast<const E*>(A.pre) + i));
        const float dh = load_f(static_cast<const H*>(A.dh) + i);
        const float dt = dh * load_f(static_cast<const H*>(A.read) + i);
        store_f(static_cast<H*>(A.d_read) + i, dh * (lam * g));
        store_f(static_cast<E*>(A.d_pre) + i, dt * lam * (1.f - g) * g);
        A.d_lam[i] = dt * g;
    }
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

template <typename E, typename H>
void residual(bool backward, const ScreenResidualArgs& A, hipStream_t s) {
    // at most 16 workgroups a CU: 3072 elements each at the preset's 3 M
    const int64_t g = (A.n + 255) / 256;
    const dim3 grid(unsigned(g < 4096 ? g : 4096));
    if (backward)
        hipLaunchKernelGGL((residual_bwd_kernel<E, H>), grid, dim3(256), 0, s,
                           A);
    else
        hipLaunchKernelGGL((residual_fwd_kernel<E, H>), grid, dim3(256), 0, s,
                           A);
}

}  // namespace

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
