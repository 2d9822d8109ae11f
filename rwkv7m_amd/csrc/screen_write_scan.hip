// The write phase's slot recurrence (read_write; src/rwkv7m/model/
// nnx_model.py:1040-1047, :1103-1115) with the write key carried along
// instead of projected from the slots at every step.
//
// The key K_t = (S_t + e) W is linear in the slots, and the slots move by
// S_{t+1} = S_t + s_t (delta_t - S_t), so
//     K_{t+1} = K_t + s_t (D_t - K_t),   D_t = (delta_t + e) W,
// with the D_t of all steps one product of [B T M, d_slot] by W before the
// serial pass.  A step then holds no matrix-vector product, only wave sums:
// |K|^2 and K . q, which the next step waits for, and the update norm of each
// 64 channels, which it does not.  K runs in float64, so that what it loses
// against the projection of the slots is the slots' own rounding.  fp32 only:
// with the slots and the key rounded to bf16 the key follows no recurrence.
//
// Backward: d K_t = dsim_t p_t with p_t = (q - k^ sim) / |K| known from the
// forward, so its projection back to the slots is dsim_t (p_t W^T): again one
// product for all steps, and a step holds one wave sum (the cotangent of its
// strength).  The queries' and keys' cotangents follow per token afterwards.
//
// One chain wave per (b, slot) with the slot's channels (lane + 64 i) and the
// key's columns in registers; the other waves stage the next steps' inputs in
// LDS, two for each array of d_slot columns.  (One staging wave, as in the
// projecting kernels of screen_kernels.hip, was the bound: its loads' round
// trips took 0.75 us a step forward and 1.14 backward, more than the chain.)
//
// Bound by the latency of a step.  At 128 slots x 512 steps of 128 channels,
// keys of 64 (B = 8, M = 16), before (projecting kernels) -> now: forward
// 570 -> 338 us, backward 958 -> 214 us, and 44 + 18 + 43 + 19 us in the
// passes that form the deltas' keys, the keys' cotangents and their
// projection, and the queries'.  Those projections are this file's own kernels:
// a library product would follow the caller's autocast and precision settings.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "wkv7_common.h"
#include "wkv7_launch.h"

namespace rwkv7m {
namespace {

constexpr int kStage = 2048;  // floats per staged array and buffer
constexpr int kMaxSteps = 32;
constexpr int kFwdThreads = 64 * 5;  // the chain; deltas x2, queries, keys
constexpr int kBwdThreads = 64 * 9;  // the chain; four arrays x2

__device__ __forceinline__ float wave_total(float x) {
    return add_swap<32>(add_swap<16>(group_sum<16>(x)));
}

__device__ __forceinline__ int chunk_steps(int64_t ds, int dk) {
    const int n = kStage / int(ds > dk ? ds : dk);
    return n < kMaxSteps ? n : kMaxSteps;
}

// Wave `part` of `parts` stages its batches of n rows of `width`, `stride`
// elements apart, as fp32: 16 loads a lane in flight, from clamped in-bounds
// addresses.
template <typename F>
__device__ __forceinline__ void stage(float* dst, const float* src, int64_t stride,
                                      int n, int width, F f, int part,
                                      int parts) {
    const int lane = threadIdx.x % 64, tot = n * width;
    for (int b0 = part * 64 * 16; b0 < tot; b0 += parts * 64 * 16) {
        float v[16];
        int col[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int i = b0 + lane + 64 * r, ic = i < tot ? i : tot - 1;
            const int u = ic / width;
            col[r] = ic - u * width;
            v[r] = src[u * stride + col[r]];
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int i = b0 + lane + 64 * r;
            if (i < tot) dst[i] = f(v[r], col[r]);
        }
    }
}

// The two products around the scans: a wave takes H tiles of 16 rows
// (b, t, m), its lane l (i = l % 16, q = l / 16) the operands of row i,
// columns 4q .. 4q + 3 of each 16, and of the result's rows 4e + q, column i
// of each 16.  Sums in float64 (v_mfma_f64_16x16x4_f64), rounded once.  At 65536
// rows of 128, keys of 64, 44 and 43 us for 1.07 GFLOP each: above the matrix
// core's 14 and the 50 MB's 10 by the loads' round trips.  (Two tiles a wave
// for the first took 54, one for the second 71; a block's loads ahead of the
// products of the block before 48 each.)
using d4 = double __attribute__((ext_vector_type(4)));

template <int H>
struct ProductRows {
    int64_t rows, row0;
    int i, q;
    __device__ __forceinline__ explicit ProductRows(const ScreenScanWArgs& A)
        : rows(A.B * A.T * A.M),
          row0((int64_t(blockIdx.x) * 4 + threadIdx.x / 64) * 16 * H),
          i(threadIdx.x % 16),
          q(threadIdx.x % 64 / 16) {}
    // this lane's operand row of tile h (the last row past the end)
    __device__ __forceinline__ int64_t in(int h) const {
        const int64_t r = row0 + 16 * h + i;
        return r < rows ? r : rows - 1;
    }
    __device__ __forceinline__ int64_t out(int h, int e) const {
        return row0 + 16 * h + 4 * e + q;
    }
};

// D_t = (delta_t + slot_embed) W for every step.
template <int NJ>
__global__ __launch_bounds__(256) void write_delta_keys_kernel(
    ScreenScanWArgs A) {
    const ProductRows<1> R(A);
    if (R.row0 >= R.rows) return;
    const int ds = int(A.ds), dk = A.dk;
    const int64_t row = R.in(0), tok = row / A.M, m = row - tok * A.M;
    const float* base = A.base + tok * ds;
    const float* st = A.slot_term + m * ds;
    const float* se = A.slot_embed + m * ds;
    d4 acc[NJ] = {};
    for (int c0 = 0; c0 < ds; c0 += 16) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int c = c0 + 4 * R.q + e, cc = c < ds ? c : ds - 1;
            const float x = tanhf(base[cc] + st[cc]) + se[cc];
            const double a = c < ds ? double(x) : 0.0;
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int col = 16 * j + R.i;
                const float w = A.kw[cc * dk + (col < dk ? col : dk - 1)];
                acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                    a, c < ds ? double(w) : 0.0, acc[j], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int64_t r = R.out(0, e);
            if (r < R.rows && 16 * j + R.i < dk)
                A.delta_keys_out[r * dk + 16 * j + R.i] = float(acc[j][e]);
        }
}

// wp = p W^T.
template <int NJ>
__global__ __launch_bounds__(256) void write_back_kernel(ScreenScanWArgs A) {
    const ProductRows<2> R(A);
    if (R.row0 >= R.rows) return;
    const int ds = int(A.ds), dk = A.dk;
    float x[2][NJ][4];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int k = 16 * j + 4 * R.q + e;
                x[h][j][e] = A.p[R.in(h) * dk + (k < dk ? k : dk - 1)];
                x[h][j][e] = k < dk ? x[h][j][e] : 0.f;
            }
    for (int c0 = 0; c0 < ds; c0 += 16) {
        const float* w = A.kw + (c0 + R.i < ds ? c0 + R.i : ds - 1) * dk;
        float wv[NJ][4];
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int k = 16 * j + 4 * R.q + e;
                wv[j][e] = w[k < dk ? k : dk - 1];
                wv[j][e] = k < dk ? wv[j][e] : 0.f;
            }
        d4 acc[2] = {};
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    acc[h] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                        double(x[h][j][e]), double(wv[j][e]), acc[h], 0, 0, 0);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t r = R.out(h, e);
                if (r < R.rows && c0 + R.i < ds)
                    A.wp_out[r * ds + c0 + R.i] = float(acc[h][e]);
            }
    }
}

template <int NCH>
__global__ __launch_bounds__(kFwdThreads) void write_scan_fwd_kernel(
    ScreenScanWArgs A) {
    __shared__ float sd[2][kStage], sq[2][kStage], sk[2][kStage];
    const int lane = threadIdx.x % 64;
    const int wave = threadIdx.x / 64;
    const bool chain = wave == 0;
    const int64_t b = blockIdx.x / A.M, m = blockIdx.x % A.M;
    const int64_t T = A.T, M = A.M, bm0 = b * T * M + m;
    const int ds = int(A.ds), dk = A.dk, ndw = (ds + 63) / 64;
    const float* base = A.base + b * T * ds;
    const float* st = A.slot_term + m * ds;
    float* seq = A.slots_seq;
    const float mu = A.mu[m], tau = *A.tau_w, den = 1.f - tau + A.eps;
    const int chunk = chunk_steps(ds, dk);
    const int64_t nch = (T + chunk - 1) / chunk;
    auto fill = [&](int64_t ci) {
        const int64_t t0 = ci * chunk;
        const int n = int(T - t0 < chunk ? T - t0 : chunk), buf = int(ci & 1);
        const auto id = [](float x, int) { return x; };
        if (wave <= 2)
            stage(sd[buf], base + t0 * ds, ds, n, ds,
                  [&](float x, int c) { return tanhf(x + st[c]); }, wave - 1,
                  2);
        else if (wave == 3)
            stage(sq[buf], A.q_w + (b * T + t0) * dk, dk, n, dk, id, 0, 1);
        else
            stage(sk[buf], A.delta_keys + (bm0 + t0 * M) * dk, M * dk, n, dk,
                  id, 0, 1);
    };
    float S[NCH];
    double K[2] = {0.0, 0.0};
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int c = lane + 64 * i;
        S[i] = c < ds ? A.slots0[(b * M + m) * ds + c] : 0.f;
    }
    if (chain) {  // K_0
        for (int c = 0; c < ds; ++c) {
            const double x = double(A.slots0[(b * M + m) * ds + c]) +
                             double(A.slot_embed[m * ds + c]);
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (lane + 64 * h < dk)
                    K[h] += x * double(A.kw[int64_t(c) * dk + lane + 64 * h]);
        }
    }
    float age = A.ages0[b * M + m];
    if (!chain && nch > 0) fill(0);
    __syncthreads();
    for (int64_t ci = 0; ci < nch; ++ci) {
        if (!chain) {
            if (ci + 1 < nch) fill(ci + 1);
        } else {
            const int buf = int(ci & 1);
            const int64_t t0 = ci * chunk;
            const int n = int(T - t0 < chunk ? T - t0 : chunk);
            for (int u = 0; u < n; ++u) {
                float q[2], D[2], k[2], dl[NCH], kk = 0.f, dot = 0.f;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int j = lane + 64 * h;
                    q[h] = j < dk ? sq[buf][u * dk + j] : 0.f;
                    D[h] = j < dk ? sk[buf][u * dk + j] : 0.f;
                    k[h] = float(K[h]);
                    kk += k[h] * k[h];
                    dot += k[h] * q[h];
                }
#pragma unroll
                for (int i = 0; i < NCH; ++i) {
                    const int c = lane + 64 * i;
                    dl[i] = c < ds ? sd[buf][u * ds + c] : 0.f;
                }
                kk = wave_total(kk);
                dot = wave_total(dot);
                const float sim = dot / sqrtf(kk + A.eps * A.eps);
                const float x = fmaxf((sim - tau) / den, 0.f);
                const float rw = x * x, s = mu * fmaxf(rw, A.floor);
                const int64_t row = bm0 + (t0 + u) * M;
                if (lane == 0) {
                    A.rel_w[row] = rw;
                    A.ages_seq[row] = age;
                }
                age = rw > 1e-3f ? 0.f : age + 1.f;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int j = lane + 64 * h;
                    if (j < dk) A.keys[row * dk + j] = k[h];
                    K[h] += double(s) * (double(D[h]) - K[h]);
                }
#pragma unroll
                for (int i = 0; i < NCH; ++i) {
                    if (64 * i >= ds) break;
                    const int c = lane + 64 * i;
                    const bool in = c < ds;
                    if (in) {
                        seq[row * ds + c] = S[i];
                        A.slots32[row * ds + c] = S[i];
                    }
                    const float du = in ? s * (dl[i] - S[i]) : 0.f;
                    const float u2 = wave_total(du * du);
                    if (lane == 0) A.upd2[row * ndw + i] = u2;
                    S[i] += du;
                }
            }
        }
        __syncthreads();  // chunk ci is read, chunk ci + 1 is staged
    }
    if (chain) {
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int c = lane + 64 * i;
            if (c < ds) A.slots_T[(b * M + m) * ds + c] = S[i];
        }
        if (lane == 0) A.ages_T[b * M + m] = age;
    }
}

// |K| with eps, and sim, of one row; every lane active.
struct KeyRow {
    float k[2], q[2], kn, sim;
    __device__ __forceinline__ KeyRow(const float* keys, const float* qw,
                                      int dk, float eps) {
        const int lane = threadIdx.x % 64;
        float kk = 0.f, dot = 0.f;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int j = lane + 64 * h;
            k[h] = j < dk ? keys[j] : 0.f;
            q[h] = j < dk ? qw[j] : 0.f;
            kk += k[h] * k[h];
            dot += k[h] * q[h];
        }
        kn = sqrtf(wave_total(kk) + eps * eps);
        sim = wave_total(dot) / kn;
    }
};

// p = (q - k^ sim) / |K| and sim, a wave per (b, t, m).
__global__ __launch_bounds__(256) void write_keys_kernel(ScreenScanWArgs A) {
    const int64_t row = int64_t(blockIdx.x) * 4 + threadIdx.x / 64;
    if (row >= A.B * A.T * A.M) return;
    const int lane = threadIdx.x % 64, dk = A.dk;
    const KeyRow r(A.keys + row * dk, A.q_w + row / A.M * dk, dk, A.eps);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int j = lane + 64 * h;
        if (j < dk)
            A.p[row * dk + j] = (r.q[h] - r.k[h] / r.kn * r.sim) / r.kn;
    }
    if (lane == 0) A.sim[row] = r.sim;
}

// After the scan: d K = dsim p in place of p, dq = sum_m dsim k^; a wave per
// (b, t).
__global__ __launch_bounds__(256) void write_queries_kernel(
    ScreenScanWArgs A) {
    const int64_t tok = int64_t(blockIdx.x) * 4 + threadIdx.x / 64;
    if (tok >= A.B * A.T) return;
    const int lane = threadIdx.x % 64, dk = A.dk;
    float dq[2] = {0.f, 0.f};
    for (int64_t m = 0; m < A.M; ++m) {
        const int64_t row = tok * A.M + m;
        const KeyRow r(A.keys + row * dk, A.keys + row * dk, dk, A.eps);
        const float g = A.d_sim[row];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int j = lane + 64 * h;
            dq[h] += g * (r.k[h] / r.kn);
            if (j < dk) A.p[row * dk + j] *= g;
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
        if (lane + 64 * h < dk) A.dq_w[tok * dk + lane + 64 * h] = dq[h];
}

template <int NCH>
__global__ __launch_bounds__(kBwdThreads) void write_scan_bwd_kernel(
    ScreenScanWArgs A) {
    __shared__ float sth[2][kStage], ss[2][kStage], sg[2][kStage],
        sp[2][kStage];
    __shared__ float ssim[2][kMaxSteps], srel[2][kMaxSteps],
        sage[2][kMaxSteps];
    const int lane = threadIdx.x % 64;
    const int wave = threadIdx.x / 64;
    const bool chain = wave == 0;
    const int64_t b = blockIdx.x / A.M, m = blockIdx.x % A.M;
    const int64_t T = A.T, M = A.M, bm0 = b * T * M + m;
    const int ds = int(A.ds);
    const float* base = A.base + b * T * ds;
    const float* dseq = A.d_slots_seq + bm0 * ds;
    const float* st = A.slot_term + m * ds;
    const int64_t Mds = M * ds;
    const float mu = A.mu[m], tau = *A.tau_w, den = 1.f - tau + A.eps;
    const int chunk = chunk_steps(ds, 1);
    const int64_t nch = (T + chunk - 1) / chunk;
    auto fill = [&](int64_t ci) {
        const int64_t t0 = ci * chunk;
        const int n = int(T - t0 < chunk ? T - t0 : chunk), buf = int(ci & 1);
        const auto id = [](float x, int) { return x; };
        const int half = wave & 1;
        if (wave <= 2)
            stage(sth[buf], base + t0 * ds, ds, n, ds,
                  [&](float x, int c) { return tanhf(x + st[c]); }, half, 2);
        else if (wave <= 4)
            stage(ss[buf], A.slots32 + bm0 * ds + t0 * Mds, Mds, n, ds, id,
                  half, 2);
        else if (wave <= 6)
            stage(sg[buf], dseq + t0 * Mds, Mds, n, ds, id, half, 2);
        else
            stage(sp[buf], A.wp + bm0 * ds + t0 * Mds, Mds, n, ds, id, half,
                  2);
        if (wave == 1 && lane < n) {
            const int64_t row = bm0 + (t0 + lane) * M;
            ssim[buf][lane] = A.sim[row];
            srel[buf][lane] = A.d_rel_w ? A.d_rel_w[row] : 0.f;
            sage[buf][lane] = A.d_ages_seq ? A.d_ages_seq[row] : 0.f;
        }
    };
    float G[NCH], de[NCH];
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int c = lane + 64 * i;
        G[i] = c < ds && A.d_slots_T ? A.d_slots_T[(b * M + m) * ds + c] : 0.f;
        de[i] = 0.f;
    }
    float dage = A.d_ages_T ? A.d_ages_T[b * M + m] : 0.f, dmu = 0.f;
    if (!chain && nch > 0) fill(nch - 1);
    __syncthreads();
    for (int64_t ci = nch - 1; ci >= 0; --ci) {
        if (!chain) {
            if (ci > 0) fill(ci - 1);
        } else {
            const int buf = int(ci & 1);
            const int64_t t0 = ci * chunk;
            const int n = int(T - t0 < chunk ? T - t0 : chunk);
            for (int u = n - 1; u >= 0; --u) {
                const int64_t row = bm0 + (t0 + u) * M;
                const float x = (ssim[buf][u] - tau) / den;
                const float r = fmaxf(x, 0.f), rw = r * r;
                const float act = fmaxf(rw, A.floor), s = mu * act;
                float th[NCH], gv[NCH], wp[NCH], part = 0.f;
#pragma unroll
                for (int i = 0; i < NCH; ++i) {
                    const int c = lane + 64 * i;
                    const bool in = c < ds;
                    th[i] = in ? sth[buf][u * ds + c] : 0.f;
                    gv[i] = in ? sg[buf][u * ds + c] : 0.f;
                    wp[i] = in ? sp[buf][u * ds + c] : 0.f;
                    if (in)
                        part += G[i] * (th[i] - ss[buf][u * ds + c]);
                }
                const float dstr = wave_total(part);
                const float drw = srel[buf][u] + (rw > A.floor ? dstr * mu : 0.f);
                const float dsim = drw * 2.f * r / den;
                dmu += dstr * act;
                if (lane == 0) {
                    A.d_sim[row] = dsim;
                    A.d_tau_w[row] = drw * 2.f * r * (x - 1.f) / den;
                }
                dage = sage[buf][u] + (rw > 1e-3f ? 0.f : dage);
#pragma unroll
                for (int i = 0; i < NCH; ++i) {
                    const int c = lane + 64 * i;
                    if (c >= ds) continue;
                    const float dsk = dsim * wp[i];
                    de[i] += dsk;
                    A.d_pre[row * ds + c] = s * G[i] * (1.f - th[i] * th[i]);
                    G[i] = G[i] * (1.f - s) + dsk + gv[i];
                }
            }
        }
        __syncthreads();  // chunk ci is read, chunk ci - 1 is staged
    }
    if (chain) {
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int c = lane + 64 * i;
            if (c < ds) {
                A.d_slots0[(b * M + m) * ds + c] = G[i];
                A.d_embed_part[(b * M + m) * ds + c] = de[i];
            }
        }
        if (lane == 0) {
            A.d_ages0[b * M + m] = dage;
            A.d_mu_bm[b * M + m] = dmu;
        }
    }
}

template <int NCH>
void scan_n(bool backward, const ScreenScanWArgs& A, hipStream_t s) {
    const dim3 grid{unsigned(A.B * A.M)};
    if (backward)
        hipLaunchKernelGGL((write_scan_bwd_kernel<NCH>), grid,
                           dim3(kBwdThreads), 0, s, A);
    else
        hipLaunchKernelGGL((write_scan_fwd_kernel<NCH>), grid,
                           dim3(kFwdThreads), 0, s, A);
}

dim3 product_grid(const ScreenScanWArgs& A, int tiles) {
    const int64_t rows = 64 * tiles;
    return dim3(unsigned((A.B * A.T * A.M + rows - 1) / rows));
}

}  // namespace

hipError_t launch_screen_write_delta_keys(const ScreenScanWArgs& A,
                                          hipStream_t s) {
    if (A.dk <= 64)
        hipLaunchKernelGGL((write_delta_keys_kernel<4>), product_grid(A, 1),
                           dim3(256), 0, s, A);
    else
        hipLaunchKernelGGL((write_delta_keys_kernel<8>), product_grid(A, 1),
                           dim3(256), 0, s, A);
    return hipGetLastError();
}

// Channels per lane: 2 and 4 at the presets (d_slot 128, 256).
hipError_t launch_screen_write_scan(bool backward, const ScreenScanWArgs& A,
                                    hipStream_t s) {
    if (A.ds <= 128)
        scan_n<2>(backward, A, s);
    else if (A.ds <= 256)
        scan_n<4>(backward, A, s);
    else
        scan_n<16>(backward, A, s);
    return hipGetLastError();
}

hipError_t launch_screen_write_keys(const ScreenScanWArgs& A, hipStream_t s) {
    hipLaunchKernelGGL(write_keys_kernel,
                       dim3(unsigned((A.B * A.T * A.M + 3) / 4)), dim3(256), 0,
                       s, A);
    if (A.dk <= 64)
        hipLaunchKernelGGL((write_back_kernel<4>), product_grid(A, 2), dim3(256),
                           0, s, A);
    else
        hipLaunchKernelGGL((write_back_kernel<8>), product_grid(A, 2), dim3(256),
                           0, s, A);
    return hipGetLastError();
}

hipError_t launch_screen_write_queries(const ScreenScanWArgs& A,
                                       hipStream_t s) {
    hipLaunchKernelGGL(write_queries_kernel,
                       dim3(unsigned((A.B * A.T + 3) / 4)), dim3(256), 0, s,
                       A);
    return hipGetLastError();
}

}  // namespace rwkv7m
