// Chunked WKV-7 in fp32 on the matrix cores (gfx950): fp32 vectors, and bf16
// vectors with N = 16, 32 or 128, whose arithmetic stays fp32 throughout.
// The products are v_mfma_f32_16x16x4_f32, those of a chunk's own 16x16 matrices
// and of the state's and its cotangent's update v_mfma_f64_16x16x4_f64; nothing
// is rounded to 16 bits.
//
// A chunk is L = 16 tokens of one head.  With P_t = d_1 ... d_t (per column;
// P_0 = 1, d = exp(-exp(w))) and
//     A~_t = a_t P_{t-1},  R~_t = r_t P_t,  B~_t = b_t / P_t,  K~_t = k_t / P_t
// and the 16x16 matrices Aab = A~ B~^T, Aak = A~ K~^T (strictly lower),
// Arb = R~ B~^T, Ark = R~ K~^T (lower), Minv = (I - Aab)^-1, the recurrence
// (reference src/rwkv7m/model/rwkv_core.py:54-86) is, over a chunk,
//     X   = W S0^T + Mak V            W = Minv A~,  Mak = Minv Aak
//     Y   = R~ S0^T + Arb X + Ark V
//     S_L = S0 diag(P_L) + X^T B^ + V^T K^    B^_t = b_t P_L / P_t, K^ alike
// and its reverse (src/rwkv7m/kernels/wkv_pallas_gpu.py:221-257), from the
// cotangent D of S_L, with D^ = D diag(P_L),
//     dU  = Wb D^^T + G dY            Wb = Minv^T B~,  G = Minv^T Arb^T
//     D0  = D^ + dU^T A~ + dY^T R~
//     dV  = K~ D^^T + Ark^T dY + Aak^T dU
//     dR~ = dY S0 + dArb B~ + dArk K~,      dA~ = dU S0 + dAab B~ + dAak K~
//     dB~ = X D^ + dArb^T R~ + dAab^T A~,   dK~ = V D^ + dArk^T R~ + dAak^T A~
// with dArb = dY X^T, dArk = dY V^T, dAab = dU X^T, dAak = dU V^T (masked),
//     dlog d_t = sum_{t'>=t} (R~ dR~ - B~ (dB~ - X D^) - K~ (dK~ - V D^))_t'
//              + sum_{t'>t} (A~ dA~)_t'
//              + sum_{t'<t} (B~ (X D^) + K~ (V D^))_t' + sum_i D^ S0.
//
// Both serial quantities (S forward, D backward) act row by row, so the work
// splits into three launches per direction with no hand-over inside one:
//   prep   one workgroup per chunk and head: factors, matrices, the inverse,
//          and the operands of the serial step in the order its lanes read;
//   chain  one wave per 16 state rows: 19 (N = 64) products of 16x16x16 a
//          chunk, the only serial part;
//   grads  (backward) one workgroup per chunk and head: the six gradients.
// The sequential kernels spend a token's time on reductions over the columns
// and rows of the state; here those are the products' sums.  Measured
// (forward with checkpoints / backward, before -> now): fp32, 96 heads of 64,
// 512 tokens 183 / 768 -> 140 / 200 us; bf16, 64 heads of 128, 1024 tokens
// 784 / 3598 -> 480 / 750 us.  Of that the float64 products are 44 and 139 us;
// without them (all float32) the errors below grew to what is said at
// `inverse` and at the chains.
//
// Errors against float64 (2-norm, fp32 vectors, 4 heads of 64, 512 tokens; in
// 1e-7, the sequential kernels' in brackets): independent keys as a model's
// y 0.8 (0.9), S_T 0.4 (0.6), dr 0.9 (1.0), dw 1.2 (1.3), dk 0.9 (1.1), dv 0.9
// (0.9), da 1.2 (1.4), db 1.2 (1.4), dS0 0.5 (0.6); keys within 0.1 of one
// direction, a near 0.95, slow decay y 2.0 (1.2), S_T 1.6 (1.1), dr 2.3 (1.4),
// dw 2.6 (1.8), dk 1.0 (1.3), dv 2.4 (2.0), da 2.6 (2.4), db 1.2 (1.4), dS0
// 0.6 (1.0); one key repeated, hardly any decay y 5.4 (4.6), S_T 6.2 (5.9),
// the gradients 5.6 to 11 (4.7 to 12).  The other head sizes are alike.
//
// Range: a chunk with P_L below 2^-60 (no trained decay comes near: the time
// mix's stays above 2^-14 a chunk), or a non-finite or huge value, is marked
// by its prep; the head then takes the sequential kernels for that time
// segment.
//
// Tile layouts.  A D tile of a 16x16 matrix M holds M[4q + e][l % 16] (lane
// l, q = l / 16, e = 0..3).  As the four 16x16x4 operands of a product over
// sixteen, it is M as the B operand and M^T as the A operand: mm(x, y) of D
// tiles of M^T and Y is a D tile of M Y.  A token-major 16xN matrix gives
// each lane 4 columns of one token (T form, a D tile of its transpose) or 4
// tokens of one column (J form, a D tile of it).

#include "wkv7_common.h"
#include "wkv7_launch.h"

namespace rwkv7m {
namespace {

using f4 = float __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f4 mm(f4 a, f4 b, f4 c) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
    return c;
}
constexpr f4 kZero = {0.f, 0.f, 0.f, 0.f};
__device__ __forceinline__ f4 mm(f4 a, f4 b) {
    f4 c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[0], b[0], kZero, 0, 0, 0);
    f4 d = __builtin_amdgcn_mfma_f32_16x16x4f32(a[2], b[2], kZero, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[1], b[1], c, 0, 0, 0);
    d = __builtin_amdgcn_mfma_f32_16x16x4f32(a[3], b[3], d, 0, 0, 0);
    return c + d;
}

// K independent products at once: a product's own two steps wait for each
// other, so the steps go round by round (a wave has its SIMD to itself here,
// and one product after the other left the matrix core idle a third of the
// time).  The sums follow behind the next use's products.
template <int K>
__device__ __forceinline__ void products(const f4 (&a)[K], const f4 (&b)[K],
                                         f4 (&o)[K]) {
    f4 c[K], d[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
        c[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][0], b[i][0], kZero, 0,
                                                    0, 0);
        d[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][2], b[i][2], kZero, 0,
                                                    0, 0);
    }
#pragma unroll
    for (int i = 0; i < K; ++i) {
        c[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][1], b[i][1], c[i], 0,
                                                    0, 0);
        d[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][3], b[i][3], d[i], 0,
                                                    0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < K; ++i) o[i] = c[i] + d[i];
}

// The same in float64, whose D tile holds rows 4e + q (an H tile): with A's
// rows permuted by i -> 4 (i % 4) + i / 4 (Rows::jp) the result's lanes are as
// mm's.  mm64(H tile of M^T, H tile of Y) is an H tile of M Y.
using d4 = double __attribute__((ext_vector_type(4)));
constexpr d4 kZero64 = {0., 0., 0., 0.};
template <typename A, typename B>
__device__ __forceinline__ d4 mm64(A a, B b, d4 c = kZero64) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
        c = __builtin_amdgcn_mfma_f64_16x16x4f64(a[e], b[e], c, 0, 0, 0);
    return c;
}

// term(0) + ... + term(n - 1), pairwise.  Products over more than 16 are
// summed as products over 16, each accumulated from zero: one long chain of
// accumulations rounds every step to the size of the whole sum (errors
// against float64 halve; the additions hide behind the products).
template <int LO, int HI, typename F>
__device__ __forceinline__ f4 tree(F term) {
    if constexpr (HI - LO == 1) {
        return term(LO);
    } else {
        constexpr int MID = (LO + HI) / 2;
        const f4 a = tree<LO, MID>(term);
        return a + tree<MID, HI>(term);
    }
}

// Four consecutive elements.
__device__ __forceinline__ f4 load4(const float* p) {
    return *reinterpret_cast<const f4*>(p);
}
__device__ __forceinline__ f4 load4(const bf16_t* p) {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    return f4{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u),
              __uint_as_float(u.y << 16), __uint_as_float(u.y & 0xffff0000u)};
}
__device__ __forceinline__ void store4(float* p, f4 x) {
    *reinterpret_cast<f4*>(p) = x;
}
__device__ __forceinline__ void store4(bf16_t* p, f4 x) {
    uint2 u;
    u.x = uint32_t(f32_to_bf16(x[0])) | uint32_t(f32_to_bf16(x[1])) << 16;
    u.y = uint32_t(f32_to_bf16(x[2])) | uint32_t(f32_to_bf16(x[3])) << 16;
    *reinterpret_cast<uint2*>(p) = u;
}

// x of lane t - n (row_shr) or t + n (row_shl) of the 16-lane row, `fill`
// where there is none.
template <int ctrl>
__device__ __forceinline__ int dpp_or(int fill, int x) {
    return __builtin_amdgcn_update_dpp(fill, x, ctrl, 0xf, 0xf, false);
}
template <int ctrl>
__device__ __forceinline__ float dpp_or(float fill, float x) {
    return __int_as_float(
        dpp_or<ctrl>(__float_as_int(fill), __float_as_int(x)));
}
template <int ctrl>
__device__ __forceinline__ double dpp_or(double fill, double x) {
    const int2 f = __builtin_bit_cast(int2, fill);
    const int2 v = __builtin_bit_cast(int2, x);
    return __builtin_bit_cast(
        double, int2{dpp_or<ctrl>(f.x, v.x), dpp_or<ctrl>(f.y, v.y)});
}
template <int n, typename F>
__device__ __forceinline__ F from_left(F x, F fill) {
    return dpp_or<0x110 + n>(fill, x);
}
template <int n, typename F>
__device__ __forceinline__ F from_right(F x, F fill) {
    return dpp_or<0x100 + n>(fill, x);
}
// The decay products run in float64: a factor and its inverse then carry one
// rounding each, and what a chunk multiplies together (P_L / P_s) two.
__device__ __forceinline__ double prefix_mul(double x) {
    x *= from_left<1>(x, 1.0);
    x *= from_left<2>(x, 1.0);
    x *= from_left<4>(x, 1.0);
    return x * from_left<8>(x, 1.0);
}
__device__ __forceinline__ float prefix_add(float x) {
    x += from_left<1>(x, 0.f);
    x += from_left<2>(x, 0.f);
    x += from_left<4>(x, 0.f);
    return x + from_left<8>(x, 0.f);
}
template <typename F>
__device__ __forceinline__ F suffix_add(F x) {
    x += from_right<1>(x, F(0));
    x += from_right<2>(x, F(0));
    x += from_right<4>(x, F(0));
    return x + from_right<8>(x, F(0));
}

// Workspace of one chunk of one head (offsets in floats).  Tiles are 256
// floats in lane order.
template <int N, bool BWD>
struct Ws {
    static constexpr int NB = N / 16;
    // forward: W, R~ in T form, B^, K^ in J form; Mak, Arb, Ark in T form;
    // backward: Wb in T form, A~, R~ in J form; G in T form, Ark, Aak D
    // tiles; then X, dU [16][N] and D^ [N][N]
    static constexpr int M0 = 0, M1 = NB * 256, M2 = 2 * NB * 256,
                         M3 = 3 * NB * 256;
    static constexpr int S = BWD ? M3 : 4 * NB * 256;  // the 16x16 tiles
    static constexpr int PL = S + 3 * 256;
    static constexpr int X = PL + N, U = X + 16 * N, DH = U + 16 * N;
    static constexpr int SIZE = BWD ? DH + N * N : PL + N;
};

struct Args {
    int64_t T, BH;  // of the whole call
    VecLayout lay;
    int64_t c0, nch;  // the segment's first chunk and chunk count
    const void *r, *w, *k, *v, *a, *b, *dy;
    const float* state_in;  // S0 (or dS_T; null: zero) of the segment
    float* state_out;
    void* y;
    float* ckpt;     // forward: written every ci / 16 chunks; null: none
    int64_t ck_every, ck_last;  // (chunks; the entry of the final state or -1)
    const float* ckpt_in;       // backward: S0 of every chunk
    void *dr, *dw, *dk, *dv, *da, *db;
    const void *add_dr, *add_dk, *add_dv;
    float* ws;
    int* flags;  // [nch][BH], nonzero: chunk out of range
};

__device__ __forceinline__ bool head_marked(const Args& A, int64_t bh) {
    int f = 0;
    for (int64_t i = threadIdx.x % 64; i < A.nch; i += 64)
        f |= A.flags[i * A.BH + bh];
    return __any(f);
}

// A lane's 4 columns of the chunk's factors at its token (T form).
struct Factors {
    f4 A, R, B, K, P, Pp, inv, ew;
    f4 Bh, Kh;  // B^ = b P_L / P_t, K^ (STATE only)
    bool bad;
};
constexpr float kMinP = 0x1p-60f, kMaxFactor = 0x1p90f;

template <typename VT, bool STATE = false>
__device__ __forceinline__ void factors(Factors& F, const Args& A, int64_t off,
                                        bool valid) {
    f4 r = kZero, w = kZero, k = kZero, a = kZero, b = kZero;
    if (valid) {
        r = load4(static_cast<const VT*>(A.r) + off);
        w = load4(static_cast<const VT*>(A.w) + off);
        k = load4(static_cast<const VT*>(A.k) + off);
        a = load4(static_cast<const VT*>(A.a) + off);
        b = load4(static_cast<const VT*>(A.b) + off);
    }
    F.bad = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        F.ew[e] = expf(w[e]);
        // a token past the end decays by nothing
        const double p = prefix_mul(valid ? double(expf(-F.ew[e])) : 1.0);
        const double pp = from_left<1>(p, 1.0), inv = 1.0 / p;
        F.P[e] = float(p);
        F.Pp[e] = float(pp);
        F.inv[e] = float(inv);
        F.A[e] = float(a[e] * pp);
        F.R[e] = float(r[e] * p);
        F.B[e] = float(b[e] * inv);
        F.K[e] = float(k[e] * inv);
        if constexpr (STATE) {
            const double left = __shfl(p, 15, 16) * inv;
            F.Bh[e] = float(b[e] * left);
            F.Kh[e] = float(k[e] * left);
        }
        // (written so that a NaN fails)
        F.bad |= !(F.P[e] >= kMinP) || !(fabsf(F.A[e]) < kMaxFactor) ||
                 !(fabsf(F.R[e]) < kMaxFactor) ||
                 !(fabsf(F.B[e]) < kMaxFactor) ||
                 !(fabsf(F.K[e]) < kMaxFactor);
    }
}

__device__ __forceinline__ bool out_of_range(f4 x) {
    bool bad = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) bad |= !(fabsf(x[e]) < kMaxFactor);
    return bad;
}

// Rows of a staged [16][N] matrix, padded so that T-form (16-byte) and J-form
// reads are free of bank conflicts.
template <int N>
struct Rows {
    float x[16][N + 4];
    __device__ __forceinline__ f4 t(int c, int l) const {
        return *reinterpret_cast<const f4*>(&x[l % 16][16 * c + 4 * (l / 16)]);
    }
    __device__ __forceinline__ f4 j(int c, int l) const {
        f4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = x[4 * (l / 16) + e][16 * c + l % 16];
        return o;
    }
    __device__ __forceinline__ f4 jp(int c, int l) const {
        f4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            o[e] = x[4 * (l / 16) + e][16 * c + 4 * (l % 4) + l % 16 / 4];
        return o;
    }
    __device__ __forceinline__ void put_t(int c, int l, f4 v) {
        *reinterpret_cast<f4*>(&x[l % 16][16 * c + 4 * (l / 16)]) = v;
    }
};

// A 16x16 matrix between waves: written from a D tile, read as a D tile of
// itself or of its transpose.
struct Mat {
    float x[16][20];
    __device__ __forceinline__ void put(int l, f4 d) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[4 * (l / 16) + e][l % 16] = d[e];
    }
    __device__ __forceinline__ f4 d(int l) const {
        f4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = x[4 * (l / 16) + e][l % 16];
        return o;
    }
    __device__ __forceinline__ f4 dt(int l) const {
        return *reinterpret_cast<const f4*>(&x[l % 16][4 * (l / 16)]);
    }
};

// A 16x16 matrix in float64 between lanes and waves, from an H tile.
struct Mat64 {
    double x[16][18];
    __device__ __forceinline__ void put(int l, d4 h) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[4 * e + l / 16][l % 16] = h[e];
    }
    __device__ __forceinline__ d4 h(int l) const {
        d4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = x[4 * e + l / 16][l % 16];
        return o;
    }
    // an H tile of the transpose
    __device__ __forceinline__ d4 ht(int l) const {
        d4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = x[l % 16][4 * e + l / 16];
        return o;
    }
    // rows 4q + e, as mm's tiles: of itself, of the transpose
    __device__ __forceinline__ d4 d(int l) const {
        d4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = x[4 * (l / 16) + e][l % 16];
        return o;
    }
    __device__ __forceinline__ d4 dt(int l) const {
        d4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = x[l % 16][4 * (l / 16) + e];
        return o;
    }
};

// An H tile, rounded, into a D tile's place in the workspace.
__device__ __forceinline__ void store_tile(float* tile, int l, d4 h) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
        tile[4 * (16 * e + l % 16) + l / 16] = float(h[e]);
}

// sum over columns of x y^T (both in T form): a D tile of the 16x16 product,
// and an H tile of it in float64.
template <int N>
__device__ __forceinline__ f4 outer(const Rows<N>& x, const Rows<N>& y,
                                    int l) {
    return tree<0, N / 16>([&](int c) { return mm(x.t(c, l), y.t(c, l)); });
}
template <int N>
__device__ __forceinline__ d4 outer64(const Rows<N>& x, const Rows<N>& y,
                                      int l) {
    d4 o = kZero64;
#pragma unroll
    for (int c = 0; c < N / 16; ++c) o = mm64(x.t(c, l), y.t(c, l), o);
    return o;
}

// D tile entries with row (4q + e) > column, or >= with the diagonal.
__device__ __forceinline__ f4 keep_lower(f4 d, int l, bool diag) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int i = 4 * (l / 16) + e, j = l % 16;
        d[e] = (i > j || (diag && i == j)) ? d[e] : 0.f;
    }
    return d;
}
// The same of an H tile (rows 4e + q), and of a matrix's transpose (upper).
__device__ __forceinline__ d4 keep_lower(d4 h, int l, bool diag) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int i = 4 * e + l / 16, j = l % 16;
        h[e] = (i > j || (diag && i == j)) ? h[e] : 0.;
    }
    return h;
}
__device__ __forceinline__ d4 keep_upper(d4 h, int l, bool diag) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int i = 4 * e + l / 16, j = l % 16;
        h[e] = (i < j || (diag && i == j)) ? h[e] : 0.;
    }
    return h;
}

// (I - A)^-1 of a strictly lower 16x16 A:
// (I + A)(I + A^2)(I + A^4)(I + A^8), A nilpotent.  a, at: H tiles of A and
// A^T.  In float64: with keys that resemble each other A is near -1 below the
// diagonal, the powers reach 3e3 and cancel to O(1), which in float32 left y
// and the gradients 1e-5 to 1e-4 off.
__device__ __forceinline__ d4 inverse(d4 a, d4 at, int l) {
    d4 one;
#pragma unroll
    for (int e = 0; e < 4; ++e) one[e] = 4 * e + l / 16 == l % 16 ? 1. : 0.;
    const d4 a2 = mm64(at, a), a2t = mm64(a, at);
    const d4 q1 = one + a + mm64(at, a2, a2), q1t = one + at + mm64(a2, at, a2t);
    const d4 a4 = mm64(a2t, a2), a4t = mm64(a2, a2t);
    const d4 q2 = mm64(q1t, a4, q1), q2t = mm64(a4, q1t, q1t);
    return mm64(q2t, mm64(a4t, a4), q2);
}

// One workgroup per chunk and head: bound by the inverse's products on one
// wave, ten in float64 of which four follow each other, hidden by the other
// chunks' workgroups on the CU (22 and 28 KB of LDS each at N = 64).  96 heads
// of 64, 32 chunks: forward 40, backward 50 us (all float32: 31 and 43).
template <int N, typename VT, bool BWD>
__global__ void __launch_bounds__(256, 2) f32_prep_kernel(Args A) {
    using W = Ws<N, BWD>;
    constexpr int NB = W::NB;
    __shared__ Rows<N> fA, fR, fB, fK;
    __shared__ Mat64 sA, sM;
    __shared__ Mat sMak;
    __shared__ f4 sW[BWD ? NB : 1][64];
    const int64_t bh = blockIdx.x, ch = blockIdx.y;
    const int wave = threadIdx.x / 64, l = threadIdx.x % 64;
    const int q = l / 16;
    const int64_t t0 = (A.c0 + ch) * 16;
    const int64_t hoff = A.lay.head(bh, N);
    float* ws = A.ws + (ch * A.BH + bh) * W::SIZE;
    const bool valid = t0 + l % 16 < A.T;
    const int64_t toff = (t0 + l % 16) * A.lay.ts + hoff;

    constexpr int PER = (NB + 3) / 4;  // column blocks of a wave
    f4 Bh[PER], Kh[PER];
    bool bad = false;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int c = wave + 4 * i, col = 16 * c + 4 * q;
        if (c >= NB) break;
        Factors F;
        factors<VT, !BWD>(F, A, toff + col, valid);
        bad |= F.bad;
        if (valid) {
            bad |= out_of_range(
                load4(static_cast<const VT*>(A.v) + toff + col));
            if (BWD && A.dy)
                bad |= out_of_range(
                    load4(static_cast<const VT*>(A.dy) + toff + col));
        }
        fA.put_t(c, l, F.A);
        fR.put_t(c, l, F.R);
        fB.put_t(c, l, F.B);
        fK.put_t(c, l, F.K);
        if constexpr (!BWD) {
            Bh[i] = F.Bh;
            Kh[i] = F.Kh;
        }
        if (l % 16 == 15) store4(ws + W::PL + col, F.P);
    }
    // (a barrier: the factors are complete)
    bad = __syncthreads_or(bad);
    if (threadIdx.x == 0) A.flags[ch * A.BH + bh] = bad;
    if (bad) return;

    // The four matrices, a wave each; H tiles of Aab, Aak, Arb^T, and Ark^T
    // (forward) or Ark (backward).  In float64 from the rounded factors, and
    // rounded once where they are stored: in float32 their sums' error,
    // times what the inverse and the serial step make of it, was most of y's.
    d4 m;
    if (wave == 0)
        m = keep_lower(outer64<N>(fA, fB, l), l, false);
    else if (wave == 1)
        m = keep_lower(outer64<N>(fA, fK, l), l, false);
    else if (wave == 2)
        m = keep_upper(outer64<N>(fB, fR, l), l, true);
    else if (!BWD)
        m = keep_upper(outer64<N>(fK, fR, l), l, true);
    else
        m = keep_lower(outer64<N>(fR, fK, l), l, true);
    if (wave == 0) {
        sA.put(l, m);
        __builtin_amdgcn_wave_barrier();
        sM.put(l, inverse(m, sA.ht(l), l));
    } else {
        // meanwhile the operands that need no inverse
        for (int c = wave - 1; c < NB; c += 3) {
            if (!BWD) {
                store4(ws + W::M1 + c * 256 + 4 * l, fR.t(c, l));
            } else {
                store4(ws + W::M1 + c * 256 + 4 * l, fA.jp(c, l));
                store4(ws + W::M2 + c * 256 + 4 * l, fR.jp(c, l));
            }
        }
        if (!BWD && wave >= 2) store_tile(ws + W::S + (wave - 1) * 256, l, m);
        if (BWD && wave == 3) store_tile(ws + W::S + 256, l, m);
        if (BWD && wave == 1) store_tile(ws + W::S + 512, l, m);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int c = wave + 4 * i;
        if (c >= NB) break;
        if constexpr (!BWD) {
            // B^ and K^ take the place of B~ and K~: a wave's own columns, to
            // lanes of the other form (two matrices more in LDS halved the
            // workgroups of a CU at N = 128, 66 -> 106 us)
            fB.put_t(c, l, Bh[i]);
            fK.put_t(c, l, Kh[i]);
            __builtin_amdgcn_wave_barrier();
            store4(ws + W::M2 + c * 256 + 4 * l, fB.jp(c, l));
            store4(ws + W::M3 + c * 256 + 4 * l, fK.jp(c, l));
        }
        const f4 wt =
            __builtin_convertvector(mm64(fA.jp(c, l), sM.dt(l)), f4);
        if (!BWD) {
            store4(ws + W::M0 + c * 256 + 4 * l, wt);
        } else {
            sW[c][l] = wt;
            store4(ws + W::M0 + c * 256 + 4 * l,
                   __builtin_convertvector(mm64(fB.jp(c, l), sM.d(l)), f4));
        }
    }
    if (wave == 1) {
        const d4 mak = mm64(m, sM.ht(l));  // T form of Minv Aak
        if (!BWD) {
            store_tile(ws + W::S, l, mak);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                sMak.x[4 * e + q][l % 16] = float(mak[e]);
        }
    }
    if (BWD && wave == 2)
        store_tile(ws + W::S, l, mm64(m, sM.h(l)));  // T form of G
    if constexpr (BWD) {
        // X = W S0^T + Mak V, 16 state rows a wave
        __syncthreads();
        const f4 mak = sMak.d(l);
        for (int ib = wave; ib < NB; ib += 4) {
            const int row = 16 * ib + l % 16;
            const float* s0 =
                A.ckpt_in + ((A.c0 + ch) * A.BH + bh) * N * N + row * N;
            f4 s[NB], v;
#pragma unroll
            for (int c = 0; c < NB; ++c) s[c] = load4(s0 + 16 * c + 4 * q);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t t = t0 + 4 * q + e;
                v[e] = t < A.T ? load_f(static_cast<const VT*>(A.v) +
                                        t * A.lay.ts + hoff + row)
                               : 0.f;
            }
            const f4 x =
                mm(mak, v) +
                tree<0, NB>([&](int c) { return mm(sW[c][l], s[c]); });
#pragma unroll
            for (int e = 0; e < 4; ++e)
                ws[W::X + (4 * q + e) * N + row] = x[e];
        }
    }
}

// One wave per 16 state rows walks the segment's chunks with its rows of S
// (or D) in registers; a workgroup's waves are row blocks of one head and
// share each chunk's operands.  Bound by a wave's own chain of products: 19
// of 16x16x16 a chunk forward at N = 64, 13 backward, 128 cycles each, and the
// update's eight (the state's, or its cotangent's) about 256: they are summed
// in float64, onto the decayed state, and rounded once.  In float32 those sums
// were the larger part of S_T's and dS0's error (0.7 and 0.9e-7 against 0.4
// and 0.5), and under the slowest decay they added up to twice the sequential
// kernels'.  At 32 chunks of 96 heads a chain takes 98 and 72 us for 77 and 59.
template <int N>
constexpr int kChainWaves = N / 16 < 4 ? N / 16 : 4;

// The operands of the chunks in LDS, three buffers: during a chunk every
// thread's share of the next but one is in flight from memory into
// registers, then written to the buffer of the chunk before, which every
// wave is past (one barrier a chunk).
template <int N, bool BWD>
struct Feed {
    using W = Ws<N, BWD>;
    static constexpr int LEN = W::PL + N;  // floats
    static constexpr int TH = 64 * kChainWaves<N>;
    static constexpr int PER = (LEN / 4 + TH - 1) / TH;
    f4 g[PER];
    __device__ __forceinline__ void load(const float* from) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int at = i * TH + threadIdx.x;
            g[i] = load4(from + 4 * (at < LEN / 4 ? at : 0));
        }
    }
    __device__ __forceinline__ void put(float* to) const {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int at = i * TH + threadIdx.x;
            if (at < LEN / 4) store4(to + 4 * at, g[i]);
        }
    }
};

// A barrier for LDS only: __syncthreads would also wait for the chunk's
// global stores to complete, a memory round trip per chunk.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ float widen(float x) { return x; }
__device__ __forceinline__ float widen(bf16_t x) { return bf16_to_f32(x); }

// A buffer of `bytes` bytes at `base`: loads past its end give zeros, stores
// past it are dropped.  The chain kernels' loops hold no branch around a
// memory operation (at a join the compiler waits for every one in flight).
using Rsrc = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ Rsrc rsrc(const void* base, int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0,
                                             int(bytes), 0x00020000);
}
// The 16 tokens from `base`, `left` of them present, none without a base.
template <typename VT>
__device__ __forceinline__ Rsrc token_rsrc(const VT* base, int64_t ts,
                                           int64_t left) {
    const int64_t n = left < 16 ? left : 16;
    return rsrc(base, base && n > 0 ? n * ts * int64_t(sizeof(VT)) : 0);
}

// Tokens from the chunk before chunk ch of a segment, `left` from ch on.  The
// segment's first chunk has none before it and stays where it is: counted on
// from there, a segment of one partial chunk would read past the tensor.
__host__ __device__ constexpr int64_t tokens_from(int64_t left, int64_t ch) {
    return ch > 0 ? left + 16 : left;
}
static_assert(tokens_from(1, 0) == 1 && tokens_from(16, 0) == 16 &&
                  tokens_from(1, 1) == 17,
              "a segment of one chunk reads its own tokens only");

__device__ __forceinline__ void fetch(float& x, Rsrc r, int off) {
    x = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off * 4, 0, 0));
}
__device__ __forceinline__ void fetch(bf16_t& x, Rsrc r, int off) {
    x = __builtin_amdgcn_raw_buffer_load_b16(r, off * 2, 0, 0);
}
__device__ __forceinline__ void put_elem(float, Rsrc r, int off, float x) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x), r, off * 4, 0, 0);
}
__device__ __forceinline__ void put_elem(bf16_t, Rsrc r, int off, float x) {
    __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16(x), r, off * 2, 0, 0);
}

// A lane's 16x16 block of a vector (tokens 4q + e of a chunk, one state row's
// entry, at element off[e] of the chunk), loaded as it is and widened only
// when used: a conversion next to the load would wait for it.
template <typename VT>
struct Block {
    VT x[4];
    __device__ __forceinline__ void load(Rsrc r, const int (&off)[4]) {
#pragma unroll
        for (int e = 0; e < 4; ++e) fetch(x[e], r, off[e]);
    }
    __device__ __forceinline__ f4 value() const {
        return f4{widen(x[0]), widen(x[1]), widen(x[2]), widen(x[3])};
    }
};

template <int N, typename VT>
__global__ void __launch_bounds__(64 * kChainWaves<N>, N <= 64 ? 2 : 1)
f32_fwd_chain_kernel(Args A) {
    using W = Ws<N, false>;
    constexpr int NB = W::NB, PARTS = NB / kChainWaves<N>;
    using Fd = Feed<N, false>;
    __shared__ float ops[3][Fd::LEN];
    const int64_t bh = blockIdx.x / PARTS;
    const int ib = int(blockIdx.x % PARTS) * kChainWaves<N> + threadIdx.x / 64;
    const int l = threadIdx.x % 64, q = l / 16, row = 16 * ib + l % 16;
    if (head_marked(A, bh)) return;
    const int64_t srow = bh * N * N + int64_t(row) * N + 4 * q;
    const float* ws = A.ws + bh * W::SIZE;
    const int64_t step = A.BH * W::SIZE;
    const int64_t last = A.nch - 1;
    f4 s[NB];
#pragma unroll
    for (int c = 0; c < NB; ++c) s[c] = load4(A.state_in + srow + 16 * c);
    Fd feed;
    feed.load(ws);
    feed.put(ops[0]);
    feed.load(ws + (last < 1 ? last : 1) * step);
    feed.put(ops[1]);
    // the chunk at hand in v and in y, and this lane's elements of it
    const int64_t ts = A.lay.ts, first = A.c0 * 16 * ts + A.lay.head(bh, N);
    const VT* vp = static_cast<const VT*>(A.v) + first;
    VT* yp = static_cast<VT*>(A.y) + first;
    int64_t left = A.T - A.c0 * 16;
    int off[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) off[e] = int((4 * q + e) * ts) + row;
    Block<VT> vb;
    vb.load(token_rsrc(vp, ts, left), off);
    f4 v = vb.value();
    int buf = 0;
    // Products go in groups of up to four column blocks; the first group of
    // W (and Mak, last) is read in the chunk before.
    constexpr int G = NB == 8 ? 2 : NB;
    f4 w[G + 1];
    auto load_x = [&](int from) __attribute__((always_inline)) {
        w[G] = load4(ops[from] + W::S + 4 * l);
#pragma unroll
        for (int c = 0; c < G; ++c)
            w[c] = load4(ops[from] + W::M0 + c * 256 + 4 * l);
    };
    // checkpoints: the next one's place, and the chunks until it
    using u4 = unsigned __attribute__((ext_vector_type(4)));
    float* ck = A.ckpt + ((A.c0 + A.ck_every - 1) / A.ck_every * A.BH + bh) *
                             N * N;
    int until = int((A.ck_every - A.c0 % A.ck_every) % A.ck_every);
    lds_barrier();
    load_x(0);
    for (int64_t ch = 0; ch < A.nch; ++ch) {
        lds_barrier();
        feed.load(ws + (ch + 2 < last ? ch + 2 : last) * step);
        vb.load(token_rsrc(vp + 16 * ts, ts, left - 16), off);
        __builtin_amdgcn_sched_barrier(0);
        {
            const bool due = A.ckpt && until == 0;
            const Rsrc to = rsrc(ck, due ? N * N * 4 : 0);
#pragma unroll
            for (int c = 0; c < NB; ++c)
                __builtin_amdgcn_raw_buffer_store_b128(
                    __builtin_bit_cast(u4, s[c]), to,
                    (row * N + 16 * c + 4 * q) * 4, 0, 0);
            ck += due ? A.BH * N * N : 0;
            until = until == 0 ? int(A.ck_every) - 1 : until - 1;
        }
        // Each phase's operands are read from LDS during the phase before.
        const float* o = ops[buf];
        auto tile = [&](int at) { return load4(o + at + 4 * l); };
        const f4 arb = tile(W::S + 256);
        auto rows = [&](int at, int c0, const f4 (&first)[G + 1])
                        __attribute__((always_inline)) {
            // the group's products with the state, and with v in the first
            f4 sum;
            if (c0 == 0) {
                f4 sv[G + 1], p[G + 1];
#pragma unroll
                for (int c = 0; c < G; ++c) sv[c] = s[c];
                sv[G] = v;
                products(first, sv, p);
                sum = p[G] + tree<0, G>([&](int c) { return p[c]; });
            } else {
                f4 m[G], sv[G], p[G];
#pragma unroll
                for (int c = 0; c < G; ++c) {
                    m[c] = tile(at + (c0 + c) * 256);
                    sv[c] = s[c0 + c];
                }
                products(m, sv, p);
                sum = tree<0, G>([&](int c) { return p[c]; });
            }
            return sum;
        };
        f4 r[G + 1];
        r[G] = tile(W::S + 512);
#pragma unroll
        for (int c = 0; c < G; ++c) r[c] = tile(W::M1 + c * 256);
        f4 x = rows(W::M0, 0, w);
#pragma unroll
        for (int c0 = G; c0 < NB; c0 += G) x += rows(W::M0, c0, w);
        f4 y = rows(W::M1, 0, r);
#pragma unroll
        for (int c0 = G; c0 < NB; c0 += G) y += rows(W::M1, c0, r);
        load_x(buf == 2 ? 0 : buf + 1);
        const f4 yx = mm(arb, x);
        // the state
#pragma unroll
        for (int c0 = 0; c0 < NB; c0 += G) {
            d4 acc[G];
            f4 bb[G], kk[G];
#pragma unroll
            for (int c = 0; c < G; ++c) {
                bb[c] = tile(W::M2 + (c0 + c) * 256);
                kk[c] = tile(W::M3 + (c0 + c) * 256);
                acc[c] = __builtin_convertvector(s[c0 + c], d4) *
                         __builtin_convertvector(
                             load4(o + W::PL + 16 * (c0 + c) + 4 * q), d4);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int c = 0; c < G; ++c)
                    acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                        kk[c][e], v[e], acc[c], 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int c = 0; c < G; ++c)
                    acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                        bb[c][e], x[e], acc[c], 0, 0, 0);
#pragma unroll
            for (int c = 0; c < G; ++c)
                s[c0 + c] = __builtin_convertvector(acc[c], f4);
        }
        y += yx;
        // (the loads' values are taken before the stores are issued: memory
        // operations are waited for in order)
        feed.put(ops[buf == 0 ? 2 : buf - 1]);
        v = vb.value();
        asm volatile("" : "+v"(v));
        __builtin_amdgcn_sched_barrier(0);
        const Rsrc yr = token_rsrc(yp, ts, left);
#pragma unroll
        for (int e = 0; e < 4; ++e) put_elem(VT(0), yr, off[e], y[e]);
        buf = buf == 2 ? 0 : buf + 1;
        vp += 16 * ts;
        yp += 16 * ts;
        left -= 16;
    }
#pragma unroll
    for (int c = 0; c < NB; ++c) store4(A.state_out + srow + 16 * c, s[c]);
    if (A.ckpt && A.ck_last >= 0) {
        float* to = A.ckpt + A.ck_last * A.BH * N * N + srow;
#pragma unroll
        for (int c = 0; c < NB; ++c) store4(to + 16 * c, s[c]);
    }
}

template <int N, typename VT>
__global__ void __launch_bounds__(64 * kChainWaves<N>, N <= 64 ? 2 : 1)
f32_bwd_chain_kernel(Args A) {
    using W = Ws<N, true>;
    constexpr int NB = W::NB, PARTS = NB / kChainWaves<N>;
    using Fd = Feed<N, true>;
    __shared__ float ops[3][Fd::LEN];
    const int64_t bh = blockIdx.x / PARTS;
    const int ib = int(blockIdx.x % PARTS) * kChainWaves<N> + threadIdx.x / 64;
    const int l = threadIdx.x % 64, q = l / 16, row = 16 * ib + l % 16;
    if (head_marked(A, bh)) return;
    const int64_t srow = bh * N * N + int64_t(row) * N + 4 * q;
    float* ws = A.ws + bh * W::SIZE;
    const int64_t step = A.BH * W::SIZE;
    f4 d[NB];
#pragma unroll
    for (int c = 0; c < NB; ++c)
        d[c] = A.state_in ? load4(A.state_in + srow + 16 * c) : kZero;
    Fd feed;
    feed.load(ws + (A.nch - 1) * step);
    feed.put(ops[0]);
    feed.load(ws + (A.nch > 1 ? A.nch - 2 : 0) * step);
    feed.put(ops[1]);
    const int64_t ts = A.lay.ts, end = A.c0 + A.nch - 1;
    const VT* yp = A.dy ? static_cast<const VT*>(A.dy) + end * 16 * ts +
                              A.lay.head(bh, N)
                        : nullptr;
    int64_t left = A.T - end * 16;
    int off[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) off[e] = int((4 * q + e) * ts) + row;
    Block<VT> yb;
    yb.load(token_rsrc(yp, ts, left), off);
    f4 dy = yb.value();
    int buf = 0;
    for (int64_t ch = A.nch - 1; ch >= 0; --ch) {
        lds_barrier();
        feed.load(ws + (ch > 2 ? ch - 2 : 0) * step);
        yp -= A.dy && ch > 0 ? 16 * ts : 0;
        left = tokens_from(left, ch);
        yb.load(token_rsrc(yp, ts, left), off);
        __builtin_amdgcn_sched_barrier(0);
        const float* o = ops[buf];
        auto tile = [&](int at) { return load4(o + at + 4 * l); };
        float* to = ws + ch * step;
        constexpr int G = NB == 8 ? 2 : NB;
        f4 u;
#pragma unroll
        for (int c0 = 0; c0 < NB; c0 += G) {
            f4 w[G + 1], dv[G + 1], p[G + 1];
            w[G] = tile(W::S);
            dv[G] = dy;
#pragma unroll
            for (int c = 0; c < G; ++c) {
                w[c] = tile(W::M0 + (c0 + c) * 256);
                d[c0 + c] *= load4(o + W::PL + 16 * (c0 + c) + 4 * q);
                dv[c] = d[c0 + c];
                store4(to + W::DH + row * N + 16 * (c0 + c) + 4 * q, dv[c]);
            }
            products(w, dv, p);
            const f4 sum = tree<0, G>([&](int c) { return p[c]; });
            u = c0 == 0 ? p[G] + sum : u + sum;
        }
#pragma unroll
        for (int c0 = 0; c0 < NB; c0 += G) {
            d4 acc[G];
            f4 aa[G], rr[G];
#pragma unroll
            for (int c = 0; c < G; ++c) {
                aa[c] = tile(W::M1 + (c0 + c) * 256);
                rr[c] = tile(W::M2 + (c0 + c) * 256);
                acc[c] = __builtin_convertvector(d[c0 + c], d4);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int c = 0; c < G; ++c)
                    acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                        rr[c][e], dy[e], acc[c], 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int c = 0; c < G; ++c)
                    acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                        aa[c][e], u[e], acc[c], 0, 0, 0);
#pragma unroll
            for (int c = 0; c < G; ++c)
                d[c0 + c] = __builtin_convertvector(acc[c], f4);
        }
        feed.put(ops[buf == 0 ? 2 : buf - 1]);
        dy = yb.value();
        asm volatile("" : "+v"(dy));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 4; ++e) to[W::U + (4 * q + e) * N + row] = u[e];
        buf = buf == 2 ? 0 : buf + 1;
    }
#pragma unroll
    for (int c = 0; c < NB; ++c) store4(A.state_out + srow + 16 * c, d[c]);
}

// The chunk's gradients from S0, D^, X and dU.  A wave owns one block of 16
// columns (dr, dw, dk, da, db) and of 16 state rows (dv).  Bound by its loads'
// round trips and the products of the waves that share a SIMD, so by the waves
// in flight: at most 128 registers a lane, for four waves a SIMD.  N = 128,
// two workgroups of eight waves a CU (73 KB of LDS each): 235 -> 115 us a
// segment (14 chunks of 128 heads, bf16) against one of four waves with two
// blocks each; N = 64, four workgroups of four waves a CU (40 KB each): 128 ->
// 122 us a segment (fp32, B8 T4096 H32) against three.
template <int N>
constexpr int kGradWaves = N <= 64 ? 4 : 8;
template <int N, typename VT>
__global__ void __launch_bounds__(64 * kGradWaves<N>, 4)
f32_grads_kernel(Args A) {
    using W = Ws<N, true>;
    constexpr int NB = W::NB;
    __shared__ Rows<N> fA, fR, fB, fK, tX, tU, tV, tY;
    __shared__ Mat mat[4];
    __shared__ float zs[N];
    const int64_t bh = blockIdx.x, ch = blockIdx.y;
    const int wave = threadIdx.x / 64, l = threadIdx.x % 64, q = l / 16;
    const int64_t t0 = (A.c0 + ch) * 16;
    const int64_t hoff = A.lay.head(bh, N);
    const float* ws = A.ws + (ch * A.BH + bh) * W::SIZE;
    const float* s0 = A.ckpt_in + ((A.c0 + ch) * A.BH + bh) * N * N;
    const bool valid = t0 + l % 16 < A.T;
    const int64_t toff = (t0 + l % 16) * A.lay.ts + hoff;

    // The state tiles of the wave's column block: in flight from the start,
    // or (N = 128) once the factors' registers are free, four blocks ahead.
    // (Buffer loads: the rows' offsets are scalars.)
    const Rsrc rs = rsrc(s0, N * N * 4), rd = rsrc(ws + W::DH, N * N * 4);
    const int at0 = (4 * q * N + 16 * (wave < NB ? wave : 0) + l % 16) * 4;
    f4 sc[NB], dc[NB];
    auto load_state = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = (16 * b + e) * N * 4;
            sc[b][e] = __uint_as_float(
                __builtin_amdgcn_raw_buffer_load_b32(rs, at0, row, 0));
            dc[b][e] = __uint_as_float(
                __builtin_amdgcn_raw_buffer_load_b32(rd, at0, row, 0));
        }
    };
    auto load_first = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < (NB < 4 ? NB : 4); ++b) load_state(b);
    };
    if constexpr (NB <= 4) load_first();
    // (from N = 64 on a phase's LDS reads stay behind the phase before)
    auto phase = []() __attribute__((always_inline)) {
        if constexpr (NB >= 4) __builtin_amdgcn_sched_barrier(0);
    };
    const int c = wave;
    f4 fP, fPp, finv, few;
    if (c < NB) {
        const int col = 16 * c + 4 * q;
        Factors F;
        factors<VT>(F, A, toff + col, valid);
        fP = F.P;
        fPp = F.Pp;
        finv = F.inv;
        few = F.ew;
        fA.put_t(c, l, F.A);
        fR.put_t(c, l, F.R);
        fB.put_t(c, l, F.B);
        fK.put_t(c, l, F.K);
        tX.put_t(c, l, load4(ws + W::X + (l % 16) * N + col));
        tU.put_t(c, l, load4(ws + W::U + (l % 16) * N + col));
        tV.put_t(c, l, valid ? load4(static_cast<const VT*>(A.v) + toff + col)
                             : kZero);
        tY.put_t(c, l,
                 valid && A.dy
                     ? load4(static_cast<const VT*>(A.dy) + toff + col)
                     : kZero);
    }
    // (a marked head's values are not used: the loads above stay in bounds)
    if (head_marked(A, bh)) return;
    phase();
    if constexpr (NB > 4) load_first();
    __syncthreads();
    phase();
    // dArb, dArk, dAab, dAak, a wave each
    if (wave < 4)
        mat[wave].put(l, keep_lower(outer<N>(wave < 2 ? tY : tU,
                                             wave & 1 ? tV : tX, l),
                                    l, wave < 2));
    __syncthreads();

    auto put = [&](void* to, const void* add, int64_t off, f4 x) {
        if (!valid) return;
        if (add) x += load4(static_cast<const VT*>(add) + off);
        store4(static_cast<VT*>(to) + off, x);
    };
    if (c < NB) {
        // products over the state rows, all T forms: dY S0, dU S0, X D^, V D^
        f4 sr = kZero, sa = kZero, xb = kZero, xk = kZero;
        float z = 0.f;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const f4 s = sc[b], dh = dc[b];
            z += (s[0] * dh[0] + s[1] * dh[1]) + (s[2] * dh[2] + s[3] * dh[3]);
            sr += mm(s, tY.t(b, l));
            sa += mm(s, tU.t(b, l));
            xb += mm(dh, tX.t(b, l));
            xk += mm(dh, tV.t(b, l));
            if (b + 4 < NB) load_state(b + 4);
            // (the sums are taken here: left to the end, they held every
            // block's products in registers)
            if constexpr (NB >= 4)
                asm volatile("" : "+v"(sr), "+v"(sa), "+v"(xb), "+v"(xk));
            phase();
        }
        z = add_swap<32>(add_swap<16>(z));  // of column 16c + l % 16
        if (q == 0) zs[16 * c + l % 16] = z;
        __builtin_amdgcn_wave_barrier();
        // The chunk's own pairs (t', s).  In the decay gradient a pair on one
        // side of token t cancels between its two tokens: in float64, from
        // the same operands, it does so exactly (in float32 dw was twice as
        // far from float64 as the rest).
        const f4 jb = fB.jp(c, l), jk = fK.jp(c, l), jr = fR.jp(c, l),
                 ja = fA.jp(c, l);
        const d4 pr = mm64(jk, mat[1].dt(l), mm64(jb, mat[0].dt(l)));
        phase();
        const d4 pa = mm64(jk, mat[3].dt(l), mm64(jb, mat[2].dt(l)));
        phase();
        const d4 pb = mm64(ja, mat[2].d(l), mm64(jr, mat[0].d(l)));
        phase();
        const d4 pk = mm64(ja, mat[3].d(l), mm64(jr, mat[1].d(l)));
        phase();
        const f4 tA = fA.t(c, l), tR = fR.t(c, l), tB = fB.t(c, l),
                 tK = fK.t(c, l);
        const f4 p = tB * xb + tK * xk;
        const f4 zt = *reinterpret_cast<const f4*>(&zs[16 * c + 4 * q]);
        f4 dR, dA, dB, dK, dw;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const double pairs = suffix_add(
                tR[e] * pr[e] - tB[e] * pb[e] - tK[e] * pk[e] +
                from_right<1>(tA[e] * pa[e], 0.0));
            const float dlogd =
                float(pairs) +
                suffix_add(tR[e] * sr[e] +
                           from_right<1>(tA[e] * sa[e], 0.f)) +
                prefix_add(from_left<1>(p[e], 0.f)) + zt[e];
            dw[e] = -few[e] * dlogd;
            // (one rounding where float32 had three)
            dR[e] = float((sr[e] + pr[e]) * fP[e]);
            dA[e] = float((sa[e] + pa[e]) * fPp[e]);
            dB[e] = float((xb[e] + pb[e]) * finv[e]);
            dK[e] = float((xk[e] + pk[e]) * finv[e]);
        }
        const int64_t off = toff + 16 * c + 4 * q;
        put(A.dr, A.add_dr, off, dR);
        put(A.dw, nullptr, off, dw);
        put(A.dk, A.add_dk, off, dK);
        put(A.da, nullptr, off, dA);
        put(A.db, nullptr, off, dB);
    }
    phase();
    const f4 ark = load4(ws + W::S + 256 + 4 * l);
    const f4 aak = load4(ws + W::S + 512 + 4 * l);
    if (c < NB) {
        const int ib = c;
        const float* dh = ws + W::DH + (16 * ib + l % 16) * N + 4 * q;
        const f4 x = (mm(tY.j(ib, l), ark) + mm(tU.j(ib, l), aak)) +
                     tree<0, NB>([&](int c) {
                         return mm(load4(dh + 16 * c), fK.t(c, l));
                     });
        put(A.dv, A.add_dv, toff + 16 * ib + 4 * q, x);
    }
}

// Workspace of one time segment: the chunks whose operands are held at once.
constexpr int64_t kWsBytes = int64_t(192) << 20;

int64_t segment_chunks(int64_t nch, int64_t BH, int64_t floats,
                       int64_t multiple) {
    int64_t n = kWsBytes / (4 * BH * (floats + 1));
    n -= n % multiple;
    if (n < multiple) n = multiple;
    if (n > 32768) n = 32768 - 32768 % multiple;
    return n < nch ? n : nch;
}

const void* at(const void* p, int64_t elems, bool bf16) {
    return p ? static_cast<const char*>(p) + elems * (bf16 ? 2 : 4) : nullptr;
}
void* at(void* p, int64_t elems, bool bf16) {
    return static_cast<char*>(p) + elems * (bf16 ? 2 : 4);
}

template <int N, typename VT>
hipError_t forward(const SeqFwdArgs& p, hipStream_t stream) {
    constexpr int FL = Ws<N, false>::SIZE;
    const int64_t BH = p.B * p.H, nch = (p.T + 15) / 16;
    const int64_t every = p.ckpt ? p.ci / 16 : 1;
    const int64_t seg = segment_chunks(nch, BH, FL, every);
    float* ws = nullptr;
    hipError_t e = pool_alloc(&ws, size_t(4 * seg * BH * (FL + 1)), stream);
    if (e != hipSuccess) return e;
    Args A{};
    A.T = p.T;
    A.BH = BH;
    A.lay = p.lay;
    A.r = p.r;
    A.w = p.w;
    A.k = p.k;
    A.v = p.v;
    A.a = p.a;
    A.b = p.b;
    A.y = p.y;
    A.state_out = p.s_t;
    A.ckpt = static_cast<float*>(p.ckpt);
    A.ck_every = every;
    A.ws = ws;
    A.flags = reinterpret_cast<int*>(ws + seg * BH * FL);
    for (int64_t c0 = 0; c0 < nch && e == hipSuccess; c0 += seg) {
        A.c0 = c0;
        A.nch = nch - c0 < seg ? nch - c0 : seg;
        A.state_in = c0 == 0 ? p.s0 : p.s_t;
        A.ck_last = c0 + A.nch == nch ? (p.T + p.ci - 1) / (p.ci ? p.ci : 1)
                                      : -1;
        hipLaunchKernelGGL((f32_prep_kernel<N, VT, false>),
                           dim3(unsigned(BH), unsigned(A.nch)), dim3(256), 0,
                           stream, A);
        hipLaunchKernelGGL(
            (f32_fwd_chain_kernel<N, VT>),
            dim3(unsigned(BH * (N / 16 / kChainWaves<N>))),
            dim3(64 * kChainWaves<N>), 0, stream, A);
        e = hipGetLastError();
        if (e != hipSuccess) break;
        // the marked heads of this segment
        SeqFwdArgs s = p;
        const int64_t t0 = c0 * 16, off = t0 * p.lay.ts;
        s.T = p.T - t0 < A.nch * 16 ? p.T - t0 : A.nch * 16;
        s.r = at(p.r, off, p.bf16);
        s.w = at(p.w, off, p.bf16);
        s.k = at(p.k, off, p.bf16);
        s.v = at(p.v, off, p.bf16);
        s.a = at(p.a, off, p.bf16);
        s.b = at(p.b, off, p.bf16);
        s.y = at(p.y, off, p.bf16);
        s.s0 = A.state_in;
        if (p.ckpt)
            s.ckpt = A.ckpt + c0 / every * BH * N * N;
        s.flags = A.flags;
        s.nflag = A.nch;
        e = launch_seq_forward(s, stream);
    }
    const hipError_t f = hipFreeAsync(ws, stream);
    return e != hipSuccess ? e : f;
}

template <int N, typename VT>
hipError_t backward(const SeqBwdArgs& p, hipStream_t stream) {
    constexpr int FL = Ws<N, true>::SIZE;
    // (a marked head's sequential pass keeps its column sums' shares in the
    // segment's workspace, which the gradients have been taken from by then)
    static_assert(N < 128 || FL >= 2 * 16 * 5 * N, "room for the shares");
    const int64_t BH = p.B * p.H, nch = (p.T + 15) / 16;
    const int64_t seg = segment_chunks(nch, BH, FL, 1);
    float* ws = nullptr;
    hipError_t e = pool_alloc(&ws, size_t(4 * seg * BH * (FL + 1)), stream);
    if (e != hipSuccess) return e;
    Args A{};
    A.T = p.T;
    A.BH = BH;
    A.lay = p.lay;
    A.r = p.r;
    A.w = p.w;
    A.k = p.k;
    A.v = p.v;
    A.a = p.a;
    A.b = p.b;
    A.dy = p.dy;
    A.ckpt_in = static_cast<const float*>(p.ckpt);
    A.state_out = p.ds0;
    A.dr = p.dr;
    A.dw = p.dw;
    A.dk = p.dk;
    A.dv = p.dv;
    A.da = p.da;
    A.db = p.db;
    A.add_dr = p.add_dr;
    A.add_dk = p.add_dk;
    A.add_dv = p.add_dv;
    A.ws = ws;
    A.flags = reinterpret_cast<int*>(ws + seg * BH * FL);
    for (int64_t c1 = nch; c1 > 0 && e == hipSuccess;) {
        A.c0 = c1 > seg ? c1 - seg : 0;
        A.nch = c1 - A.c0;
        A.state_in = c1 == nch ? p.ds_t : p.ds0;
        const dim3 grid{unsigned(BH), unsigned(A.nch)};
        hipLaunchKernelGGL((f32_prep_kernel<N, VT, true>), grid, dim3(256), 0,
                           stream, A);
        hipLaunchKernelGGL(
            (f32_bwd_chain_kernel<N, VT>),
            dim3(unsigned(BH * (N / 16 / kChainWaves<N>))),
            dim3(64 * kChainWaves<N>), 0, stream, A);
        hipLaunchKernelGGL((f32_grads_kernel<N, VT>), grid,
                           dim3(64 * kGradWaves<N>), 0, stream, A);
        e = hipGetLastError();
        if (e != hipSuccess) break;
        SeqBwdArgs s = p;
        const int64_t t0 = A.c0 * 16, off = t0 * p.lay.ts;
        s.T = p.T - t0 < A.nch * 16 ? p.T - t0 : A.nch * 16;
        s.r = at(p.r, off, p.bf16);
        s.w = at(p.w, off, p.bf16);
        s.k = at(p.k, off, p.bf16);
        s.v = at(p.v, off, p.bf16);
        s.a = at(p.a, off, p.bf16);
        s.b = at(p.b, off, p.bf16);
        s.dy = at(p.dy, off, p.bf16);
        s.dr = at(p.dr, off, p.bf16);
        s.dw = at(p.dw, off, p.bf16);
        s.dk = at(p.dk, off, p.bf16);
        s.dv = at(p.dv, off, p.bf16);
        s.da = at(p.da, off, p.bf16);
        s.db = at(p.db, off, p.bf16);
        s.add_dr = at(p.add_dr, off, p.bf16);
        s.add_dk = at(p.add_dk, off, p.bf16);
        s.add_dv = at(p.add_dv, off, p.bf16);
        s.ds_t = A.state_in;
        s.ckpt = A.ckpt_in + A.c0 * BH * N * N;
        s.flags = A.flags;
        s.nflag = A.nch;
        s.part = ws;
        e = launch_seq_backward(s, stream);
        c1 = A.c0;
    }
    const hipError_t f = hipFreeAsync(ws, stream);
    return e != hipSuccess ? e : f;
}

}  // namespace

hipError_t launch_f32_forward(const SeqFwdArgs& p, hipStream_t stream) {
    switch (p.N) {
        case 16: return p.bf16 ? forward<16, bf16_t>(p, stream)
                               : forward<16, float>(p, stream);
        case 32: return p.bf16 ? forward<32, bf16_t>(p, stream)
                               : forward<32, float>(p, stream);
        case 64: return p.bf16 ? hipErrorInvalidValue
                               : forward<64, float>(p, stream);
        case 128: return p.bf16 ? forward<128, bf16_t>(p, stream)
                                : forward<128, float>(p, stream);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_f32_backward(const SeqBwdArgs& p, hipStream_t stream) {
    switch (p.N) {
        case 16: return p.bf16 ? backward<16, bf16_t>(p, stream)
                               : backward<16, float>(p, stream);
        case 32: return p.bf16 ? backward<32, bf16_t>(p, stream)
                               : backward<32, float>(p, stream);
        case 64: return p.bf16 ? hipErrorInvalidValue
                               : backward<64, float>(p, stream);
        case 128: return p.bf16 ? backward<128, bf16_t>(p, stream)
                                : backward<128, float>(p, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace rwkv7m
