// Learned SGS closure: pointwise features, stress and training loss of the
// tensor-basis MLP (no counterpart in the reference; its baseline is the
// eddy-viscosity family of src/incompressible/sgs_models).
//
// From the resolved velocity gradient A_ij = du_i/dx_j (igrid's duidxj
// order, component 3 i + j, components `stride` apart) and the scale
// g = sqrt(mean over the field of |A|^2) the kernels form the normalised
// gradient a = A / g, its strain s = sym(a) - tr(a)/3 I and rotation
// r = skew(a), and
//   features x (10): sqrt tr s^2, sqrt -tr r^2, cbrt tr s^3, cbrt tr r^2 s,
//     (-tr r^2 s^2)^(1/4), signed (tr r^2 s r s^2)^(1/6) (Pope's integrity
//     basis of (s, r), each root taken to the degree of its invariant), the
//     three principal strains of s (descending), and Delta / Delta_0;
//   basis (6 symmetric traceless tensors, Pope 1975):
//     T1 = s, T2 = s r - r s, T3 = s^2 - tr(s^2)/3 I, T4 = r^2 - tr(r^2)/3 I,
//     T5 = r s^2 - s^2 r, T6 = r^2 s + s r^2 - 2/3 tr(s r^2) I;
//   stress tau = Delta^2 g^2 sum_n G_n T_n, G the network's 6 outputs.
// The stress is frame-indifferent: rotating A rotates tau and leaves x and G
// unchanged.  Arithmetic is FP64 per point (full rate on gfx950), except the
// FP32 roots and principal-strain trigonometry of the features.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "pdo_closure.hpp"
#include "pdo_mlp_dev.hpp"

namespace pdo {

namespace {

struct M3 {
    double a[3][3];
};

__device__ __forceinline__ M3 mul(const M3 &x, const M3 &y)
{
    M3 z;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) z.a[i][j] = x.a[i][0] * y.a[0][j] + x.a[i][1] * y.a[1][j] + x.a[i][2] * y.a[2][j];
    return z;
}

__device__ __forceinline__ double tr(const M3 &x) { return x.a[0][0] + x.a[1][1] + x.a[2][2]; }

// the six independent components (11 12 13 22 23 33) of a symmetric tensor
__device__ __forceinline__ void sym6(const M3 &x, double (&o)[6])
{
    o[0] = x.a[0][0];
    o[1] = 0.5 * (x.a[0][1] + x.a[1][0]);
    o[2] = 0.5 * (x.a[0][2] + x.a[2][0]);
    o[3] = x.a[1][1];
    o[4] = 0.5 * (x.a[1][2] + x.a[2][1]);
    o[5] = x.a[2][2];
}

template <typename TS>
__device__ __forceinline__ void strain_rotation(const TS *g, long t, long stride, double inv, M3 &s, M3 &r)
{
    double A[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) A[i][j] = inv * (double)g[t + (3 * i + j) * stride];
    const double t3 = (A[0][0] + A[1][1] + A[2][2]) / 3.0;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            s.a[i][j] = 0.5 * (A[i][j] + A[j][i]) - (i == j ? t3 : 0.0);
            r.a[i][j] = 0.5 * (A[i][j] - A[j][i]);
        }
}

// strain s (11 12 13 22 23 33) and rotation w (r12, r13, r23) of a normalised
// gradient
struct Split {
    double s[6], w[3];
};
__device__ __forceinline__ Split split_of(const double (&A)[9])
{
    const double t3 = (A[0] + A[4] + A[8]) / 3.0;
    return {{A[0] - t3, 0.5 * (A[1] + A[3]), 0.5 * (A[2] + A[6]), A[4] - t3, 0.5 * (A[5] + A[7]), A[8] - t3},
            {0.5 * (A[1] - A[3]), 0.5 * (A[2] - A[6]), 0.5 * (A[5] - A[7])}};
}

// trace of the product of two symmetric tensors
__device__ __forceinline__ double tr2(const double (&x)[6], const double (&y)[6])
{
    return x[0] * y[0] + x[3] * y[3] + x[5] * y[5] + 2.0 * (x[1] * y[1] + x[2] * y[2] + x[4] * y[4]);
}
__device__ __forceinline__ void squares(const Split &q, double (&s2)[6], double (&r2)[6])
{
    const double(&s)[6] = q.s;
    s2[0] = s[0] * s[0] + s[1] * s[1] + s[2] * s[2];
    s2[1] = s[0] * s[1] + s[1] * s[3] + s[2] * s[4];
    s2[2] = s[0] * s[2] + s[1] * s[4] + s[2] * s[5];
    s2[3] = s[1] * s[1] + s[3] * s[3] + s[4] * s[4];
    s2[4] = s[1] * s[2] + s[3] * s[4] + s[4] * s[5];
    s2[5] = s[2] * s[2] + s[4] * s[4] + s[5] * s[5];
    const double a = q.w[0], b = q.w[1], c = q.w[2];
    r2[0] = -(a * a + b * b);
    r2[1] = -(b * c);
    r2[2] = a * c;
    r2[3] = -(a * a + c * c);
    r2[4] = -(a * b);
    r2[5] = -(b * b + c * c);
}
// z = x y for symmetric x, y / x r for any x
__device__ __forceinline__ void mul_ss(const double (&x)[6], const double (&y)[6], double (&z)[9])
{
    constexpr int I[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            z[3 * i + j] = x[I[i][0]] * y[I[0][j]] + x[I[i][1]] * y[I[1][j]] + x[I[i][2]] * y[I[2][j]];
}
template <class F> __device__ __forceinline__ void mul_r(F x, const double (&w)[3], double (&z)[9])
{
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        z[3 * i] = -(x(i, 1) * w[0] + x(i, 2) * w[1]);
        z[3 * i + 1] = x(i, 0) * w[0] - x(i, 2) * w[2];
        z[3 * i + 2] = x(i, 0) * w[1] + x(i, 1) * w[2];
    }
}
__device__ __forceinline__ double sym_at(const double (&x)[6], int i, int j)
{
    constexpr int I[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};
    return x[I[i][j]];
}

// sine and cosine on [0, pi/3] by their Taylor polynomials (to x^11 and x^12:
// truncated below 1e-9, FP32 rounding of about 6e-8 remains)
__device__ __forceinline__ void sincos_third(float x, float &sn, float &cs)
{
    const float z = x * x;
    sn = x * (1.0f + z * (-1.0f / 6 + z * (1.0f / 120 + z * (-1.0f / 5040 + z * (1.0f / 362880 - z * (1.0f / 39916800))))));
    cs = 1.0f + z * (-0.5f + z * (1.0f / 24 + z * (-1.0f / 720 + z * (1.0f / 40320 - z * (1.0f / 3628800 - z * (1.0f / 479001600))))));
}

// The invariants (traces, where cancellation lives) are FP64; their roots and
// the principal-strain trigonometry are FP32, whose ~1e-7 relative error is
// far below the BF16 rounding the network applies to its inputs.
__device__ __forceinline__ void features_of(const Split &d, double dratio, float (&x)[10])
{
    double s2[6], r2[6], r2s[9], s2r[9];
    squares(d, s2, r2);
    const double i1 = s2[0] + s2[3] + s2[5], i2 = -(r2[0] + r2[3] + r2[5]);
    const double i3 = tr2(s2, d.s), i4 = tr2(r2, d.s), i5 = tr2(r2, s2);
    // tr(r^2 s r s^2), r s^2 = -(s^2 r)^T
    mul_ss(r2, d.s, r2s);
    mul_r([&](int i, int j) { return sym_at(s2, i, j); }, d.w, s2r);
    double i6 = 0;
#pragma unroll
    for (int c = 0; c < 9; ++c) i6 -= r2s[c] * s2r[c];
    x[0] = sqrtf(i1 > 0 ? (float)i1 : 0.0f);
    x[1] = sqrtf(i2 > 0 ? (float)i2 : 0.0f);
    x[2] = cbrtf((float)i3);
    x[3] = cbrtf((float)i4);
    x[4] = sqrtf(sqrtf(-i5 > 0 ? (float)-i5 : 0.0f));
    x[5] = copysignf(cbrtf(sqrtf(fabsf((float)i6))), (float)i6);
    // principal strains: roots of l^3 - p l - q = 0, p = tr(s^2)/2, q = det s = tr(s^3)/3
    const double p = 0.5 * i1, q = i3 / 3.0;
    float l0 = 0, l1 = 0, l2 = 0;
    if (p > 1e-300) {
        double c = 1.5 * q / p * sqrt(3.0 / p);
        c = c > 1.0 ? 1.0 : (c < -1.0 ? -1.0 : c);
        const float ph = acosf((float)c) / 3.0f, m = sqrtf((float)(p / 3.0));
        float sn, cs;
        sincos_third(ph, sn, cs);
        // 2 m cos(ph - 2 pi k / 3)
        l0 = 2.0f * m * cs;
        l1 = m * (1.7320508075688772f * sn - cs);
        l2 = -m * (1.7320508075688772f * sn + cs);
    }
    // descending order: l0 >= l1 >= l2 for ph in [0, pi/3]
    x[6] = l0;
    x[7] = l1;
    x[8] = l2;
    x[9] = (float)dratio;
}

// sum_n G_n T_n, components (11 12 13 22 23 33).  T2 = s r + (s r)^T,
// T5 = -(s^2 r + (s^2 r)^T) and T6 = s r r + (s r r)^T up to its trace, so
// the three are N r + (N r)^T with N = G2 s - G5 s^2 + G6 s r.
__device__ __forceinline__ void stress_of(const Split &d, const float (&G)[6], double (&t)[6])
{
    double s2[6], r2[6], sr[9], N[9], Nr[9];
    squares(d, s2, r2);
    mul_r([&](int i, int j) { return sym_at(d.s, i, j); }, d.w, sr);
    const double g2 = G[1], g5 = G[4], g6 = G[5];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            N[3 * i + j] = g2 * sym_at(d.s, i, j) - g5 * sym_at(s2, i, j) + g6 * sr[3 * i + j];
    mul_r([&](int i, int j) { return N[3 * i + j]; }, d.w, Nr);
    const double iso = ((double)G[2] * (s2[0] + s2[3] + s2[5]) + (double)G[3] * (r2[0] + r2[3] + r2[5]) +
                        2.0 * g6 * tr2(d.s, r2)) / 3.0;
    constexpr int I[6] = {0, 0, 0, 1, 1, 2}, J[6] = {0, 1, 2, 1, 2, 2};
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        t[c] = (double)G[0] * d.s[c] + (double)G[2] * s2[c] + (double)G[3] * r2[c] + Nr[3 * I[c] + J[c]] +
               Nr[3 * J[c] + I[c]];
        if (I[c] == J[c]) t[c] -= iso;
    }
}

// the six basis tensors, components (11 12 13 22 23 33)
__device__ void basis_of(const M3 &s, const M3 &r, double (&T)[6][6])
{
    const M3 s2 = mul(s, s), r2 = mul(r, r), sr = mul(s, r), rs = mul(r, s);
    const M3 rs2 = mul(r, s2), s2r = mul(s2, r), r2s = mul(r2, s), sr2 = mul(s, r2);
    const double ts2 = tr(s2) / 3.0, tr2 = tr(r2) / 3.0, tsr2 = 2.0 * tr(sr2) / 3.0;
    M3 b[6];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const double d = i == j ? 1.0 : 0.0;
            b[0].a[i][j] = s.a[i][j];
            b[1].a[i][j] = sr.a[i][j] - rs.a[i][j];
            b[2].a[i][j] = s2.a[i][j] - ts2 * d;
            b[3].a[i][j] = r2.a[i][j] - tr2 * d;
            b[4].a[i][j] = rs2.a[i][j] - s2r.a[i][j];
            b[5].a[i][j] = r2s.a[i][j] + sr2.a[i][j] - tsr2 * d;
        }
#pragma unroll
    for (int n = 0; n < 6; ++n) sym6(b[n], T[n]);
}

__device__ __forceinline__ double inv_scale(const double *sumsq, long npts)
{
    const double ms = sumsq[0] / (double)npts;
    return ms > 0 ? 1.0 / sqrt(ms) : 0.0;
}

unsigned grid_of(long n)
{
    long b = (n + 255) / 256;
    return (unsigned)(b < 8192 ? (b > 0 ? b : 1) : 8192);
}

}  // namespace

// ---------------------------------------------------------------------------
// sum over the field of |A|^2 (partials per block, then one block in order)
// ---------------------------------------------------------------------------
template <typename TS>
__global__ void __launch_bounds__(256) k_grad_sumsq(const TS *__restrict__ g, long n, long stride,
                                                   double *__restrict__ partial)
{
    __shared__ double red[256];
    double acc = 0;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x) {
#pragma unroll
        for (int c = 0; c < 9; ++c) {
            const double v = (double)g[t + c * stride];
            acc = fma(v, v, acc);
        }
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ void __launch_bounds__(256) k_sum_partials(const double *__restrict__ partial, int nb,
                                                     double *__restrict__ out)
{
    __shared__ double red[256];
    double acc = 0;
    for (int i = threadIdx.x; i < nb; i += blockDim.x) acc += partial[i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0];
}

// ---------------------------------------------------------------------------
// features X (n, 10) and, optionally, the normalised gradient a (n, 9).  Bound
// by HBM (FP32: 76 bytes per point after the scale's 36), so one point per
// thread: in a loop over points the compiler held 104 registers for 82, four
// waves per SIMD for five (2^24 FP32 points with their scale 548 us, now 420).
// ---------------------------------------------------------------------------
template <typename TS>
__global__ void __launch_bounds__(256) k_closure_features(const TS *__restrict__ g, long n, long stride,
                                                         const double *__restrict__ sumsq, long nnorm, double dratio,
                                                         float *__restrict__ X, float *__restrict__ A9)
{
    const double inv = inv_scale(sumsq, nnorm);
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    double A[9];
#pragma unroll
    for (int c = 0; c < 9; ++c) A[c] = inv * (double)g[t + c * stride];
    float x[10];
    features_of(split_of(A), dratio, x);
#pragma unroll
    for (int k = 0; k < 10; ++k) X[t * 10 + k] = x[k];
    if (A9) {
#pragma unroll
        for (int c = 0; c < 9; ++c) A9[t * 9 + c] = (float)A[c];
    }
}

// ---------------------------------------------------------------------------
// stress: features, network and basis of a point in one pass.  A wave takes 64
// points; its lanes form the features of one point each, hand them (BF16)
// through LDS to the network's operands, 32 points at a time, and take the
// outputs (FP32) back the same way.  which = 0: write tau 11 12 22 33
// to tau (4 components, stride apart, cells); 1: tau 13 23 (2, edges);
// 2: all six (11 12 13 22 23 33).  fallback: keep the value already in tau
// wherever the network's dissipation -tau_ij S_ij is negative; the number
// of such points of each block goes to nfall[blockIdx.x].
// Bound by the vector unit: the GELUs of the network, then the FP64 algebra.
// 256^3 FP32: features, network and stress as three passes that moved 224
// bytes per point took 1.9 ms (2.3 in a kernel trace: 335, 1600 and 350 us),
// one that moves 60 takes 1.4 (1.65).
// ---------------------------------------------------------------------------
template <typename TS>
__global__ void __launch_bounds__(256, 4)
k_closure_stress(const TS *g, long n, long stride, const double *__restrict__ sumsq, long nnorm, double delta2,
                 double dratio, const unsigned short *__restrict__ Wb, const float *__restrict__ P, int which,
                 int fallback, TS *tau, long tstride, unsigned *__restrict__ nfall)
{
    __shared__ MlpLds L;
    __shared__ u32x4 rows[256 * 2];  // 32 bytes per point: features, then outputs
    __shared__ unsigned cnt[4];
    mlp_stage(L, Wb, P);
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, gq = lane >> 4;
    unsigned *mine = (unsigned *)(rows + (wave * 64 + lane) * 2);
    const double inv = inv_scale(sumsq, nnorm);
    // tau = Delta^2 g^2 sum G_n T_n(a), a = A / g
    const double scale = inv > 0 ? delta2 / (inv * inv) : 0.0;
    unsigned kept = 0;
    const long chunks = (n + 63) / 64;
    for (long ch = (long)blockIdx.x * 4 + wave; ch < chunks; ch += (long)gridDim.x * 4) {
        const long t = 64 * ch + lane;
        TS a[9];
#pragma unroll
        for (int c = 0; c < 9; ++c) a[c] = t < n ? g[t + c * stride] : TS(0);
        {
            double A[9];
            float x[10];
#pragma unroll
            for (int c = 0; c < 9; ++c) A[c] = inv * (double)a[c];
            features_of(split_of(A), dratio, x);
            ((u32x4 *)mine)[0] = (u32x4){pack2(x[0], x[1]), pack2(x[2], x[3]), pack2(x[4], x[5]), pack2(x[6], x[7])};
            ((u32x4 *)mine)[1] = (u32x4){pack2(x[8], x[9]), 0u, 0u, 0u};
        }
        // the lanes of a wave exchange through its own rows: LDS operations
        // of a wave complete in order, the fences keep them in program order
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll 1
        for (int half = 0; half < 2; ++half) {
            u32x2 x[2];
            f32x4 y[2];
#pragma unroll
            for (int q = 0; q < 2; ++q)
                x[q] = ((const u32x2 *)(rows + (wave * 64 + 32 * half + 16 * q + (lane & 15)) * 2))[gq];
            mlp_eval<2>(L, x, y);
            // the rows read above belong to these 32 points alone
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int q = 0; q < 2; ++q)
                if (gq < 2)
                    rows[(wave * 64 + 32 * half + 16 * q + (lane & 15)) * 2 + gq] = __builtin_bit_cast(u32x4, y[q]);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        float G[6];
        {
            const f32x4 y0 = __builtin_bit_cast(f32x4, ((u32x4 *)mine)[0]);
            const u32x2 y1 = ((u32x2 *)mine)[2];
#pragma unroll
            for (int i = 0; i < 4; ++i) G[i] = y0[i];
            G[4] = __uint_as_float(y1[0]);
            G[5] = __uint_as_float(y1[1]);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        double A[9], tv[6];
#pragma unroll
        for (int c = 0; c < 9; ++c) A[c] = inv * (double)a[c];
        const Split d = split_of(A);
        stress_of(d, G, tv);
        if (t >= n) continue;
        // dissipation sign of the normalised stress against the strain
        if (fallback && -tr2(tv, d.s) < 0) {
            ++kept;
            continue;
        }
        if (which == 0) {
            tau[t] = (TS)(scale * tv[0]);
            tau[t + tstride] = (TS)(scale * tv[1]);
            tau[t + 2 * tstride] = (TS)(scale * tv[3]);
            tau[t + 3 * tstride] = (TS)(scale * tv[5]);
        } else if (which == 1) {
            tau[t] = (TS)(scale * tv[2]);
            tau[t + tstride] = (TS)(scale * tv[4]);
        } else {
#pragma unroll
            for (int c = 0; c < 6; ++c) tau[t + c * tstride] = (TS)(scale * tv[c]);
        }
    }
    if (!nfall) return;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) kept += __shfl_xor(kept, o);
    if (lane == 0) cnt[wave] = kept;
    __syncthreads();
    if (threadIdx.x == 0) nfall[blockIdx.x] = cnt[0] + cnt[1] + cnt[2] + cnt[3];
}

// ---------------------------------------------------------------------------
// training loss: L = sum over the batch and the six components of
// w_c (p_c - t_c)^2 / (9 B), w = (1 2 2 1 2 1) (the tensor's nine entries),
// p = sum_n G_n T_n(a); dG (B, 6) = dL/dG; per-block loss partials
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_closure_loss(const float *__restrict__ G, const float *__restrict__ A9,
                                                     const float *__restrict__ Tt, long B, float *__restrict__ dG,
                                                     double *__restrict__ partial)
{
    __shared__ double red[256];
    const double wc[6] = {1, 2, 2, 1, 2, 1};
    const double nrm = 1.0 / (9.0 * (double)B);
    double acc = 0;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < B; t += (long)gridDim.x * blockDim.x) {
        M3 s, r;
        strain_rotation(A9, t * 9, 1, 1.0, s, r);
        double T[6][6];
        basis_of(s, r, T);
        double p[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            const double gk = (double)G[t * 6 + k];
#pragma unroll
            for (int c = 0; c < 6; ++c) p[c] = fma(gk, T[k][c], p[c]);
        }
        double e[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            e[c] = p[c] - (double)Tt[t * 6 + c];
            acc += wc[c] * e[c] * e[c];
        }
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            double d = 0;
#pragma unroll
            for (int c = 0; c < 6; ++c) d = fma(2.0 * wc[c] * e[c], T[k][c], d);
            dG[t * 6 + k] = (float)(d * nrm);
        }
    }
    red[threadIdx.x] = acc * nrm;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
hipError_t launch_grad_sumsq(bool dbl, const void *g, long n, long stride, double *partial, double *out,
                             hipStream_t st)
{
    const unsigned nb = grid_of(n);
    if (dbl)
        hipLaunchKernelGGL(k_grad_sumsq<double>, dim3(nb), dim3(256), 0, st, (const double *)g, n, stride, partial);
    else
        hipLaunchKernelGGL(k_grad_sumsq<float>, dim3(nb), dim3(256), 0, st, (const float *)g, n, stride, partial);
    hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(256), 0, st, partial, (int)nb, out);
    return hipGetLastError();
}

hipError_t launch_closure_features(bool dbl, const void *g, long n, long stride, const double *sumsq, long nnorm,
                                   double dratio, float *X, float *A9, hipStream_t st)
{
    const unsigned nb = (unsigned)((n + 255) / 256);
    if (dbl)
        hipLaunchKernelGGL(k_closure_features<double>, dim3(nb), dim3(256), 0, st, (const double *)g, n, stride,
                           sumsq, nnorm, dratio, X, A9);
    else
        hipLaunchKernelGGL(k_closure_features<float>, dim3(nb), dim3(256), 0, st, (const float *)g, n, stride,
                           sumsq, nnorm, dratio, X, A9);
    return hipGetLastError();
}

template <typename TS>
static hipError_t stress_t(const void *g, long n, long stride, const double *sumsq, long nnorm, double delta2,
                           double dratio, const unsigned short *Wb, const float *P, int which, int fallback, void *tau,
                           long tstride, unsigned *nfall, int *blocks, hipStream_t st)
{
    static Resident resident;
    int res = 0;
    const hipError_t e = resident_blocks(resident, (const void *)k_closure_stress<TS>, 256, &res);
    if (e != hipSuccess) return e;
    const long need = (n + 255) / 256;
    const long nb = std::min(std::min(need, (long)res), 8192L);
    *blocks = (int)nb;
    hipLaunchKernelGGL(k_closure_stress<TS>, dim3((unsigned)nb), dim3(256), 0, st, (const TS *)g, n, stride, sumsq,
                       nnorm, delta2, dratio, Wb, P, which, fallback, (TS *)tau, tstride, nfall);
    return hipGetLastError();
}

hipError_t launch_closure_stress(bool dbl, const void *g, long n, long stride, const double *sumsq, long nnorm,
                                 double delta2, double dratio, const unsigned short *Wb, const float *P, int which,
                                 int fallback, void *tau, long tstride, unsigned *nfall, int *blocks, hipStream_t st)
{
    return (dbl ? stress_t<double> : stress_t<float>)(g, n, stride, sumsq, nnorm, delta2, dratio, Wb, P, which,
                                                      fallback, tau, tstride, nfall, blocks, st);
}

hipError_t launch_closure_loss(const float *G, const float *A9, const float *T, long B, float *dG, double *partial,
                               double *loss, hipStream_t st)
{
    const unsigned nb = grid_of(B);
    hipLaunchKernelGGL(k_closure_loss, dim3(nb), dim3(256), 0, st, G, A9, T, B, dG, partial);
    hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(256), 0, st, partial, (int)nb, loss);
    return hipGetLastError();
}

}  // namespace pdo
