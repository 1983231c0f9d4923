// Pointwise kernels of the igrid pieces (interp_PrimitiveVars, getRHS_SGS,
// the nonlinear and viscous terms, the Runge-Kutta stage updates).  All of
// them stream their operands once (HBM-bound, grid-stride loops).  mode: 0
// FP64, 1 FP32, 2 FP32 storage with FP64 arithmetic.
#include <hip/hip_runtime.h>

#include "pdo_igrid.hpp"
#include "pdo_sgs_dev.hpp"

namespace pdo {

namespace {

template <typename TS> struct C2;
template <> struct C2<double> { using V = double2; };
template <> struct C2<float> { using V = float2; };

unsigned blocks_for(long n)
{
    long b = (n + 255) / 256;
    return (unsigned)(b < 8192 ? (b > 0 ? b : 1) : 8192);
}

#define PDO_GRID_STRIDE(t, n) \
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < (n); t += (long)gridDim.x * blockDim.x)

// plane 0 of a (nxh, ny, nz+1) spectrum set to zero, its mean mode to v
template <typename TS>
__global__ void __launch_bounds__(256) k_surface_plane(TS *f, long nplane, double v)
{
    using V = typename C2<TS>::V;
    V *z = (V *)f;
    PDO_GRID_STRIDE(t, nplane) z[t] = V{(TS)(t == 0 ? v : 0.0), (TS)0};
}

// 32-bit index arithmetic of (i, j) of a complex value: fields of a plane
// count below 2^31 values
__device__ __forceinline__ void line_of(unsigned t, unsigned nxh, unsigned ny, unsigned &i, unsigned &j)
{
    const unsigned q = t / nxh;
    i = t - q * nxh;
    j = q % ny;
}

// subgrid viscosity and stress in one pass over the gradients: the strain
// stays in registers (it was a field of six components, written, and read
// again by the stress kernel: 36 words per cell and 24 per edge, now 14 and
// 8).  nu is the model kernel times its constant.
template <typename TS, typename TC, bool EDGES>
__global__ void __launch_bounds__(256) k_sgs_tau(const TS *__restrict__ g, TS *__restrict__ nu, TS *__restrict__ tau,
                                                long n, long nxy, int model, TC cx, TC cy, TC cz,
                                                const double *__restrict__ cplane, double cglobal)
{
    PDO_GRID_STRIDE(t, n)
    {
        TC d[9], s[6];
#pragma unroll
        for (int c = 0; c < 9; ++c) d[c] = (TC)g[t + c * n];
        strain<TC>(d, s);
        const TS v = (TS)((double)(TS)sgs_viscosity<TC>(d, s, model, cx, cy, cz) * (cplane ? cplane[t / nxy] : cglobal));
        nu[t] = v;
        const TC m = (TC)-2 * (TC)v;
        if constexpr (EDGES) {
            tau[t] = (TS)(m * s[2]);
            tau[t + n] = (TS)(m * s[4]);
        } else {
            tau[t] = (TS)(m * s[0]);
            tau[t + n] = (TS)(m * s[1]);
            tau[t + 2 * n] = (TS)(m * s[3]);
            tau[t + 3 * n] = (TS)(m * s[5]);
        }
    }
}

// edge stresses 13, 23 from an interpolated viscosity
template <typename TS, typename TC>
__global__ void __launch_bounds__(256) k_edge_tau(const TS *__restrict__ g, TS *nu, TS *__restrict__ tau, long n,
                                                 bool clip)
{
    PDO_GRID_STRIDE(t, n)
    {
        TS v = nu[t];
        if (clip && v < (TS)0) {
            v = (TS)0;
            nu[t] = v;
        }
        const TC m = (TC)-2 * (TC)v;
        const TC s13 = (TC)0.5 * ((TC)g[t + 2 * n] + (TC)g[t + 6 * n]);
        const TC s23 = (TC)0.5 * ((TC)g[t + 5 * n] + (TC)g[t + 7 * n]);
        tau[t] = (TS)(m * s13);
        tau[t + n] = (TS)(m * s23);
    }
}

// the stress divergence of the three components in one pass (it was a
// read-modify-write of the right-hand side per term: 27 words, now 14)
template <typename TS, typename TC>
__global__ void __launch_bounds__(256) k_stress_div(TS *u, TS *v, TS *w, StressSpectra S,
                                                   const double *__restrict__ k1, const double *__restrict__ k2,
                                                   unsigned nxh, unsigned ny, long ncell, long nedge)
{
    using V = typename C2<TS>::V;
    auto at = [](const void *p, long t) { return ((const V *)p)[t]; };
    // r -= i (a p + b q) + z
    auto term = [](V *r, long t, TC a, V p, TC b, V q, V z) {
        const V o = r[t];
        r[t] = V{(TS)((TC)o.x + a * (TC)p.y + b * (TC)q.y - (TC)z.x), (TS)((TC)o.y - a * (TC)p.x - b * (TC)q.x - (TC)z.y)};
    };
    PDO_GRID_STRIDE(t, nedge)
    {
        unsigned i, j;
        line_of((unsigned)t, nxh, ny, i, j);
        const TC a = (TC)k1[i], b = (TC)k2[j];
        if (t < ncell) {
            const V t12 = at(S.t12, t);
            term((V *)u, t, a, at(S.t11, t), b, t12, at(S.z13, t));
            term((V *)v, t, a, t12, b, at(S.t22, t), at(S.z23, t));
        }
        term((V *)w, t, a, at(S.t13, t), b, at(S.t23, t), at(S.z33, t));
    }
}

// the nonlinear term's cell part and addViscousTerm (igrid.F90:1914-1959)
template <typename TS, typename TC>
__global__ void __launch_bounds__(256) k_rhs_terms(RhsTerms T, const double *__restrict__ k1,
                                                  const double *__restrict__ k2, unsigned nxh, unsigned ny, long ncell,
                                                  long nedge, TC invRe)
{
    using V = typename C2<TS>::V;
    PDO_GRID_STRIDE(t, nedge)
    {
        unsigned i, j;
        line_of((unsigned)t, nxh, ny, i, j);
        const TC ks = (TC)(k1[i] * k1[i] + k2[j] * k2[j]);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            if (c < 2 && t >= ncell) continue;
            if (!T.s[c] && invRe == (TC)0) continue;
            V *r = (V *)T.rhs[c];
            V o = r[t];
            if (T.s[c]) {
                const V x = ((const V *)T.s[c])[t];
                o.x = (TS)((TC)o.x + (TC)x.x);
                o.y = (TS)((TC)o.y + (TC)x.y);
            }
            if (invRe != (TC)0) {
                const V x = ((const V *)T.f[c])[t], y = ((const V *)T.d2[c])[t];
                o.x = (TS)((TC)o.x + invRe * (-ks * (TC)x.x + (TC)y.x));
                o.y = (TS)((TC)o.y + invRe * (-ks * (TC)x.y + (TC)y.y));
            }
            r[t] = o;
        }
    }
}

// a Runge-Kutta stage of the three components with the x-y dealiasing mask
template <typename TS, typename TC>
__global__ void __launch_bounds__(256) k_stage(StageTerms T, const double *__restrict__ g1,
                                              const double *__restrict__ g2, unsigned nxh, unsigned ny, long ncell,
                                              long nedge)
{
    using V = typename C2<TS>::V;
    PDO_GRID_STRIDE(t, nedge)
    {
        unsigned i, j;
        line_of((unsigned)t, nxh, ny, i, j);
        const bool keep = g1[i] * g2[j] != 0.0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            if (c < 2 && t >= ncell) continue;
            V o{(TS)0, (TS)0};
            if (keep) {
                const V x0 = ((const V *)T.x[0][c])[t];
                TC re = (TC)T.coef[0] * (TC)x0.x, im = (TC)T.coef[0] * (TC)x0.y;
#pragma unroll
                for (int q = 1; q < 5; ++q)
                    if (q < T.nterms) {
                        const V x = ((const V *)T.x[q][c])[t];
                        re += (TC)T.coef[q] * (TC)x.x;
                        im += (TC)T.coef[q] * (TC)x.y;
                    }
                o = V{(TS)re, (TS)im};
            }
            ((V *)T.out[c])[t] = o;
        }
    }
}

// partial maxima of |u|/dx + |v|/dy + |w|/dz over the blocks of the grid
template <typename TS>
__global__ void __launch_bounds__(256) k_cfl(const TS *u, const TS *v, const TS *w, long n, double idx, double idy,
                                           double idz, double *partial)
{
    __shared__ double red[256];
    double m = 0.0;
    PDO_GRID_STRIDE(t, n)
    {
        const double s = fabs((double)u[t] * idx) + fabs((double)v[t] * idy) + fabs((double)w[t] * idz);
        m = s > m ? s : m;
    }
    red[threadIdx.x] = m;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + o]);
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// ---------------------------------------------------------------------------
// HIT_shell_forcing (forcingIsotropic.F90:123-314) on a periodic-z grid: for
// each of nwaves random wave vectors (kx, ky, kz) >= 0 the 3D Fourier
// coefficients of (uhat, vhat, what) at that mode (a z transform of the
// 2D spectra at one frequency; w shifted from edges to cells), the forcing
// fac conj(u_k) with fac = normfact eps / (|u_k|^2 + |v_k|^2 + |w_k|^2 +
// 1e-14) / nwaves, and its inverse z transform (1/nz; w shifted back to the
// edges, plane nz repeating plane 0) added to the right-hand sides.  One
// workgroup takes the modes in order, so repeated modes add up as in the
// reference.  The random draws: splitmix64 of (seed, draw counter, wave,
// variable), uniform in [0, 1) from the top 53 bits.
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned long long splitmix64(unsigned long long x)
{
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

__device__ __forceinline__ double uniform01(unsigned long long seed, unsigned long long draw, int ik, int q)
{
    const unsigned long long key = splitmix64(splitmix64(seed + draw) + 3ull * (unsigned long long)ik + (unsigned)q);
    return (double)(key >> 11) * 0x1.0p-53;
}

template <typename TS>
__global__ void __launch_bounds__(256) k_hit_forcing(const TS *uhat, const TS *vhat, const TS *what, TS *urhs,
                                                   TS *vrhs, TS *wrhs, HitForcingArgs F)
{
    using V = typename C2<TS>::V;
    __shared__ double red[6][256];
    __shared__ double sfac[7];
    const int tid = threadIdx.x;
    const long plane = (long)F.nxh * F.ny;
    const int nz = F.nz;
    for (int ik = 0; ik < F.nwaves; ++ik) {
        // pick_random_wavenumbers (:133-156)
        const double kabs = F.kmin + (F.kmax - F.kmin) * uniform01(F.seed, F.draw, ik, 0);
        const double zeta = -1.0 + 2.0 * uniform01(F.seed, F.draw, ik, 1);
        const double theta = 2.0 * M_PI * uniform01(F.seed, F.draw, ik, 2);
        const double sz = sqrt(1.0 - zeta * zeta);
        const int wx = (int)ceil(fabs(kabs * sz * cos(theta)));
        const int wy = (int)ceil(fabs(kabs * sz * sin(theta)));
        const int wz = (int)ceil(fabs(kabs * zeta));
        // the host keeps ceil(kmax) below nx/2, ny and nz
        const long col = (long)wx + (long)F.nxh * wy;
        double acc[6] = {0, 0, 0, 0, 0, 0};
        for (int k = tid; k < nz; k += 256) {
            double sn, cs;
            sincospi(-2.0 * (double)((long)wz * k % nz) / (double)nz, &sn, &cs);
            const V a = ((const V *)uhat)[col + (long)k * plane];
            const V b = ((const V *)vhat)[col + (long)k * plane];
            const V c = ((const V *)what)[col + (long)k * plane];
            acc[0] += (double)a.x * cs - (double)a.y * sn;
            acc[1] += (double)a.x * sn + (double)a.y * cs;
            acc[2] += (double)b.x * cs - (double)b.y * sn;
            acc[3] += (double)b.x * sn + (double)b.y * cs;
            acc[4] += (double)c.x * cs - (double)c.y * sn;
            acc[5] += (double)c.x * sn + (double)c.y * cs;
        }
        for (int q = 0; q < 6; ++q) red[q][tid] = acc[q];
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            if (tid < o)
                for (int q = 0; q < 6; ++q) red[q][tid] += red[q][tid + o];
            __syncthreads();
        }
        if (tid == 0) {
            // w: shiftz_E2C, times exp(i k3 dz / 2)
            const double k3 = F.k3[wz];
            double es, ec;
            sincos(0.5 * k3 * F.dz, &es, &ec);
            const double wr = red[4][0] * ec - red[5][0] * es, wi = red[4][0] * es + red[5][0] * ec;
            const double den = red[0][0] * red[0][0] + red[1][0] * red[1][0] + red[2][0] * red[2][0] +
                               red[3][0] * red[3][0] + wr * wr + wi * wi + 1.0e-14;
            const double fac = F.normfact * F.eps / den / (double)F.nwaves;
            // forcing coefficients fac conj(.) ; w shifted back by exp(-i k3 dz / 2)
            sfac[0] = fac * red[0][0];
            sfac[1] = -fac * red[1][0];
            sfac[2] = fac * red[2][0];
            sfac[3] = -fac * red[3][0];
            const double fr = fac * wr, fi = -fac * wi;
            sfac[4] = fr * ec + fi * es;
            sfac[5] = -fr * es + fi * ec;
        }
        __syncthreads();
        // inverse z transform (1/nz) of the single mode into every plane
        const double inz = 1.0 / (double)nz;
        for (int k = tid; k <= nz; k += 256) {
            const int kk = k == nz ? 0 : k;
            double sn, cs;
            sincospi(2.0 * (double)((long)wz * kk % nz) / (double)nz, &sn, &cs);
            const long idx = col + (long)k * plane;
            if (k < nz) {
                V *ru = (V *)urhs + idx;
                V *rv = (V *)vrhs + idx;
                V o = *ru;
                o.x = (TS)((double)o.x + (sfac[0] * cs - sfac[1] * sn) * inz);
                o.y = (TS)((double)o.y + (sfac[0] * sn + sfac[1] * cs) * inz);
                *ru = o;
                o = *rv;
                o.x = (TS)((double)o.x + (sfac[2] * cs - sfac[3] * sn) * inz);
                o.y = (TS)((double)o.y + (sfac[2] * sn + sfac[3] * cs) * inz);
                *rv = o;
            }
            V *rw = (V *)wrhs + idx;
            V o = *rw;
            o.x = (TS)((double)o.x + (sfac[4] * cs - sfac[5] * sn) * inz);
            o.y = (TS)((double)o.y + (sfac[4] * sn + sfac[5] * cs) * inz);
            *rw = o;
        }
        __syncthreads();
    }
}

template <typename TS, typename TC>
hipError_t surface_t(void *f, long nplane, double v, hipStream_t st)
{
    hipLaunchKernelGGL((k_surface_plane<TS>), dim3(blocks_for(nplane)), dim3(256), 0, st, (TS *)f, nplane, v);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_surface_plane(int mode, void *f, long nplane, double v, hipStream_t st)
{
    if (mode == 0) return surface_t<double, double>(f, nplane, v, st);
    return surface_t<float, float>(f, nplane, v, st);
}

// ---------------------------------------------------------------------------
// Moeng wall model: first-plane sums, the surface quantities, the embedded
// wall stresses
// ---------------------------------------------------------------------------
namespace {

template <typename TS>
__global__ void __launch_bounds__(256) k_wall_sums(const TS *u, const TS *v, long nxy, double *part)
{
    __shared__ double ss[256], su[256];
    double a = 0, b = 0;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < nxy; i += (long)gridDim.x * 256) {
        const double x = (double)u[i], y = (double)v[i];
        a += sqrt(x * x + y * y);
        b += x;
    }
    ss[threadIdx.x] = a;
    su[threadIdx.x] = b;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            ss[threadIdx.x] += ss[threadIdx.x + w];
            su[threadIdx.x] += su[threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = ss[0];
        part[2 * blockIdx.x + 1] = su[0];
    }
}

__global__ void __launch_bounds__(256) k_wall_finalize(const double *part, int nb, double meanfact, double kappa,
                                                      double lg, double *wm)
{
    __shared__ double ss[256], su[256];
    double a = 0, b = 0;
    for (int i = threadIdx.x; i < nb; i += 256) {
        a += part[2 * i];
        b += part[2 * i + 1];
    }
    ss[threadIdx.x] = a;
    su[threadIdx.x] = b;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            ss[threadIdx.x] += ss[threadIdx.x + w];
            su[threadIdx.x] += su[threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double Uspmn = ss[0] * meanfact;
        const double ustar = Uspmn * kappa / lg;
        wm[0] = Uspmn;
        wm[1] = ustar;
        wm[2] = -ustar * ustar / (Uspmn + 1.0e-13);
        wm[3] = su[0] * meanfact;
    }
}

template <typename TS>
__global__ void __launch_bounds__(256) k_wall_embed(const TS *u, const TS *v, TS *tauE, long nxy, long nE,
                                                   const double *wm)
{
    const double M = wm[2];
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < nxy; i += (long)gridDim.x * 256) {
        tauE[i] = (TS)(M * (double)u[i]);
        tauE[nE + i] = (TS)(M * (double)v[i]);
    }
}

template <typename TS>
hipError_t wall_t(const void *u, const void *v, void *tauE, long nxy, long nE, double *part, int nb, double kappa,
                  double lg, double *wm, hipStream_t st)
{
    hipLaunchKernelGGL((k_wall_sums<TS>), dim3(nb), dim3(256), 0, st, (const TS *)u, (const TS *)v, nxy, part);
    hipLaunchKernelGGL(k_wall_finalize, dim3(1), dim3(256), 0, st, (const double *)part, nb, 1.0 / (double)nxy,
                       kappa, lg, wm);
    hipLaunchKernelGGL((k_wall_embed<TS>), dim3(blocks_for(nxy)), dim3(256), 0, st, (const TS *)u, (const TS *)v,
                       (TS *)tauE, nxy, nE, (const double *)wm);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_wall_model(int mode, const void *u, const void *v, void *tauE, long nxy, long nE, double *part,
                             int nb, double kappa, double lg, double *wm, hipStream_t st)
{
    if (mode == 0) return wall_t<double>(u, v, tauE, nxy, nE, part, nb, kappa, lg, wm, st);
    return wall_t<float>(u, v, tauE, nxy, nE, part, nb, kappa, lg, wm, st);
}

namespace {
template <typename TS>
__global__ void __launch_bounds__(256) k_mean_add(TS *f, long nplane, int nz, double v)
{
    for (int k = blockIdx.x * 256 + threadIdx.x; k < nz; k += gridDim.x * 256) {
        TS *m = f + 2 * (long)k * nplane;
        *m = (TS)((double)*m + v);
    }
}
}  // namespace

hipError_t launch_mean_add(int mode, void *f, long nplane, int nz, double v, hipStream_t st)
{
    const dim3 g((unsigned)((nz + 255) / 256));
    if (mode == 0) hipLaunchKernelGGL((k_mean_add<double>), g, dim3(256), 0, st, (double *)f, nplane, nz, v);
    else hipLaunchKernelGGL((k_mean_add<float>), g, dim3(256), 0, st, (float *)f, nplane, nz, v);
    return hipGetLastError();
}

// calls F<TS, TC> of the mode
#define PDO_MODES(CALL)                        \
    switch (mode) {                            \
    case 0: { CALL(double, double); break; }   \
    case 1: { CALL(float, float); break; }     \
    default: { CALL(float, double); }          \
    }                                          \
    return hipGetLastError();

hipError_t launch_sgs_tau(int mode, bool edges, const void *g, void *nu, void *tau, long n, long nxy, int model,
                          const double (&camd)[3], const double *cplane, double cglobal, hipStream_t st)
{
    const dim3 gr(blocks_for(n)), b(256);
#define PDO_CALL(TS, TC)                                                                                          \
    if (edges)                                                                                                    \
        hipLaunchKernelGGL((k_sgs_tau<TS, TC, true>), gr, b, 0, st, (const TS *)g, (TS *)nu, (TS *)tau, n, nxy,   \
                           model, (TC)camd[0], (TC)camd[1], (TC)camd[2], cplane, cglobal);                        \
    else                                                                                                          \
        hipLaunchKernelGGL((k_sgs_tau<TS, TC, false>), gr, b, 0, st, (const TS *)g, (TS *)nu, (TS *)tau, n, nxy,  \
                           model, (TC)camd[0], (TC)camd[1], (TC)camd[2], cplane, cglobal);
    PDO_MODES(PDO_CALL)
#undef PDO_CALL
}

hipError_t launch_edge_tau(int mode, bool clip, const void *g, void *nu, void *tau, long n, hipStream_t st)
{
#define PDO_CALL(TS, TC)                                                                                           \
    hipLaunchKernelGGL((k_edge_tau<TS, TC>), dim3(blocks_for(n)), dim3(256), 0, st, (const TS *)g, (TS *)nu,       \
                       (TS *)tau, n, clip)
    PDO_MODES(PDO_CALL)
#undef PDO_CALL
}

hipError_t launch_stress_div(int mode, void *u, void *v, void *w, const StressSpectra &S, const double *k1,
                             const double *k2, int nxh, int ny, long ncell, long nedge, hipStream_t st)
{
#define PDO_CALL(TS, TC)                                                                                         \
    hipLaunchKernelGGL((k_stress_div<TS, TC>), dim3(blocks_for(nedge)), dim3(256), 0, st, (TS *)u, (TS *)v,      \
                       (TS *)w, S, k1, k2, (unsigned)nxh, (unsigned)ny, ncell, nedge)
    PDO_MODES(PDO_CALL)
#undef PDO_CALL
}

hipError_t launch_rhs_terms(int mode, const RhsTerms &T, const double *k1, const double *k2, int nxh, int ny,
                            long ncell, long nedge, double invRe, hipStream_t st)
{
#define PDO_CALL(TS, TC)                                                                                           \
    hipLaunchKernelGGL((k_rhs_terms<TS, TC>), dim3(blocks_for(nedge)), dim3(256), 0, st, T, k1, k2, (unsigned)nxh, \
                       (unsigned)ny, ncell, nedge, (TC)invRe)
    PDO_MODES(PDO_CALL)
#undef PDO_CALL
}

hipError_t launch_stage(int mode, const StageTerms &T, const double *g1, const double *g2, int nxh, int ny, long ncell,
                        long nedge, hipStream_t st)
{
    if (T.nterms < 1 || T.nterms > 5) return hipErrorInvalidValue;
#define PDO_CALL(TS, TC)                                                                                       \
    hipLaunchKernelGGL((k_stage<TS, TC>), dim3(blocks_for(nedge)), dim3(256), 0, st, T, g1, g2, (unsigned)nxh, \
                       (unsigned)ny, ncell, nedge)
    PDO_MODES(PDO_CALL)
#undef PDO_CALL
}

hipError_t launch_cfl(int mode, const void *u, const void *v, const void *w, long n, double idx, double idy,
                      double idz, double *partial, int nblocks, hipStream_t st)
{
    if (mode == 0)
        hipLaunchKernelGGL((k_cfl<double>), dim3(nblocks), dim3(256), 0, st, (const double *)u, (const double *)v,
                           (const double *)w, n, idx, idy, idz, partial);
    else
        hipLaunchKernelGGL((k_cfl<float>), dim3(nblocks), dim3(256), 0, st, (const float *)u, (const float *)v,
                           (const float *)w, n, idx, idy, idz, partial);
    return hipGetLastError();
}

hipError_t launch_hit_forcing(int mode, const void *uhat, const void *vhat, const void *what, void *urhs, void *vrhs,
                              void *wrhs, const HitForcingArgs &F, hipStream_t st)
{
    if (mode == 0)
        hipLaunchKernelGGL((k_hit_forcing<double>), dim3(1), dim3(256), 0, st, (const double *)uhat,
                           (const double *)vhat, (const double *)what, (double *)urhs, (double *)vrhs,
                           (double *)wrhs, F);
    else
        hipLaunchKernelGGL((k_hit_forcing<float>), dim3(1), dim3(256), 0, st, (const float *)uhat, (const float *)vhat,
                           (const float *)what, (float *)urhs, (float *)vrhs, (float *)wrhs, F);
    return hipGetLastError();
}

}  // namespace pdo
