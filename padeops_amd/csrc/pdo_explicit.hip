// Explicit symmetric 9-point filters (gaussianstuff, lstsqstuff: the
// Gaussian filter of width 4 dx and the least-squares filter) along x, y or
// z of a field f(n, na, nb) / (na, n, nb) / (na, nb, n).
//
// Interior rows use the symmetric stencil c0 f_j + sum_q c_q (f_{j+q} +
// f_{j-q}); periodic rows wrap; the first and last NB rows of a
// non-periodic pencil take their weights from a closure table (NB rows of
// WB weights against the first / last WB points).  FP64 arithmetic for both
// storage types.
//
// The filter is applied NP = 1 or 2 times in one pass over HBM, which bounds
// it (2 words per point).  y and z: a lane carries T consecutive rows of its
// pencil in registers and reads 4 NP rows more on either side, which its
// neighbours in the direction read too (from the cache); the first and last
// chunk are flush with the pencil, so closure rows sit at fixed registers.  x:
// whole lines staged in LDS.  One thread per point with nine loads each spends
// its time on 64-bit index divisions (256^3 FP64, two applications 2 x 116 us,
// in one pass 52 us along y and z, 81 us along x); it is the shorter way for
// fields of few points (launch_fast).
#include <algorithm>

#include "pdo_explicit.hpp"

namespace pdo {

constexpr int EXPL_T = 16;  // rows of a lane

// one application on registers: in[w] is row r0 - 4 PASSES + w, out[j] row
// r0 - 4 (PASSES - 1) + j; first / last: the chunk holds the pencil's ends
template <int PASSES, typename TW>
__device__ __forceinline__ void filter_rows(const ExplicitArgs &E, const TW (&in)[EXPL_T + 8 * PASSES],
                                            double (&out)[EXPL_T + 8 * (PASSES - 1)], bool first, bool last)
{
    constexpr int N = EXPL_T + 8 * (PASSES - 1);
#pragma unroll
    for (int j = 0; j < N; ++j) {
        double acc = E.c[0] * (double)in[j + 4];
#pragma unroll
        for (int q = 1; q <= EXPL_R; ++q) acc += E.c[q] * ((double)in[j + 4 + q] + (double)in[j + 4 - q]);
        out[j] = acc;
    }
    // row 0 of the pencil is in[4 PASSES] of the first chunk, row n - 1
    // in[T - 1 + 4 PASSES] of the last
    if (first) {
#pragma unroll
        for (int i = 0; i < EXPL_NB; ++i) {
            double acc = 0;
#pragma unroll
            for (int q = 0; q < EXPL_WB; ++q) acc += E.left[i * EXPL_WB + q] * (double)in[4 * PASSES + q];
            out[4 * (PASSES - 1) + i] = acc;
        }
    }
    if (last) {
#pragma unroll
        for (int i = 0; i < EXPL_NB; ++i) {
            double acc = 0;
#pragma unroll
            for (int q = 0; q < EXPL_WB; ++q)
                acc += E.right[i * EXPL_WB + q] * (double)in[EXPL_T - EXPL_WB + 4 * PASSES + q];
            out[EXPL_T - EXPL_NB + 4 * (PASSES - 1) + i] = acc;
        }
    }
}

// y and z: lanes over the pencils, blockIdx.y over chunks of T rows (chunked(n))
template <typename TS, int NP>
__global__ void __launch_bounds__(256) k_expl_strided(ExplicitArgs E, ExplicitFields F)
{
    const TS *f = (const TS *)F.f[blockIdx.z];
    TS *out = (TS *)F.out[blockIdx.z];
    const unsigned id = blockIdx.x * 256 + threadIdx.x, na = (unsigned)E.na;
    const unsigned pencils = na * (unsigned)E.nb;
    if (id >= pencils) return;
    // element of row 0, and the row stride
    const unsigned b = E.dir == 2 ? id / na : 0;
    const size_t base = E.dir == 2 ? (size_t)b * na * E.n + (id - b * na) : id;
    const size_t st = E.dir == 2 ? na : pencils;
    // chunks of T rows, evenly spaced from the pencil's start to its end, each
    // storing the rows up to the next one's start
    const int n = E.n, steps = (int)gridDim.y - 1, c = (int)blockIdx.y;
    const int r0 = steps > 0 ? c * (n - EXPL_T) / steps : 0;
    const int own = c < steps ? (c + 1) * (n - EXPL_T) / steps - r0 : EXPL_T;
    const bool first = !E.periodic && c == 0, last = !E.periodic && c == steps;
    TS win[EXPL_T + 8 * NP];
#pragma unroll
    for (int w = 0; w < EXPL_T + 8 * NP; ++w) {
        // rows past the ends wrap; without periodicity they enter closure
        // rows' places only
        int r = r0 - 4 * NP + w;
        r += r < 0 ? n : 0;
        r -= r >= n ? n : 0;
        win[w] = f[base + (size_t)r * st];
    }
    double y[EXPL_T];
    if constexpr (NP == 2) {
        double x[EXPL_T + 8];
        filter_rows<2>(E, win, x, first, last);
        filter_rows<1>(E, x, y, first, last);
    } else {
        filter_rows<1>(E, win, y, first, last);
    }
#pragma unroll
    for (int j = 0; j < EXPL_T; ++j)
        if (j < own) out[base + (size_t)(r0 + j) * st] = (TS)y[j];
}

// x: `lines` whole lines per workgroup in LDS; element e is point
// e % n of line e / n (magic: the rounded-up reciprocal of n).  NT: 256
// threads, or up to 1024
template <typename TS, int NP, int NT>
__global__ void __launch_bounds__(NT) k_expl_x(ExplicitArgs E, ExplicitFields F, int lines, unsigned magic)
{
    const int nt = NT == 256 ? 256 : blockDim.x;
    const TS *f = (const TS *)F.f[blockIdx.z];
    TS *out = (TS *)F.out[blockIdx.z];
    extern __shared__ double lds[];
    const int n = E.n;
    const long l0 = (long)blockIdx.x * lines, left = (long)E.na * E.nb - l0;
    const int total = (int)(left < lines ? left : lines) * n;
    TS *tile = (TS *)(lds + (NP == 2 ? lines * n : 0));
    f += l0 * n;
    out += l0 * n;
#pragma unroll 4
    for (int e = threadIdx.x; e < total; e += nt) tile[e] = f[e];
    __syncthreads();
    auto apply = [&](const auto *src, auto put) {
#pragma unroll 2
        for (int e = threadIdx.x; e < total; e += nt) {
            const int r = e - (int)__umulhi((unsigned)e, magic) * n;
            const auto *p = src + (e - r);
            double acc;
            if (!E.periodic && r < EXPL_NB) {
                acc = 0;
                for (int q = 0; q < EXPL_WB; ++q) acc += E.left[r * EXPL_WB + q] * (double)p[q];
            } else if (!E.periodic && r >= n - EXPL_NB) {
                acc = 0;
                for (int q = 0; q < EXPL_WB; ++q)
                    acc += E.right[(r - (n - EXPL_NB)) * EXPL_WB + q] * (double)p[n - EXPL_WB + q];
            } else {
                acc = E.c[0] * (double)p[r];
#pragma unroll
                for (int q = 1; q <= EXPL_R; ++q) {
                    int hi = r + q, lo = r - q;
                    hi -= hi >= n ? n : 0;
                    lo += lo < 0 ? n : 0;
                    acc += E.c[q] * ((double)p[hi] + (double)p[lo]);
                }
            }
            put(e, acc);
        }
    };
    if constexpr (NP == 2) {
        apply(tile, [&](int e, double v) { lds[e] = v; });
        __syncthreads();
        apply(lds, [&](int e, double v) { out[e] = (TS)v; });
    } else {
        apply(tile, [&](int e, double v) { out[e] = (TS)v; });
    }
}

// one application, what the two others don't take (y, z: 8 .. 15 rows, 17 ..
// 23 without periodicity; x: above 4096) or take longer for (launch_fast): one
// thread per output point along the contiguous index
template <typename TS, typename TA>
__global__ void __launch_bounds__(256) k_explicit(ExplicitArgs E, const TS *__restrict__ f, TS *__restrict__ out)
{
    const long total = (long)E.n * E.na * E.nb;
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
        // row r of the pencil through element e, and the element stride of rows
        long r, st;
        if (E.dir == 1) { r = e % E.n; st = 1; }
        else if (E.dir == 2) { r = (e / E.na) % E.n; st = E.na; }
        else { r = e / ((long)E.na * E.nb); st = (long)E.na * E.nb; }
        const TS *p = f + (e - r * st);  // row 0 of this pencil
        TA acc;
        if (E.periodic) {
            acc = (TA)E.c[0] * (TA)p[r * st];
#pragma unroll
            for (int q = 1; q <= EXPL_R; ++q) {
                long a = r + q, b = r - q;
                a -= (a >= E.n) ? E.n : 0;
                b += (b < 0) ? E.n : 0;
                acc += (TA)E.c[q] * ((TA)p[a * st] + (TA)p[b * st]);
            }
        } else if (r < EXPL_NB) {
            acc = 0;
#pragma unroll
            for (int q = 0; q < EXPL_WB; ++q) acc += (TA)E.left[r * EXPL_WB + q] * (TA)p[q * st];
        } else if (r >= E.n - EXPL_NB) {
            const long j = r - (E.n - EXPL_NB);
            const TS *pe = p + (E.n - EXPL_WB) * st;
            acc = 0;
#pragma unroll
            for (int q = 0; q < EXPL_WB; ++q) acc += (TA)E.right[j * EXPL_WB + q] * (TA)pe[q * st];
        } else {
            acc = (TA)E.c[0] * (TA)p[r * st];
#pragma unroll
            for (int q = 1; q <= EXPL_R; ++q) acc += (TA)E.c[q] * ((TA)p[(r + q) * st] + (TA)p[(r - q) * st]);
        }
        out[e] = (TS)acc;
    }
}

// whether a strided pencil can be cut into chunks: without periodicity only
// the first and the last may reach closure rows, with the 4 rows of the first
// application's margin, so the second starts 8 rows in (all n but 17 .. 23).
// 2^17 rows bound the grid and the products of the chunk starts.
static bool chunked(const ExplicitArgs &E)
{
    const int C = (E.n + EXPL_T - 1) / EXPL_T;
    return E.n >= EXPL_T && E.n <= 1 << 17 && (E.periodic || C == 1 || (E.n - EXPL_T) / (C - 1) >= 2 * EXPL_R);
}

// Fields of few points leave most of the chip idle, and a pass takes as long
// as the chain of one thread, which is shortest with a point per thread
// (k_explicit): one application along z and y of 32^3 FP64 points takes 2.4
// us there and 3.2 in chunks of 16 rows, of 64^3 3.2 and 3.3, of 80^3 5.7 and
// 3.7; FP32 2.2 and 3.1, 3.1 and 3.2, 3.9 and 3.4.
constexpr long FEW_POINTS = 1 << 18;
// Lines along x: as many per workgroup as make 1024 workgroups, within 256 to
// 2048 points (1 to 8 per thread): 32^3 FP64 2.0 us with 256 points, 4.2 with
// 2048; 64^3 2.6 and 4.5; 128^3 9.1 both.  Long lines without 512 workgroups
// take a thread per point (4096 x 16 FP64 lines 2.3 us against 6.5 in lines,
// 3000 x 256 5.9 and 6.7, 2000 x 512 7.4 and 6.6), and for two applications up
// to 1024 threads (3000 x 256 FP64, the filter twice along each direction,
// 23.3 us, with 256 threads 27.5).
constexpr long LINE_GROUPS = 1024, FEW_LINES = 512;

template <typename TS, int NP>
static bool launch_fast(const ExplicitArgs &E, const ExplicitFields &F, int count, hipStream_t st)
{
    const long pencils = (long)E.na * E.nb * count;  // of all fields
    const unsigned nz = (unsigned)count;
    if (E.dir != 1) {
        if (!chunked(E) || (NP == 1 && pencils * E.n <= FEW_POINTS)) return false;
        const dim3 grid((unsigned)(((long)E.na * E.nb + 255) / 256), (unsigned)((E.n + EXPL_T - 1) / EXPL_T), nz);
        hipLaunchKernelGGL((k_expl_strided<TS, NP>), grid, dim3(256), 0, st, E, F);
        return true;
    }
    const bool few = E.n > 256 && pencils < FEW_LINES;
    if (E.n > 4096 || (NP == 1 && few)) return false;
    // at most 64 KiB of LDS
    const long lo = E.n < 256 ? 256 / E.n : 1, hi = E.n < 2048 ? 2048 / E.n : 1;
    const int lines = (int)std::min(std::max(pencils / LINE_GROUPS, lo), hi);
    const size_t lds = (size_t)lines * E.n * (sizeof(TS) + (NP == 2 ? 8 : 0));
    const unsigned magic = (unsigned)(((unsigned long long)1 << 32) / E.n + 1);
    const dim3 grid((unsigned)(((long)E.na * E.nb + lines - 1) / lines), 1, nz);
    if constexpr (NP == 2) {
        if (few) {
            const dim3 block(std::min((E.n + 63) / 64 * 64, 1024));
            hipLaunchKernelGGL((k_expl_x<TS, NP, 1024>), grid, block, lds, st, E, F, lines, magic);
            return true;
        }
    }
    hipLaunchKernelGGL((k_expl_x<TS, NP, 256>), grid, dim3(256), lds, st, E, F, lines, magic);
    return true;
}

bool explicit_twice(const ExplicitArgs &E) { return E.dir == 1 ? E.n <= 4096 : chunked(E); }

hipError_t launch_explicit(bool dbl, const ExplicitArgs &E, const ExplicitFields &F, int count, hipStream_t st,
                           int times)
{
    const long total = (long)E.n * E.na * E.nb;
    if (total <= 0) return hipSuccess;
    const bool done = times == 2 ? (dbl ? launch_fast<double, 2> : launch_fast<float, 2>)(E, F, count, st)
                                 : (dbl ? launch_fast<double, 1> : launch_fast<float, 1>)(E, F, count, st);
    if (done) return hipGetLastError();
    if (times == 2) return hipErrorInvalidValue;
    long blocks = (total + 255) / 256;
    if (blocks > 1 << 20) blocks = 1 << 20;
    for (int i = 0; i < count; i++) {
        if (dbl)
            hipLaunchKernelGGL((k_explicit<double, double>), dim3((unsigned)blocks), dim3(256), 0, st, E,
                               (const double *)F.f[i], (double *)F.out[i]);
        else
            hipLaunchKernelGGL((k_explicit<float, double>), dim3((unsigned)blocks), dim3(256), 0, st, E,
                               (const float *)F.f[i], (float *)F.out[i]);
    }
    return hipGetLastError();
}

// out = a + s * b (the sums of the operators module)
template <typename T>
__global__ void __launch_bounds__(256) k_axpy(T *out, const T *a, const T *b, double s, long n)
{
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        out[i] = (T)((double)a[i] + s * (double)b[i]);
}

hipError_t launch_axpy(bool dbl, void *out, const void *a, const void *b, double s, long n, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    long blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    if (dbl)
        hipLaunchKernelGGL((k_axpy<double>), dim3((unsigned)blocks), dim3(256), 0, st, (double *)out,
                           (const double *)a, (const double *)b, s, n);
    else
        hipLaunchKernelGGL((k_axpy<float>), dim3((unsigned)blocks), dim3(256), 0, st, (float *)out,
                           (const float *)a, (const float *)b, s, n);
    return hipGetLastError();
}

}  // namespace pdo
