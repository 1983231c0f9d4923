// Two-dimensional transforms of several fields in few passes, for the time
// loop (compute_duidxj, interp_PrimitiveVars, the nonlinear and subgrid
// terms of populate_rhs):
//
//   inverse: a spectrum F gives the field and, on request, its x and y
//     derivatives.  The y pass reads F once and writes the y transforms of F
//     and of i k2 F; the x pass reads those and writes f, df/dx (from
//     i k1 times the first) and df/dy.  8 words per point for the three, where
//     two products by i k and three transforms of their own move 16.  Modes
//     beyond the dealiasing band are zero in the spectra of the loop: their
//     lines are neither transformed nor written nor read.
//   forward: the x pass forms its input, (a1 - b1) c1 + (a2 - b2) c2, from the
//     fields it reads, so the products of the rotational form cost no pass.
//
// A launch takes as many fields as together stay within the 256 MB Infinity
// Cache between its y and its x pass: small grids need two launches for all
// fields (their passes last as long as a launch), large ones two per field.
// All passes are HBM-bound.  Measured, a velocity set and one SSP-RK45 step
// (six preparations, five right-hand sides), together with the one-pass
// pointwise terms of pdo_igrid.hip, before -> after: 512 x 512 x 256 FP32 with
// walls 113.6 -> 79.2 ms, 256^3 FP64 41.2 -> 31.1 ms, 64^3 FP32 3.43 -> 1.58
// ms (762 -> 320 launches).
#include <hip/hip_runtime.h>

#include "pdo_fft_dev.hpp"

namespace pdo {

namespace {

// the task of tile row `r` of a launch and the row within it
template <class B> __device__ __forceinline__ int task_of(const B &b, unsigned &r)
{
    int q = 0;
    while (q < b.count - 1 && r >= b.end[q]) ++q;
    r -= q > 0 ? b.end[q - 1] : 0u;
    return q;
}

// y pass of the inverse transforms: lines kx < kxc of each plane; elements
// from kyc to L - kyc are zero
template <typename TS, typename TC, int L, int TX>
__global__ void __launch_bounds__(1024) k_inv_y(InvBatch bt, int nxh, int kxc, int kyc, const TC *__restrict__ twL,
                                               const double *__restrict__ ky)
{
    extern __shared__ unsigned char smem[];
    constexpr int L8 = L / 8;
    C2<TC> *tile = (C2<TC> *)smem, *twl = tile + TX * L;
    const int ln = threadIdx.x & (TX - 1), jb = threadIdx.x / TX;
    unsigned bx, by;
    xcd_tile(bx, by);
    const InvTask &t = bt.t[task_of(bt, by)];
    const int a = (int)bx * TX + ln;
    const bool act = a < kxc;
    const long off = 2 * ((act ? a : 0) + (long)by * nxh * L);
    using IO = CLoad<TS, TC>;
    const TS *src = (const TS *)t.src + off;
    C2<TC> x[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const int i = jb + r * L8;
        x[r] = C2<TC>{0, 0};
        if (act && (i < kyc || i > L - kyc)) x[r] = IO::ld(src, (long)i * nxh);
    }
    for (int i = threadIdx.x; i < L; i += TX * L8) twl[i] = ((const C2<TC> *)twL)[i];
    __syncthreads();
    constexpr int SLOTS = 256 / (int)sizeof(C2<TC>);
    constexpr int SW = (PDO_FFT_STRIDED_SWZ && SLOTS > TX) ? (SLOTS / TX - 1 < 7 ? SLOTS / TX - 1 : 7) : 0;
    auto buf = [&](int i) -> C2<TC> & { return tile[(i ^ ((i >> 3) & SW)) * TX + ln]; };
    // the first stage's element i = jb + r L/8 is the thread's r-th
    auto ldr = [&](int i) { return x[(i - jb) / L8]; };
    TS *da = (TS *)t.A + off;
    auto sta = [&](int i, C2<TC> v) { IO::st(da, (long)i * nxh, v); };
    line_fft<TC, +1, false, L>(ldr, sta, buf, (const C2<TC> *)twl, jb, act);
    if (!t.B) return;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const TC k = (TC)ky[jb + r * L8];
        x[r] = C2<TC>{-k * x[r].y, k * x[r].x};
    }
    TS *db = (TS *)t.B + off;
    auto stb = [&](int i, C2<TC> v) { IO::st(db, (long)i * nxh, v); };
    line_fft<TC, +1, false, L>(ldr, stb, buf, (const C2<TC> *)twl, jb, act);
}

// x pass: f and fx from A, fy from B; modes kx >= kxc are zero and not read
template <typename TS, typename TC, int L>
__global__ void __launch_bounds__(256) k_inv_x(InvBatch bt, int ny, int nxh, int kxc, const TC *__restrict__ twL,
                                              const TC *__restrict__ twN, const double *__restrict__ kx, int TXL,
                                              TC scale)
{
    extern __shared__ unsigned char smem[];
    C2<TC> *tile = (C2<TC> *)smem;
    const C2<TC> *twl = x_twiddles<TC, L>(tile, TXL, twL);
    const C2<TC> *wN = x_split_twiddles<TC, L>(tile, TXL, twN);
    const TC *kl = x_wavenumbers<TC, L>(tile, TXL, kx);
    constexpr int nx = 2 * L, L8 = L >> 3, LDL = xline_pitch<L>();
    const int line = threadIdx.x / L8, jb = threadIdx.x - line * L8;
    unsigned row = blockIdx.x;
    const InvTask &t = bt.t[task_of(bt, row)];
    const long l = (long)row * TXL + line;
    const bool act = line < TXL && l < (long)t.planes * ny;
    using IO = CLoad<TS, TC>;
    auto buf = [&](int i) -> C2<TC> & { return tile[line * LDL + xslot<L>(i)]; };
    auto ldb = [&](int i) { return buf(i); };
    C2<TC> v[8], vl;
    auto load = [&](const void *p) {
        const TS *src = (const TS *)p + (act ? l : 0) * (long)nxh * 2;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int k = jb + q * L8;
            v[q] = C2<TC>{0, 0};
            if (act && k < kxc) v[q] = IO::ld(src, k);
        }
        vl = C2<TC>{0, 0};
        if (act && jb == 0 && L < kxc) vl = IO::ld(src, L);
    };
    // the modes in v (times i kx with DX), transformed into out
    auto transform = [&](void *out, auto dx) {
        if (act) {
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int k = jb + q * L8;
                if constexpr (dx.value) {
                    const TC kk = kl[k];
                    buf(k) = C2<TC>{-kk * v[q].y, kk * v[q].x};
                } else {
                    buf(k) = v[q];
                }
            }
            if (jb == 0) {
                if constexpr (dx.value) buf(L) = C2<TC>{-kl[L] * vl.y, kl[L] * vl.x};
                else buf(L) = vl;
            }
        }
        __syncthreads();
        if (act) c2r_merge<TC, L>(buf, wN, jb, 0);
        __syncthreads();
        TS *dst = (TS *)out + (act ? l : 0) * (long)nx;
        auto st = [&](int i, C2<TC> x) { IO::st(dst, i, C2<TC>{x.x * scale, x.y * scale}); };
        line_fft<TC, +1, true, L>(ldb, st, buf, twl, jb, act);
    };
    load(t.A);
    __syncthreads();  // the staged tables
    transform(t.f, std::false_type{});
    if (t.fx) {
        __syncthreads();  // every read of the buffer is done
        transform(t.fx, std::true_type{});
    }
    if (t.fy) {
        load(t.B);
        __syncthreads();
        transform(t.fy, std::false_type{});
    }
}

// x pass of the forward transforms of (a1 - b1) c1 + (a2 - b2) c2 (b1 null:
// of a1; a2 null: of the first product)
template <typename TS, typename TC, int L>
__global__ void __launch_bounds__(256) k_fwd_x(FwdBatch bt, int ny, const TC *__restrict__ twL,
                                              const TC *__restrict__ twN, int TXL)
{
    extern __shared__ unsigned char smem[];
    C2<TC> *tile = (C2<TC> *)smem;
    const C2<TC> *twl = x_twiddles<TC, L>(tile, TXL, twL);
    constexpr int nx = 2 * L, L8 = L >> 3, LDL = xline_pitch<L>(), nxh = L + 1;
    const int line = threadIdx.x / L8, jb = threadIdx.x - line * L8;
    unsigned row = blockIdx.x;
    const FwdTask &t = bt.t[task_of(bt, row)];
    const long l = (long)row * TXL + line;
    const bool act = line < TXL && l < (long)t.planes * ny;
    using IO = CLoad<TS, TC>;
    const long o = (act ? l : 0) * (long)nx;
    C2<TC> x[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const int i = jb + r * L8;
        x[r] = IO::ld((const TS *)t.a1 + o, i);
        if (t.b1) {
            const C2<TC> b = IO::ld((const TS *)t.b1 + o, i), c = IO::ld((const TS *)t.c1 + o, i);
            x[r] = C2<TC>{(x[r].x - b.x) * c.x, (x[r].y - b.y) * c.y};
        }
        if (t.a2) {
            const C2<TC> a = IO::ld((const TS *)t.a2 + o, i), b = IO::ld((const TS *)t.b2 + o, i),
                         c = IO::ld((const TS *)t.c2 + o, i);
            x[r].x += (a.x - b.x) * c.x;
            x[r].y += (a.y - b.y) * c.y;
        }
    }
    auto buf = [&](int i) -> C2<TC> & { return tile[line * LDL + xslot<L>(i)]; };
    auto ldr = [&](int i) { return x[(i - jb) / L8]; };
    auto sts = [&](int i, C2<TC> v) { buf(i) = v; };
    line_fft<TC, -1, false, L>(ldr, sts, buf, twl, jb, act);
    __syncthreads();
    const C2<TC> *wN = (const C2<TC> *)twN;
    TS *dst = (TS *)t.spec + (act ? l : 0) * (long)nxh * 2;
    if (act)
        for (int k = jb; k < nxh; k += L8) IO::st(dst, k, r2c_split<TC, L>(buf, wN, k));
}

// y pass of the forward transforms, in place
template <typename TS, typename TC, int L, int TX>
__global__ void __launch_bounds__(1024) k_fwd_y(FwdBatch bt, int nxh, const TC *__restrict__ twL)
{
    extern __shared__ unsigned char smem[];
    C2<TC> *tile = (C2<TC> *)smem, *twl = tile + TX * L;
    const int ln = threadIdx.x & (TX - 1), jb = threadIdx.x / TX;
    unsigned bx, by;
    xcd_tile(bx, by);
    const FwdTask &t = bt.t[task_of(bt, by)];
    const int a = (int)bx * TX + ln;
    const bool act = a < nxh;
    TS *p = (TS *)t.spec + 2 * ((act ? a : 0) + (long)by * nxh * L);
    for (int i = threadIdx.x; i < L; i += TX * (L / 8)) twl[i] = ((const C2<TC> *)twL)[i];
    __syncthreads();
    using IO = CLoad<TS, TC>;
    auto ldg = [&](int i) { return IO::ld(p, (long)i * nxh); };
    auto stg = [&](int i, C2<TC> v) { IO::st(p, (long)i * nxh, v); };
    constexpr int SLOTS = 256 / (int)sizeof(C2<TC>);
    constexpr int SW = (PDO_FFT_STRIDED_SWZ && SLOTS > TX) ? (SLOTS / TX - 1 < 7 ? SLOTS / TX - 1 : 7) : 0;
    auto buf = [&](int i) -> C2<TC> & { return tile[(i ^ ((i >> 3) & SW)) * TX + ln]; };
    line_fft<TC, -1, false, L>(ldg, stg, buf, (const C2<TC> *)twl, jb, act);
}

template <int L, class B> static void x_grid(B &b, int ny, int TXL, unsigned &blocks)
{
    blocks = 0;
    for (int q = 0; q < b.count; ++q) b.end[q] = blocks += (unsigned)(((long)b.t[q].planes * ny + TXL - 1) / TXL);
}

template <class B> static unsigned y_rows(B &b)
{
    unsigned n = 0;
    for (int q = 0; q < b.count; ++q) b.end[q] = n += (unsigned)b.t[q].planes;
    return n;
}

template <int L> static int x_lines(size_t ce)
{
    int TXL = PDO_FFT_X_THREADS / (L / 8);
    while (TXL > 1 && (size_t)TXL * xline_pitch<L>() * ce > 64 * 1024) TXL >>= 1;
    return TXL < 1 ? 1 : TXL;
}

template <typename TS, typename TC, int L>
static void launch_inv_x(const PoissonPlanDev &pl, InvBatch b, int kxc, const double *kx, hipStream_t st)
{
    constexpr size_t ce = 2 * sizeof(TC);
    const Tw<TC> tw(pl);
    const int TXL = x_lines<L>(ce);
    unsigned blocks;
    x_grid<L>(b, pl.ny, TXL, blocks);
    hipLaunchKernelGGL((k_inv_x<TS, TC, L>), dim3(blocks), dim3(TXL * (L / 8)), xline_lds<L>(TXL, ce, true), st, b,
                       pl.ny, pl.nx / 2 + 1, kxc, tw.x, tw.xn, kx, TXL, (TC)(1.0 / ((double)L * pl.ny)));
}

template <typename TS, typename TC, int L>
static void launch_fwd_x(const PoissonPlanDev &pl, FwdBatch b, hipStream_t st)
{
    constexpr size_t ce = 2 * sizeof(TC);
    const Tw<TC> tw(pl);
    const int TXL = x_lines<L>(ce);
    unsigned blocks;
    x_grid<L>(b, pl.ny, TXL, blocks);
    hipLaunchKernelGGL((k_fwd_x<TS, TC, L>), dim3(blocks), dim3(TXL * (L / 8)), xline_lds<L>(TXL, ce), st, b, pl.ny,
                       tw.x, tw.xn, TXL);
}

template <typename TS, typename TC, int L>
static void launch_inv_y(const PoissonPlanDev &pl, InvBatch b, int kxc, int kyc, const double *ky, hipStream_t st)
{
    constexpr size_t ce = 2 * sizeof(TC);
    constexpr int TX = strided_fft_lines<L, ce, 1>();
    const dim3 grid((unsigned)((kxc + TX - 1) / TX), y_rows(b));
    hipLaunchKernelGGL((k_inv_y<TS, TC, L, TX>), grid, dim3(TX * (L / 8)), (size_t)(TX + 1) * L * ce, st, b,
                       pl.nx / 2 + 1, kxc, kyc, Tw<TC>(pl).y, ky);
}

template <typename TS, typename TC, int L>
static void launch_fwd_y(const PoissonPlanDev &pl, FwdBatch b, hipStream_t st)
{
    constexpr size_t ce = 2 * sizeof(TC);
    constexpr int TX = strided_fft_lines<L, ce, 0>();
    const int nxh = pl.nx / 2 + 1;
    const dim3 grid((unsigned)((nxh + TX - 1) / TX), y_rows(b));
    hipLaunchKernelGGL((k_fwd_y<TS, TC, L, TX>), grid, dim3(TX * (L / 8)), (size_t)(TX + 1) * L * ce, st, b, nxh,
                       Tw<TC>(pl).y);
}

#define PDO_X_LENGTHS(L, CALL)                                                                   \
    switch (L) {                                                                                 \
    case 8: CALL(8); break;                                                                      \
    case 16: CALL(16); break;                                                                    \
    case 32: CALL(32); break;                                                                    \
    case 64: CALL(64); break;                                                                    \
    case 128: CALL(128); break;                                                                  \
    case 256: CALL(256); break;                                                                  \
    case 512: CALL(512); break;                                                                  \
    default: return hipErrorInvalidValue;                                                        \
    }
#define PDO_Y_LENGTHS(L, CALL)                                                                   \
    switch (L) {                                                                                 \
    case 1024: CALL(1024); break;                                                                \
    default: PDO_X_LENGTHS(L, CALL)                                                              \
    }

// fields per launch: those whose spectra between the two passes stay within
// half the Infinity Cache (and at least one)
template <class B, class T, class F>
static hipError_t in_groups(const T *t, int count, size_t plane_bytes, F run)
{
    for (int i = 0; i < count;) {
        B b{};
        size_t bytes = 0;
        while (i < count && b.count < MULTI_TASKS) {
            const size_t n = plane_bytes * (size_t)t[i].planes;
            if (b.count > 0 && bytes + n > ((size_t)128 << 20)) break;
            bytes += n;
            b.t[b.count++] = t[i++];
        }
        const hipError_t e = run(b);
        if (e != hipSuccess) return e;
    }
    return hipGetLastError();
}

template <typename TS, typename TC>
static hipError_t inv_multi_t(const PoissonPlanDev &pl, const InvTask *t, int count, const BandLimit &bl,
                              const double *kx, const double *ky, hipStream_t st)
{
    const int nxh = pl.nx / 2 + 1;
    return in_groups<InvBatch>(t, count, (size_t)nxh * pl.ny * 4 * sizeof(TS), [&](const InvBatch &b) -> hipError_t {
#define PDO_CALL(N) launch_inv_y<TS, TC, N>(pl, b, bl.kxc, bl.kyc, ky, st)
        PDO_Y_LENGTHS(pl.ny, PDO_CALL)
#undef PDO_CALL
#define PDO_CALL(N) launch_inv_x<TS, TC, N>(pl, b, bl.kxc, kx, st)
        PDO_X_LENGTHS(pl.nx / 2, PDO_CALL)
#undef PDO_CALL
        return hipSuccess;
    });
}

template <typename TS, typename TC>
static hipError_t fwd_multi_t(const PoissonPlanDev &pl, const FwdTask *t, int count, hipStream_t st)
{
    const int nxh = pl.nx / 2 + 1;
    return in_groups<FwdBatch>(t, count, (size_t)nxh * pl.ny * 2 * sizeof(TS), [&](const FwdBatch &b) -> hipError_t {
#define PDO_CALL(N) launch_fwd_x<TS, TC, N>(pl, b, st)
        PDO_X_LENGTHS(pl.nx / 2, PDO_CALL)
#undef PDO_CALL
#define PDO_CALL(N) launch_fwd_y<TS, TC, N>(pl, b, st)
        PDO_Y_LENGTHS(pl.ny, PDO_CALL)
#undef PDO_CALL
        return hipSuccess;
    });
}

}  // namespace

hipError_t run_inv_multi(const PoissonPlanDev &pl, int mode, const InvTask *t, int count, const BandLimit &bl,
                         const double *kx, const double *ky, hipStream_t st)
{
    switch (mode) {
    case 0: return inv_multi_t<double, double>(pl, t, count, bl, kx, ky, st);
    case 1: return inv_multi_t<float, float>(pl, t, count, bl, kx, ky, st);
    case 2: return inv_multi_t<float, double>(pl, t, count, bl, kx, ky, st);
    }
    return hipErrorInvalidValue;
}

hipError_t run_fwd_multi(const PoissonPlanDev &pl, int mode, const FwdTask *t, int count, hipStream_t st)
{
    switch (mode) {
    case 0: return fwd_multi_t<double, double>(pl, t, count, st);
    case 1: return fwd_multi_t<float, float>(pl, t, count, st);
    case 2: return fwd_multi_t<float, double>(pl, t, count, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace pdo
