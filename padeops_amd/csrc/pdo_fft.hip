// Periodic FFT Poisson solver kernels for gfx950.
//
// A real field f(nx, ny, nz) (x fastest) is transformed in five passes, each
// one HBM read and one HBM write of the half spectrum (nx/2+1, ny, nz):
//   1. x   real-to-complex: nx/2-point complex FFT of the packed line of
//          (even, odd) samples, then the split step to the nx/2+1 modes
//   2. y   complex FFT of every y line
//   3. z   complex FFT, multiply by -1/|k'|^2 (modified wavenumbers), inverse
//          complex FFT -- one pass, the line never leaves LDS
//   4. y   inverse complex FFT
//   5. x   complex-to-real (inverse split + nx/2-point inverse FFT), scaled by
//          1/(nx ny nz)
// Each pass runs a mixed radix-8/4/2 Stockham FFT on a tile of lines: the
// first stage reads its operands straight from HBM, the intermediate stages
// go through LDS, and the last stage writes straight to HBM, so a 512-point
// line costs two LDS round trips.  Every thread holds exactly 8 complex
// values per stage (one radix-8, two radix-4 or four radix-2 butterflies).
// For y and z the tile is TX consecutive lines, so each global row access is
// a contiguous run of TX complex values; twiddles come from a table.
#include <hip/hip_runtime.h>

#include "pdo_fft_dev.hpp"

namespace pdo {

// ---------------------------------------------------------------------------
// passes 2-4: complex FFT of strided lines.  Line (a, b) starts at a + b*sb
// (complex units), element stride se; a in [0, na) is the contiguous index.
// Tile: TX = 1 << lgtx consecutive lines; thread = (line, jb), line fastest.
// MODE 0 forward, 1 inverse, 2 forward -> Poisson multiply -> inverse.
// ---------------------------------------------------------------------------
template <typename TS, typename TC, int MODE, int L, int TX>
__global__ void __launch_bounds__(1024) k_fft_strided(const TS *src, TS *dst, long na, long sb, int se,
                                                     const TC *__restrict__ twL, SpecMul pm)
{
    extern __shared__ unsigned char smem[];
    C2<TC> *tile = (C2<TC> *)smem;
    // TX is a compile-time constant so that the LDS addresses of a thread's
    // elements are one base register plus immediate offsets
    const int ln = threadIdx.x & (TX - 1), jb = threadIdx.x / TX;
    unsigned bx, by;
    xcd_tile(bx, by);
    const long a = (long)bx * TX + ln;
    const bool act = a < na;
    const long off = 2 * ((act ? a : 0) + (long)by * sb);
    if (MODE == 2 && blockIdx.z) src = dst = (TS *)pm.more[blockIdx.z - 1];
    const TS *const lin = src + off;
    TS *const lout = dst + off;
    const C2<TC> *tw = (const C2<TC> *)twL;
    const TC *azl = nullptr;
    if constexpr (PDO_FFT_TW_LDS) {
        // the twiddle table (L values) in LDS after the tile: every stage
        // reads it with broadcast LDS loads instead of vector memory loads;
        // the fused pass also stages its per-element factors az (L values)
        C2<TC> *twl = tile + TX * L;
        for (int i = threadIdx.x; i < L; i += TX * (L / 8)) twl[i] = tw[i];
        if constexpr (MODE == 2) {
            TC *a = (TC *)(twl + L);
            for (int i = threadIdx.x; i < L; i += TX * (L / 8)) a[i] = (TC)pm.az[i];
            azl = a;
        }
        __syncthreads();
        tw = twl;
    }
    using IO = CLoad<TS, TC>;
    auto ldg = [&](int i) { return IO::ld(lin, i * se); };
    auto stg = [&](int i, C2<TC> v) { IO::st(lout, i * se, v); };
    // element i of the line at row i ^ ((i >> 3) & SW): a half-wave spans
    // SW + 1 = 256 B / (TX complex) rows, and the first Stockham stage stores
    // rows 8 j + r, one per value of j in the half-wave; the swizzle sends
    // them to distinct parts of the 256-byte bank row
    constexpr int SLOTS = 256 / (int)sizeof(C2<TC>);
    constexpr int SW = (PDO_FFT_STRIDED_SWZ && SLOTS > TX) ? (SLOTS / TX - 1 < 7 ? SLOTS / TX - 1 : 7) : 0;
    auto buf = [&](int i) -> C2<TC> & { return tile[(i ^ ((i >> 3) & SW)) * TX + ln]; };
    if constexpr (MODE == 0) {
        line_fft<TC, -1, false, L>(ldg, stg, buf, tw, jb, act);
    } else if constexpr (MODE == 1) {
        line_fft<TC, +1, false, L>(ldg, stg, buf, tw, jb, act);
    } else {
        // forward into LDS, multiply by the spectral factor of (kx, ky, kz) =
        // (a, by, i), inverse from LDS to HBM
        // the factor is formed in the arithmetic of the transform (an FP64
        // division per point costs as much as the transforms in FP32)
        const int kx = (int)a, ky = (int)by;
        const bool line_only = pm.kind == 3 || pm.kind == 4;  // factors of the line index alone
        const TC fxy = (act && !line_only)
                           ? (TC)(pm.kind == 5 ? pm.ax[kx] : pm.kind == 2 ? pm.ax[kx] * pm.ay[ky] : pm.ax[kx] + pm.ay[ky])
                           : TC(0);
        const TC scale = (TC)pm.scale;
        auto sts = [&](int i, C2<TC> v) {
            TC fac;
            const TC az = PDO_FFT_TW_LDS ? azl[i] : (TC)pm.az[i];
            if (pm.kind == 3) {
                // i az: (x + i y) i a = -a y + i a x
                const TC s = az * scale;
                buf(i) = C2<TC>{-s * v.y, s * v.x};
                return;
            }
            if (pm.kind == 4) {
                fac = az;
            } else if (pm.kind == 2 || pm.kind == 5) {
                fac = fxy * az;
            } else {
                const TC ks = fxy + az;
                if (pm.kind == 0) fac = (kx == 0 && ky == 0 && i == 0) ? TC(0) : -recip(ks + TC(1.0e-20));
                else fac = (ks <= TC(1.0e-14)) ? TC(0) : -recip(ks);
            }
            fac *= scale;
            v.x *= fac;
            v.y *= fac;
            buf(i) = v;
        };
        line_fft<TC, -1, false, L>(ldg, sts, buf, tw, jb, act);
        __syncthreads();
        auto ldb = [&](int i) { return buf(i); };
        line_fft<TC, +1, true, L>(ldb, stg, buf, tw, jb, act);
    }
}

// ---------------------------------------------------------------------------
// pass 1: x real-to-complex.  nlines lines of nx reals -> nx/2+1 complex.
// Tile: TXL lines; thread = (line, jb), jb fastest.
// ---------------------------------------------------------------------------
template <typename TS, typename TC, int L>
__global__ void __launch_bounds__(1024) k_fft_x_r2c(const TS *__restrict__ in, TS *__restrict__ out, long nlines,
                                                   const TC *__restrict__ twL, const TC *__restrict__ twN, int TXL,
                                                   int nxp)
{
    extern __shared__ unsigned char smem[];
    C2<TC> *tile = (C2<TC> *)smem;
    const C2<TC> *twl = x_twiddles<TC, L>(tile, TXL, twL);
    constexpr int nx = 2 * L, L8 = L >> 3, LDL = xline_pitch<L>(), nxh = L + 1;
    const int line = threadIdx.x / L8, jb = threadIdx.x - line * L8;
    const long l = (long)blockIdx.x * TXL + line;
    const bool act = (line < TXL) && (l < nlines);
    using IO = CLoad<TS, TC>;
    const TS *src = in + (act ? l : 0) * (long)nx;
    auto ldg = [&](int i) { return IO::ld(src, i); };  // packed z_j = (x_2j, x_2j+1)
    auto buf = [&](int i) -> C2<TC> & { return tile[line * LDL + xslot<L>(i)]; };
    auto sts = [&](int i, C2<TC> v) { buf(i) = v; };
    line_fft<TC, -1, false, L>(ldg, sts, buf, twl, jb, act);
    __syncthreads();
    const C2<TC> *wN = (const C2<TC> *)twN;
    TS *dst = out + (act ? l : 0) * (long)nxp * 2;
    if (act) {
        for (int k = jb; k < nxh; k += L8) IO::st(dst, k, r2c_split<TC, L>(buf, wN, k));
    }
}

// pass 5: x complex-to-real, scaled by `scale`.  Like a Hermitian c2r, only
// the real parts of the kx = 0 and kx = nx/2 modes enter; with oddball != 0
// the kx = nx/2 mode is dropped altogether.
template <typename TS, typename TC, int L>
__global__ void __launch_bounds__(1024) k_fft_x_c2r(const TS *__restrict__ in, TS *__restrict__ out, long nlines,
                                                   const TC *__restrict__ twL, const TC *__restrict__ twN, int TXL,
                                                   TC scale, int nxp, int oddball)
{
    extern __shared__ unsigned char smem[];
    C2<TC> *tile = (C2<TC> *)smem;
    const C2<TC> *twl = x_twiddles<TC, L>(tile, TXL, twL);
    constexpr int nx = 2 * L, L8 = L >> 3, LDL = xline_pitch<L>();
    const int line = threadIdx.x / L8, jb = threadIdx.x - line * L8;
    const long l = (long)blockIdx.x * TXL + line;
    const bool act = (line < TXL) && (l < nlines);
    using IO = CLoad<TS, TC>;
    const TS *src = in + (act ? l : 0) * (long)nxp * 2;
    auto buf = [&](int i) -> C2<TC> & { return tile[line * LDL + xslot<L>(i)]; };
    const C2<TC> *wN = (const C2<TC> *)twN;
    // stage the nx/2+1 modes of the line in LDS (coalesced, all loads of a
    // thread in flight together), then form Z_k = E_k + i O_k in place, one
    // thread per pair (k, L-k):
    // E = (X_k + conj X_{L-k})/2, O = (X_k - conj X_{L-k}) conj(W^k)/2
    if (act) {
        C2<TC> v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = IO::ld(src, jb + q * L8);
        C2<TC> vl = {};
        if (jb == 0) vl = IO::ld(src, L);
#pragma unroll
        for (int q = 0; q < 8; ++q) buf(jb + q * L8) = v[q];
        if (jb == 0) buf(L) = vl;
    }
    __syncthreads();
    if (act) c2r_merge<TC, L>(buf, wN, jb, oddball);
    __syncthreads();
    TS *dst = out + (act ? l : 0) * (long)nx;
    auto ldb = [&](int i) { return buf(i); };
    auto stg = [&](int i, C2<TC> v) {
        v.x *= scale;
        v.y *= scale;
        IO::st(dst, i, v);
    };
    line_fft<TC, +1, true, L>(ldb, stg, buf, twl, jb, act);
}

// The x transforms of the full-RHS Poisson solve with the x derivatives of
// its divergence and of its projection taken in spectral space.  On a
// periodic grid the cd06 first derivative is diagonal in Fourier space, with
// eigenvalue i k'(kx) on mode kx (k' the modified wavenumber, zero at kx = 0
// and kx = nx/2), so these passes form the same operators as a compact x
// solve, without the extra pass over HBM.
//
// r2c: X = FFT_x(div) + i k'(kx) FFT_x(ut), line by line.
template <typename TS, typename TC, int L>
__global__ void __launch_bounds__(1024) k_fft_x_r2c_dx(const TS *__restrict__ div, const TS *__restrict__ ut,
                                                      TS *__restrict__ out, long nlines, const TC *__restrict__ twL,
                                                      const TC *__restrict__ twN, int TXL, int nxp,
                                                      const double *__restrict__ kp)
{
    extern __shared__ unsigned char smem[];
    C2<TC> *tile = (C2<TC> *)smem;
    const C2<TC> *twl = x_twiddles<TC, L>(tile, TXL, twL);
    constexpr int nx = 2 * L, L8 = L >> 3, LDL = xline_pitch<L>(), nxh = L + 1;
    constexpr int NK = (nxh + L8 - 1) / L8;  // modes per thread
    const int line = threadIdx.x / L8, jb = threadIdx.x - line * L8;
    const long l = (long)blockIdx.x * TXL + line;
    const bool act = (line < TXL) && (l < nlines);
    using IO = CLoad<TS, TC>;
    auto buf = [&](int i) -> C2<TC> & { return tile[line * LDL + xslot<L>(i)]; };
    auto sts = [&](int i, C2<TC> v) { buf(i) = v; };
    const C2<TC> *wN = x_split_twiddles<TC, L>(tile, TXL, twN);
    const TC *kl = x_wavenumbers<TC, L>(tile, TXL, kp);
    auto kpr = [&](int k) { return PDO_FFT_X_TW_LDS ? kl[k] : (TC)kp[k]; };
    // i k' FFT(ut), held in registers
    C2<TC> du[NK];
    {
        const TS *src = ut + (act ? l : 0) * (long)nx;
        auto ldg = [&](int i) { return IO::ld(src, i); };
        line_fft<TC, -1, false, L>(ldg, sts, buf, twl, jb, act);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < NK; ++q) {
            const int k = jb + q * L8;
            du[q] = C2<TC>{0, 0};
            if (act && k < nxh) {
                const C2<TC> x = r2c_split<TC, L>(buf, wN, k);
                const TC kk = kpr(k);
                du[q] = C2<TC>{-kk * x.y, kk * x.x};
            }
        }
        __syncthreads();  // every read of the buffer is done
    }
    const TS *src = div + (act ? l : 0) * (long)nx;
    auto ldg = [&](int i) { return IO::ld(src, i); };
    line_fft<TC, -1, false, L>(ldg, sts, buf, twl, jb, act);
    __syncthreads();
    TS *dst = out + (act ? l : 0) * (long)nxp * 2;
    if (act) {
#pragma unroll
        for (int q = 0; q < NK; ++q) {
            const int k = jb + q * L8;
            if (k < nxh) IO::st(dst, k, cadd(r2c_split<TC, L>(buf, wN, k), du[q]));
        }
    }
}

// c2r: p = scale IFFT_x(P) and u = ut - scale IFFT_x(i k'(kx) P), line by line.
template <typename TS, typename TC, int L>
__global__ void __launch_bounds__(1024) k_fft_x_c2r_dx(const TS *__restrict__ in, TS *__restrict__ p,
                                                      const TS *__restrict__ ut, TS *__restrict__ u, long nlines,
                                                      const TC *__restrict__ twL, const TC *__restrict__ twN, int TXL,
                                                      TC scale, int nxp, const double *__restrict__ kp)
{
    extern __shared__ unsigned char smem[];
    C2<TC> *tile = (C2<TC> *)smem;
    const C2<TC> *twl = x_twiddles<TC, L>(tile, TXL, twL);
    constexpr int nx = 2 * L, L8 = L >> 3, LDL = xline_pitch<L>();
    const int line = threadIdx.x / L8, jb = threadIdx.x - line * L8;
    const long l = (long)blockIdx.x * TXL + line;
    const bool act = (line < TXL) && (l < nlines);
    using IO = CLoad<TS, TC>;
    const TS *src = in + (act ? l : 0) * (long)nxp * 2;
    auto buf = [&](int i) -> C2<TC> & { return tile[line * LDL + xslot<L>(i)]; };
    auto ldb = [&](int i) { return buf(i); };
    const C2<TC> *wN = x_split_twiddles<TC, L>(tile, TXL, twN);
    const TC *kl = x_wavenumbers<TC, L>(tile, TXL, kp);
    auto kpr = [&](int k) { return PDO_FFT_X_TW_LDS ? kl[k] : (TC)kp[k]; };
    C2<TC> v[8];
    C2<TC> vl = {};
    if (act) {
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = IO::ld(src, jb + q * L8);
        if (jb == 0) vl = IO::ld(src, L);
#pragma unroll
        for (int q = 0; q < 8; ++q) buf(jb + q * L8) = v[q];
        if (jb == 0) buf(L) = vl;
    }
    __syncthreads();
    if (act) c2r_merge<TC, L>(buf, wN, jb, 0);
    __syncthreads();
    TS *pl = p + (act ? l : 0) * (long)nx;
    auto stp = [&](int i, C2<TC> x) {
        x.x *= scale;
        x.y *= scale;
        IO::st(pl, i, x);
    };
    line_fft<TC, +1, true, L>(ldb, stp, buf, twl, jb, act);
    __syncthreads();  // every read of the buffer by the first transform is done
    // i k' P, from the modes still in registers
    if (act) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const TC kk = kpr(jb + q * L8);
            buf(jb + q * L8) = C2<TC>{-kk * v[q].y, kk * v[q].x};
        }
        if (jb == 0) {
            const TC kk = kpr(L);
            buf(L) = C2<TC>{-kk * vl.y, kk * vl.x};
        }
    }
    __syncthreads();
    if (act) c2r_merge<TC, L>(buf, wN, jb, 0);
    __syncthreads();
    const TS *ul = ut + (act ? l : 0) * (long)nx;
    TS *uo = u + (act ? l : 0) * (long)nx;
    auto stu = [&](int i, C2<TC> x) {
        const C2<TC> a = IO::ld(ul, i);
        IO::st(uo, i, C2<TC>{a.x - scale * x.x, a.y - scale * x.y});
    };
    line_fft<TC, +1, true, L>(ldb, stu, buf, twl, jb, act);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static int ilog2(int v)
{
    int l = 0;
    while ((1 << l) < v) l++;
    return l;
}

template <typename TS, typename TC, int MODE, int L>
static void launch_strided_fft(const TS *src, TS *dst, long na, long sb, long se, const TC *tw, const SpecMul &pm,
                               int nb, hipStream_t st)
{
    constexpr size_t ce = 2 * sizeof(TC);
    constexpr int TX = strided_fft_lines<L, ce, MODE>();
    dim3 grid((unsigned)((na + TX - 1) / TX), (unsigned)nb, MODE == 2 ? (unsigned)pm.fields : 1u);
    hipLaunchKernelGGL((k_fft_strided<TS, TC, MODE, L, TX>), grid, dim3(TX * (L / 8)),
                       (size_t)(TX + (PDO_FFT_TW_LDS ? 1 : 0)) * L * ce +
                           ((PDO_FFT_TW_LDS && MODE == 2) ? (size_t)L * sizeof(TC) : 0),
                       st, src,
                       dst, na, sb, (int)se, tw, pm);
}

template <typename TS, typename TC, int MODE>
static void strided_fft(int L, const TS *src, TS *dst, long na, long sb, long se, const TC *tw, const SpecMul &pm,
                        int nb, hipStream_t st)
{
    switch (L) {
    case 8: launch_strided_fft<TS, TC, MODE, 8>(src, dst, na, sb, se, tw, pm, nb, st); break;
    case 16: launch_strided_fft<TS, TC, MODE, 16>(src, dst, na, sb, se, tw, pm, nb, st); break;
    case 32: launch_strided_fft<TS, TC, MODE, 32>(src, dst, na, sb, se, tw, pm, nb, st); break;
    case 64: launch_strided_fft<TS, TC, MODE, 64>(src, dst, na, sb, se, tw, pm, nb, st); break;
    case 128: launch_strided_fft<TS, TC, MODE, 128>(src, dst, na, sb, se, tw, pm, nb, st); break;
    case 256: launch_strided_fft<TS, TC, MODE, 256>(src, dst, na, sb, se, tw, pm, nb, st); break;
    case 512: launch_strided_fft<TS, TC, MODE, 512>(src, dst, na, sb, se, tw, pm, nb, st); break;
    case 1024: launch_strided_fft<TS, TC, MODE, 1024>(src, dst, na, sb, se, tw, pm, nb, st); break;
    }
}

template <typename TS, typename TC, int L>
static void launch_x_fft(bool inverse, const TS *in, TS *out, long nlines, const TC *tw, const TC *twn, TC scale,
                         int nxp, int oddball, hipStream_t st)
{
    const size_t ce = 2 * sizeof(TC);
    int TXL = PDO_FFT_X_THREADS / (L / 8);
    if (TXL < 1) TXL = 1;
    while (TXL > 1 && (size_t)TXL * xline_pitch<L>() * ce > 64 * 1024) TXL >>= 1;
    dim3 grid((unsigned)((nlines + TXL - 1) / TXL));
    if (!inverse)
        hipLaunchKernelGGL((k_fft_x_r2c<TS, TC, L>), grid, dim3(TXL * (L / 8)), xline_lds<L>(TXL, ce), st, in,
                           out, nlines, tw, twn, TXL, nxp);
    else
        hipLaunchKernelGGL((k_fft_x_c2r<TS, TC, L>), grid, dim3(TXL * (L / 8)), xline_lds<L>(TXL, ce), st, in,
                           out, nlines, tw, twn, TXL, scale, nxp, oddball);
}

template <typename TS, typename TC>
static void x_fft(int L, bool inverse, const TS *in, TS *out, long nlines, const TC *tw, const TC *twn, TC scale,
                  int nxp, int oddball, hipStream_t st)
{
    switch (L) {
    case 8: launch_x_fft<TS, TC, 8>(inverse, in, out, nlines, tw, twn, scale, nxp, oddball, st); break;
    case 16: launch_x_fft<TS, TC, 16>(inverse, in, out, nlines, tw, twn, scale, nxp, oddball, st); break;
    case 32: launch_x_fft<TS, TC, 32>(inverse, in, out, nlines, tw, twn, scale, nxp, oddball, st); break;
    case 64: launch_x_fft<TS, TC, 64>(inverse, in, out, nlines, tw, twn, scale, nxp, oddball, st); break;
    case 128: launch_x_fft<TS, TC, 128>(inverse, in, out, nlines, tw, twn, scale, nxp, oddball, st); break;
    case 256: launch_x_fft<TS, TC, 256>(inverse, in, out, nlines, tw, twn, scale, nxp, oddball, st); break;
    case 512: launch_x_fft<TS, TC, 512>(inverse, in, out, nlines, tw, twn, scale, nxp, oddball, st); break;
    }
}

// the x passes with the spectral x derivative (k_fft_x_r2c_dx / _c2r_dx)
template <typename TS, typename TC, int L>
static void launch_x_fft_dx(bool inverse, const TS *a, const TS *b, TS *o1, TS *o2, long nlines, const TC *tw,
                            const TC *twn, TC scale, int nxp, const double *kp, hipStream_t st)
{
    const size_t ce = 2 * sizeof(TC);
    int TXL = PDO_FFT_X_THREADS / (L / 8);
    if (TXL < 1) TXL = 1;
    while (TXL > 1 && (size_t)TXL * xline_pitch<L>() * ce > 64 * 1024) TXL >>= 1;
    dim3 grid((unsigned)((nlines + TXL - 1) / TXL));
    if (!inverse)
        hipLaunchKernelGGL((k_fft_x_r2c_dx<TS, TC, L>), grid, dim3(TXL * (L / 8)), xline_lds<L>(TXL, ce, true), st, a,
                           b, o1, nlines, tw, twn, TXL, nxp, kp);
    else
        hipLaunchKernelGGL((k_fft_x_c2r_dx<TS, TC, L>), grid, dim3(TXL * (L / 8)), xline_lds<L>(TXL, ce, true), st, a,
                           o1, b, o2, nlines, tw, twn, TXL, scale, nxp, kp);
}

template <typename TS, typename TC>
static void x_fft_dx(int L, bool inverse, const TS *a, const TS *b, TS *o1, TS *o2, long nlines, const TC *tw,
                     const TC *twn, TC scale, int nxp, const double *kp, hipStream_t st)
{
    switch (L) {
    case 8: launch_x_fft_dx<TS, TC, 8>(inverse, a, b, o1, o2, nlines, tw, twn, scale, nxp, kp, st); break;
    case 16: launch_x_fft_dx<TS, TC, 16>(inverse, a, b, o1, o2, nlines, tw, twn, scale, nxp, kp, st); break;
    case 32: launch_x_fft_dx<TS, TC, 32>(inverse, a, b, o1, o2, nlines, tw, twn, scale, nxp, kp, st); break;
    case 64: launch_x_fft_dx<TS, TC, 64>(inverse, a, b, o1, o2, nlines, tw, twn, scale, nxp, kp, st); break;
    case 128: launch_x_fft_dx<TS, TC, 128>(inverse, a, b, o1, o2, nlines, tw, twn, scale, nxp, kp, st); break;
    case 256: launch_x_fft_dx<TS, TC, 256>(inverse, a, b, o1, o2, nlines, tw, twn, scale, nxp, kp, st); break;
    case 512: launch_x_fft_dx<TS, TC, 512>(inverse, a, b, o1, o2, nlines, tw, twn, scale, nxp, kp, st); break;
    }
}

template <typename TS, typename TC>
static hipError_t run_poisson_t(const PoissonPlanDev &pl, const TS *rhs, TS *f, TS *spec, hipStream_t st)
{
    const int nx = pl.nx, ny = pl.ny, nz = pl.nz, nxh = nx / 2 + 1, L = nx / 2;
    const Tw<TC> tw(pl);
    const SpecMul pm{pl.kx2, pl.ky2, pl.kz2, pl.zero_policy, 1.0};
    const long nlines = (long)ny * nz;
    const TC scale = (TC)(1.0 / ((double)L * ny * nz));
    // half spectrum (nxh, ny, nz) stored with row pitch nxp (a multiple of 16
    // complex values) so every tile row starts on a 128-byte boundary
    const int nxp = pl.nxp;
    x_fft<TS, TC>(L, false, rhs, spec, nlines, tw.x, tw.xn, scale, nxp, 0, st);
    strided_fft<TS, TC, 0>(ny, spec, spec, (long)nxh, (long)nxp * ny, (long)nxp, tw.y, pm, nz, st);
    strided_fft<TS, TC, 2>(nz, spec, spec, (long)nxh, (long)nxp, (long)nxp * ny, tw.z, pm, ny, st);
    strided_fft<TS, TC, 1>(ny, spec, spec, (long)nxh, (long)nxp * ny, (long)nxp, tw.y, pm, nz, st);
    x_fft<TS, TC>(L, true, spec, f, nlines, tw.x, tw.xn, scale, nxp, 0, st);
    return hipGetLastError();
}

template <typename TS, typename TC>
static hipError_t run_poisson_dx_t(const PoissonPlanDev &pl, const TS *div, const TS *ut, TS *p, TS *ux, TS *spec,
                                   const double *kp, hipStream_t st)
{
    const int nx = pl.nx, ny = pl.ny, nz = pl.nz, nxh = nx / 2 + 1, L = nx / 2;
    const Tw<TC> tw(pl);
    const SpecMul pm{pl.kx2, pl.ky2, pl.kz2, pl.zero_policy, 1.0};
    const long nlines = (long)ny * nz;
    const TC scale = (TC)(1.0 / ((double)L * ny * nz));
    const int nxp = pl.nxp;
    x_fft_dx<TS, TC>(L, false, div, ut, spec, nullptr, nlines, tw.x, tw.xn, (TC)1, nxp, kp, st);
    strided_fft<TS, TC, 0>(ny, spec, spec, (long)nxh, (long)nxp * ny, (long)nxp, tw.y, pm, nz, st);
    strided_fft<TS, TC, 2>(nz, spec, spec, (long)nxh, (long)nxp, (long)nxp * ny, tw.z, pm, ny, st);
    strided_fft<TS, TC, 1>(ny, spec, spec, (long)nxh, (long)nxp * ny, (long)nxp, tw.y, pm, nz, st);
    x_fft_dx<TS, TC>(L, true, spec, ut, p, ux, nlines, tw.x, tw.xn, scale, nxp, kp, st);
    return hipGetLastError();
}

hipError_t run_poisson_dx(const PoissonPlanDev &pl, int mode, const void *div, const void *ut, void *p, void *ux,
                          void *spec, const double *kp, hipStream_t st)
{
    switch (mode) {
    case 0:
        return run_poisson_dx_t<double, double>(pl, (const double *)div, (const double *)ut, (double *)p,
                                                (double *)ux, (double *)spec, kp, st);
    case 1:
        return run_poisson_dx_t<float, float>(pl, (const float *)div, (const float *)ut, (float *)p, (float *)ux,
                                              (float *)spec, kp, st);
    case 2:
        return run_poisson_dx_t<float, double>(pl, (const float *)div, (const float *)ut, (float *)p, (float *)ux,
                                               (float *)spec, kp, st);
    }
    return hipErrorInvalidValue;
}

hipError_t run_poisson(const PoissonPlanDev &pl, int mode, const void *rhs, void *f, void *spec, hipStream_t st)
{
    switch (mode) {
    case 0: return run_poisson_t<double, double>(pl, (const double *)rhs, (double *)f, (double *)spec, st);
    case 1: return run_poisson_t<float, float>(pl, (const float *)rhs, (float *)f, (float *)spec, st);
    case 2: return run_poisson_t<float, double>(pl, (const float *)rhs, (float *)f, (float *)spec, st);
    }
    return hipErrorInvalidValue;
}

// 2D transforms of the (x, y) planes of (nx, ny, nplanes) data; the half
// spectrum is (nx/2+1, ny, nplanes) without padding.
template <typename TS, typename TC>
static hipError_t run_fft2_t(const PoissonPlanDev &pl, const TS *in, TS *out, int nplanes, hipStream_t st)
{
    const int nx = pl.nx, ny = pl.ny, nxh = nx / 2 + 1, L = nx / 2;
    const Tw<TC> tw(pl);
    const SpecMul pm{};
    x_fft<TS, TC>(L, false, in, out, (long)ny * nplanes, tw.x, tw.xn, (TC)1, nxh, 0, st);
    strided_fft<TS, TC, 0>(ny, out, out, (long)nxh, (long)nxh * ny, (long)nxh, tw.y, pm, nplanes, st);
    return hipGetLastError();
}

// 2D spectral filtering of real (nx, ny, nplanes) data by the separable
// factor t1(kx) t2(ky) (host-side 0/1 cutoffs, device arrays of nx/2+1 and
// ny): the x r2c pass into spec, then one fused pass per y line (forward
// transform, the factor, inverse transform, in place), then the x c2r pass
// into out.  Two passes fewer than fft2, a pointwise multiply and ifft2.
template <typename TS, typename TC>
static hipError_t run_filter2_t(const PoissonPlanDev &pl, const TS *in, TS *spec, TS *out, int nplanes,
                                const double *t1, const double *t2, hipStream_t st)
{
    const int nx = pl.nx, ny = pl.ny, nxh = nx / 2 + 1, L = nx / 2;
    const Tw<TC> tw(pl);
    x_fft<TS, TC>(L, false, in, spec, (long)ny * nplanes, tw.x, tw.xn, (TC)1, nxh, 0, st);
    // kind 5: factor t1[kx] t2[ky] of the line (kx) and element (ky) indices
    const SpecMul pm{t1, nullptr, t2, 5, 1.0};
    strided_fft<TS, TC, 2>(ny, spec, spec, (long)nxh, (long)nxh * ny, (long)nxh, tw.y, pm, nplanes, st);
    const TC scale = (TC)(1.0 / ((double)L * ny));
    x_fft<TS, TC>(L, true, spec, out, (long)ny * nplanes, tw.x, tw.xn, scale, nxh, 0, st);
    return hipGetLastError();
}

hipError_t run_filter2(const PoissonPlanDev &pl, int mode, const void *in, void *spec, void *out, int nplanes,
                       const double *t1, const double *t2, hipStream_t st)
{
    switch (mode) {
    case 0: return run_filter2_t<double, double>(pl, (const double *)in, (double *)spec, (double *)out, nplanes, t1, t2, st);
    case 1: return run_filter2_t<float, float>(pl, (const float *)in, (float *)spec, (float *)out, nplanes, t1, t2, st);
    case 2: return run_filter2_t<float, double>(pl, (const float *)in, (float *)spec, (float *)out, nplanes, t1, t2, st);
    }
    return hipErrorInvalidValue;
}

template <typename TS, typename TC>
static hipError_t run_ifft2_t(const PoissonPlanDev &pl, const TS *in, TS *work, TS *out, int nplanes, int oddball,
                              hipStream_t st)
{
    const int nx = pl.nx, ny = pl.ny, nxh = nx / 2 + 1, L = nx / 2;
    const Tw<TC> tw(pl);
    const SpecMul pm{};
    // the c2r pass returns L times the inverse transform: scale to 1/(nx ny)
    const TC scale = (TC)(1.0 / ((double)L * ny));
    strided_fft<TS, TC, 1>(ny, in, work, (long)nxh, (long)nxh * ny, (long)nxh, tw.y, pm, nplanes, st);
    x_fft<TS, TC>(L, true, work, out, (long)ny * nplanes, tw.x, tw.xn, scale, nxh, oddball, st);
    return hipGetLastError();
}

// forward z transform -> multiply -> inverse z transform of (nxh, ny, nz) complex data
template <typename TS, typename TC>
static hipError_t run_zmul_t(const PoissonPlanDev &pl, const TS *in, TS *out, const SpecMul &m, hipStream_t st,
                             int lines)
{
    const int ny = pl.ny, nz = pl.nz, nxh = pl.nx / 2 + 1;
    const Tw<TC> tw(pl);
    strided_fft<TS, TC, 2>(nz, in, out, (long)(lines > 0 ? lines : nxh), (long)nxh, (long)nxh * ny, tw.z, m, ny, st);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// PadePoisson with walls in z (PadePoisson.F90:472-603), one workgroup per TX
// (kx) lines of a ky: the 2 nz-point even extension of f (cells, nz points:
// nz-1 .. 0, 0 .. nz-1) and odd extension of w (edges, nz+1 points:
// -w[nz-1] .. -w[1], w[0] .. w[nz]) are transformed in LDS, then
//   P = -(F + i kcm W) / |k|^2   (|k|^2 = ax[kx] + ay[ky] + az[kz], <= 1e-14: 0)
//   W = W - i kcp P
// with kcm, kcp = k3' exp(-+ i k3 dz / 2), both are transformed back (scale
// 1 / L), f takes the second half of P and w points nz-1 .. L-1 of W, zero on
// the two walls.  f and w are updated in place.  UPD false (getPressure,
// :834-871): only P goes back to f, w is read only.
// ---------------------------------------------------------------------------
template <typename TS, typename TC, int L, int TX, bool UPD>
__global__ void __launch_bounds__(1024) k_pp_walls(TS *f, TS *w, long na, long sb, int se, const TC *__restrict__ twL,
                                                  const double *__restrict__ ax, const double *__restrict__ ay,
                                                  const double *__restrict__ az, const double *__restrict__ kcm,
                                                  const double *__restrict__ kcp)
{
    extern __shared__ unsigned char smem[];
    constexpr int H = L / 2;
    C2<TC> *tF = (C2<TC> *)smem;
    C2<TC> *tW = tF + TX * L;
    C2<TC> *twl = tW + TX * L;
    const int ln = threadIdx.x & (TX - 1), jb = threadIdx.x / TX;
    unsigned bx, by;
    xcd_tile(bx, by);
    const long a = (long)bx * TX + ln;
    const bool act = a < na;
    const long off = 2 * ((act ? a : 0) + (long)by * sb);
    TS *const lf = f + off;
    TS *const lw = w + off;
    for (int i = threadIdx.x; i < L; i += TX * (L / 8)) twl[i] = ((const C2<TC> *)twL)[i];
    __syncthreads();
    using IO = CLoad<TS, TC>;
    constexpr int SLOTS = 256 / (int)sizeof(C2<TC>);
    constexpr int SW = (PDO_FFT_STRIDED_SWZ && SLOTS > TX) ? (SLOTS / TX - 1 < 7 ? SLOTS / TX - 1 : 7) : 0;
    auto bufF = [&](int i) -> C2<TC> & { return tF[(i ^ ((i >> 3) & SW)) * TX + ln]; };
    auto bufW = [&](int i) -> C2<TC> & { return tW[(i ^ ((i >> 3) & SW)) * TX + ln]; };
    // forward transforms of the extensions into LDS
    auto ldF = [&](int i) { return IO::ld(lf, (i < H ? H - 1 - i : i - H) * se); };
    auto ldW = [&](int i) {
        if (i < H - 1) {
            const C2<TC> v = IO::ld(lw, (H - 1 - i) * se);
            return C2<TC>{-v.x, -v.y};
        }
        return IO::ld(lw, (i - (H - 1)) * se);
    };
    auto stF = [&](int i, C2<TC> v) { bufF(i) = v; };
    auto stW = [&](int i, C2<TC> v) { bufW(i) = v; };
    line_fft<TC, -1, false, L>(ldF, stF, bufF, (const C2<TC> *)twl, jb, act);
    __syncthreads();
    line_fft<TC, -1, false, L>(ldW, stW, bufW, (const C2<TC> *)twl, jb, act);
    __syncthreads();
    // the pressure and the w update, 8 modes per thread
    if (act) {
        const TC fxy = (TC)(ax[a] + ay[by]);
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const int i = jb * 8 + r;
            const C2<TC> F = bufF(i), W = bufW(i);
            const TC ks = fxy + (TC)az[i];
            const TC kinv = (ks <= TC(1.0e-14)) ? TC(0) : recip(ks);
            // P = -(F + i cm W) kinv
            const C2<TC> cw = cmul(C2<TC>{(TC)kcm[2 * i], (TC)kcm[2 * i + 1]}, W);
            const C2<TC> Pv{-(F.x - cw.y) * kinv, -(F.y + cw.x) * kinv};
            // W -= i cp P
            bufF(i) = Pv;
            if constexpr (UPD) {
                const C2<TC> cpp = cmul(C2<TC>{(TC)kcp[2 * i], (TC)kcp[2 * i + 1]}, Pv);
                bufW(i) = C2<TC>{W.x + cpp.y, W.y - cpp.x};
            }
        }
    }
    __syncthreads();
    const TC scale = TC(1) / TC(L);
    auto lbF = [&](int i) { return bufF(i); };
    auto lbW = [&](int i) { return bufW(i); };
    auto sgF = [&](int i, C2<TC> v) {
        if (i >= H) IO::st(lf, (i - H) * se, C2<TC>{v.x * scale, v.y * scale});
    };
    auto sgW = [&](int i, C2<TC> v) {
        if (i >= H - 1) {
            const int k = i - (H - 1);
            const bool wall = (k == 0 || k == H);
            IO::st(lw, k * se, wall ? C2<TC>{TC(0), TC(0)} : C2<TC>{v.x * scale, v.y * scale});
        }
    };
    line_fft<TC, +1, true, L>(lbF, sgF, bufF, (const C2<TC> *)twl, jb, act);
    if constexpr (UPD) {
        __syncthreads();
        line_fft<TC, +1, true, L>(lbW, sgW, bufW, (const C2<TC> *)twl, jb, act);
    }
}

// lines per workgroup of the wall projection: two line tiles and the twiddles
// in at most `kib` KiB, 8 points per thread; above 256 threads only for rows
// of up to 64 bytes (VAL: bytes of a stored value)
template <int L, size_t CE, size_t VAL, size_t KIB> constexpr int pp_walls_lines()
{
    int tx = 512 / (L / 8);
    if (tx < 1) tx = 1;
    while (tx > 1 && ((2 * (size_t)tx + 1) * L * CE > KIB * 1024 || (tx * (L / 8) > 256 && tx * VAL > 64))) tx >>= 1;
    return tx;
}

template <typename TS, typename TC, int L, int TX>
static void launch_pp_walls_tx(TS *f, TS *w, long na, long sb, long se, const TC *tw, const PadeWallTables &t, int nb,
                               bool upd, hipStream_t st)
{
    const size_t lds = (2 * (size_t)TX + 1) * L * 2 * sizeof(TC);
    dim3 grid((unsigned)((na + TX - 1) / TX), (unsigned)nb);
    if (upd)
        hipLaunchKernelGGL((k_pp_walls<TS, TC, L, TX, true>), grid, dim3(TX * (L / 8)), lds, st, f, w, na, sb, (int)se,
                           tw, t.ax, t.ay, t.az, t.kcm, t.kcp);
    else
        hipLaunchKernelGGL((k_pp_walls<TS, TC, L, TX, false>), grid, dim3(TX * (L / 8)), lds, st, f, w, na, sb,
                           (int)se, tw, t.ax, t.ay, t.az, t.kcm, t.kcp);
}

// 80 KiB (two workgroups to a CU) doubles the rows of the longer lines, which
// fields beyond the caches need: 256 x 256 planes, a projection with 512-point
// lines, FP64 680 us in 64 KiB and 568 in 80, FP32 236 and 234 (in the band of
// 512 x 512 planes more).  Where that leaves a few workgroups per CU the last
// ones cost more: 64 x 64 x 256 FP32 25.1 and 28.7, 128 x 128 x 256 FP32 64 and
// 69, 128 x 128 x 32 FP64 19.9 and 21.1; at most one per CU, 64 x 64 x 64 FP64
// 19.4 and 17.5.
template <typename TS, typename TC, int L>
static void launch_pp_walls(TS *f, TS *w, long na, long sb, long se, const TC *tw, const PadeWallTables &t, int nb,
                            bool upd, hipStream_t st)
{
    constexpr int BIG = pp_walls_lines<L, 2 * sizeof(TC), 2 * sizeof(TS), 80>();
    constexpr int SMALL = pp_walls_lines<L, 2 * sizeof(TC), 2 * sizeof(TS), 64>();
    const long groups = (na + BIG - 1) / BIG * nb;
    if constexpr (BIG != SMALL) {
        if (groups > 256 && groups < 2048)
            return launch_pp_walls_tx<TS, TC, L, SMALL>(f, w, na, sb, se, tw, t, nb, upd, st);
    }
    launch_pp_walls_tx<TS, TC, L, BIG>(f, w, na, sb, se, tw, t, nb, upd, st);
}

template <typename TS, typename TC>
static hipError_t run_pp_walls_t(const PoissonPlanDev &pl, TS *f, TS *w, const PadeWallTables &t, bool upd,
                                 hipStream_t st, int lines)
{
    const int ny = pl.ny, L = pl.nz, nxh = pl.nx / 2 + 1;
    const Tw<TC> tw(pl);
    const long na = lines > 0 ? lines : nxh, sb = nxh, se = (long)nxh * ny;
    switch (L) {
    case 8: launch_pp_walls<TS, TC, 8>(f, w, na, sb, se, tw.z, t, ny, upd, st); break;
    case 16: launch_pp_walls<TS, TC, 16>(f, w, na, sb, se, tw.z, t, ny, upd, st); break;
    case 32: launch_pp_walls<TS, TC, 32>(f, w, na, sb, se, tw.z, t, ny, upd, st); break;
    case 64: launch_pp_walls<TS, TC, 64>(f, w, na, sb, se, tw.z, t, ny, upd, st); break;
    case 128: launch_pp_walls<TS, TC, 128>(f, w, na, sb, se, tw.z, t, ny, upd, st); break;
    case 256: launch_pp_walls<TS, TC, 256>(f, w, na, sb, se, tw.z, t, ny, upd, st); break;
    case 512: launch_pp_walls<TS, TC, 512>(f, w, na, sb, se, tw.z, t, ny, upd, st); break;
    case 1024: launch_pp_walls<TS, TC, 1024>(f, w, na, sb, se, tw.z, t, ny, upd, st); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t run_pp_walls(const PoissonPlanDev &pl, int mode, void *f, void *w, const PadeWallTables &t, bool upd,
                        hipStream_t st, int lines)
{
    switch (mode) {
    case 0: return run_pp_walls_t<double, double>(pl, (double *)f, (double *)w, t, upd, st, lines);
    case 1: return run_pp_walls_t<float, float>(pl, (float *)f, (float *)w, t, upd, st, lines);
    case 2: return run_pp_walls_t<float, double>(pl, (float *)f, (float *)w, t, upd, st, lines);
    }
    return hipErrorInvalidValue;
}

hipError_t run_fft2(const PoissonPlanDev &pl, int mode, const void *in, void *out, int nplanes, hipStream_t st)
{
    switch (mode) {
    case 0: return run_fft2_t<double, double>(pl, (const double *)in, (double *)out, nplanes, st);
    case 1: return run_fft2_t<float, float>(pl, (const float *)in, (float *)out, nplanes, st);
    case 2: return run_fft2_t<float, double>(pl, (const float *)in, (float *)out, nplanes, st);
    }
    return hipErrorInvalidValue;
}

hipError_t run_ifft2(const PoissonPlanDev &pl, int mode, const void *in, void *work, void *out, int nplanes,
                     int oddball, hipStream_t st)
{
    switch (mode) {
    case 0:
        return run_ifft2_t<double, double>(pl, (const double *)in, (double *)work, (double *)out, nplanes, oddball,
                                           st);
    case 1:
        return run_ifft2_t<float, float>(pl, (const float *)in, (float *)work, (float *)out, nplanes, oddball, st);
    case 2:
        return run_ifft2_t<float, double>(pl, (const float *)in, (float *)work, (float *)out, nplanes, oddball, st);
    }
    return hipErrorInvalidValue;
}

hipError_t run_zmul(const PoissonPlanDev &pl, int mode, const void *in, void *out, const SpecMul &m, hipStream_t st,
                    int lines)
{
    switch (mode) {
    case 0: return run_zmul_t<double, double>(pl, (const double *)in, (double *)out, m, st, lines);
    case 1: return run_zmul_t<float, float>(pl, (const float *)in, (float *)out, m, st, lines);
    case 2: return run_zmul_t<float, double>(pl, (const float *)in, (float *)out, m, st, lines);
    }
    return hipErrorInvalidValue;
}

// x lines of the half spectrum (pitch nxp complex): v *= i kv[kx] (imag) or kv[kx]
template <typename TS>
__global__ void __launch_bounds__(256) k_xline_mul(TS *spec, int nxp, int nxh, long nlines, const double *kv, int imag)
{
    const long total = (long)nxh * nlines;
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
        const long line = e / nxh;
        const int kx = (int)(e - line * nxh);
        TS *p = spec + 2 * (line * nxp + kx);
        const double k = kv[kx];
        const double re = (double)p[0], im = (double)p[1];
        if (imag) {
            p[0] = (TS)(-k * im);
            p[1] = (TS)(k * re);
        } else {
            p[0] = (TS)(k * re);
            p[1] = (TS)(k * im);
        }
    }
}

template <typename TS, typename TC>
static hipError_t run_fourier_deriv_t(const PoissonPlanDev &pl, int dir, int imag, const TS *in, TS *out, TS *work,
                                      long na, long nb, const double *kv, hipStream_t st)
{
    const Tw<TC> tw(pl);
    if (dir == 1) {
        // r2c lines, multiply, c2r: the c2r returns L times the inverse transform
        const int nx = pl.nx, L = nx / 2, nxh = L + 1, nxp = pl.nxp;
        const long nlines = na * nb;
        x_fft<TS, TC>(L, false, in, work, nlines, tw.x, tw.xn, (TC)1, nxp, 0, st);
        long blocks = ((long)nxh * nlines + 255) / 256;
        if (blocks > 65536) blocks = 65536;
        hipLaunchKernelGGL((k_xline_mul<TS>), dim3((unsigned)blocks), dim3(256), 0, st, work, nxp, nxh, nlines, kv,
                           imag);
        x_fft<TS, TC>(L, true, work, out, nlines, tw.x, tw.xn, (TC)(1.0 / L), nxp, 0, st);
        return hipGetLastError();
    }
    // y / z: consecutive pairs along the contiguous index read as one complex
    // value (the operator is real and maps real lines to real lines, so the
    // real and imaginary parts come back as the two derivatives); one fused
    // forward -> multiply -> inverse pass along the direction
    SpecMul pm{};
    pm.az = kv;
    pm.kind = imag ? 3 : 4;
    if (dir == 2) {
        const int n = pl.ny;
        pm.scale = 1.0 / n;
        strided_fft<TS, TC, 2>(n, in, out, na / 2, (long)(na / 2) * n, na / 2, tw.y, pm, (int)nb, st);
    } else {
        const int n = pl.nz;
        pm.scale = 1.0 / n;
        strided_fft<TS, TC, 2>(n, in, out, na * nb / 2, 0, na * nb / 2, tw.z, pm, 1, st);
    }
    return hipGetLastError();
}

hipError_t run_fourier_deriv(const PoissonPlanDev &pl, int mode, int dir, int imag, const void *in, void *out,
                             void *work, long na, long nb, const double *kv, hipStream_t st)
{
    switch (mode) {
    case 0:
        return run_fourier_deriv_t<double, double>(pl, dir, imag, (const double *)in, (double *)out, (double *)work,
                                                   na, nb, kv, st);
    case 1:
        return run_fourier_deriv_t<float, float>(pl, dir, imag, (const float *)in, (float *)out, (float *)work, na,
                                                 nb, kv, st);
    case 2:
        return run_fourier_deriv_t<float, double>(pl, dir, imag, (const float *)in, (float *)out, (float *)work, na,
                                                  nb, kv, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace pdo
