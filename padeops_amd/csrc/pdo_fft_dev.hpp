// Device code of the line transforms: Stockham stages, LDS layouts and the
// real-complex split and merge steps (see pdo_fft.hip for the passes).
#pragma once

#include <hip/hip_runtime.h>

#include "pdo_fft.hpp"

namespace pdo {

// complex value; aligned to its size so that LDS and HBM accesses are single
// 8-byte (FP32) or 16-byte (FP64) operations rather than pairs of words
template <typename T> struct alignas(2 * sizeof(T)) C2 { T x, y; };

template <typename T> __device__ __forceinline__ C2<T> cmul(C2<T> a, C2<T> b)
{
    return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <typename T> __device__ __forceinline__ C2<T> cadd(C2<T> a, C2<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T> __device__ __forceinline__ C2<T> csub(C2<T> a, C2<T> b) { return {a.x - b.x, a.y - b.y}; }
// multiply by SIGN*i
template <typename T, int SIGN> __device__ __forceinline__ C2<T> mul_i(C2<T> a)
{
    return SIGN > 0 ? C2<T>{-a.y, a.x} : C2<T>{a.y, -a.x};
}

template <typename T, int SIGN> __device__ __forceinline__ void dft2(C2<T> &a, C2<T> &b)
{
    const C2<T> t = csub(a, b);
    a = cadd(a, b);
    b = t;
}

// y_m = sum_r x_r (SIGN i)^(r m), in place, on x[o], x[o+s], x[o+2s], x[o+3s]
template <typename T, int SIGN> __device__ __forceinline__ void dft4(C2<T> &x0, C2<T> &x1, C2<T> &x2, C2<T> &x3)
{
    const C2<T> a0 = cadd(x0, x2), a1 = csub(x0, x2);
    const C2<T> b0 = cadd(x1, x3), b1 = mul_i<T, SIGN>(csub(x1, x3));
    x0 = cadd(a0, b0);
    x1 = cadd(a1, b1);
    x2 = csub(a0, b0);
    x3 = csub(a1, b1);
}

// 8-point DFT with exp(SIGN 2 pi i / 8): radix-2 split into two DFT4
template <typename T, int SIGN> __device__ __forceinline__ void dft8(C2<T> (&v)[8])
{
    const T h = (T)0.70710678118654752440084436210484903928;
    C2<T> a[4], b[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        a[k] = cadd(v[k], v[k + 4]);
        b[k] = csub(v[k], v[k + 4]);
    }
    // b_k *= W8^k
    b[1] = cmul(b[1], C2<T>{h, SIGN * h});
    b[2] = mul_i<T, SIGN>(b[2]);
    b[3] = cmul(b[3], C2<T>{-h, SIGN * h});
    dft4<T, SIGN>(a[0], a[1], a[2], a[3]);
    dft4<T, SIGN>(b[0], b[1], b[2], b[3]);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        v[2 * m] = a[m];
        v[2 * m + 1] = b[m];
    }
}

// One Stockham stage of radix R on one line of length L, current sub-size Ns.
// The thread owns base index jb in [0, L/8) and handles items
// j = jb + it*(L/8), it < 8/R.  LD(i) reads element i of the stage input,
// ST(i, v) writes element i of the stage output.  The caller synchronizes.
template <typename T, int R, int SIGN> struct Stage {
    template <class LD>
    __device__ __forceinline__ static void load(C2<T> (&v)[8], LD ld, const C2<T> *__restrict__ tw, int L, int Ns,
                                                int jb)
    {
        const int Q = L / R, L8 = L >> 3;
#pragma unroll
        for (int it = 0; it < 8 / R; ++it) {
            const int j = jb + it * L8;
            const int k = j & (Ns - 1);
            const int step = L / (Ns * R);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                C2<T> x = ld(j + r * Q);
                if (r > 0 && Ns > 1) {  // the first stage's twiddles are all 1
                    C2<T> w = tw[(k * r * step) & (L - 1)];
                    if (SIGN > 0) w.y = -w.y;
                    x = cmul(x, w);
                }
                v[it * R + r] = x;
            }
        }
    }
    __device__ __forceinline__ static void butterfly(C2<T> (&v)[8])
    {
        if constexpr (R == 8) {
            dft8<T, SIGN>(v);
        } else if constexpr (R == 4) {
            dft4<T, SIGN>(v[0], v[1], v[2], v[3]);
            dft4<T, SIGN>(v[4], v[5], v[6], v[7]);
        } else {
#pragma unroll
            for (int it = 0; it < 4; ++it) dft2<T, SIGN>(v[2 * it], v[2 * it + 1]);
        }
    }
    template <class STO>
    __device__ __forceinline__ static void store(const C2<T> (&v)[8], STO st, int L, int Ns, int jb)
    {
        const int L8 = L >> 3;
#pragma unroll
        for (int it = 0; it < 8 / R; ++it) {
            const int j = jb + it * L8;
            const int k = j & (Ns - 1);
            const int base = (j - k) * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) st(base + r * Ns, v[it * R + r]);
        }
    }
};

// Full FFT of one line: the first stage reads through LDG, the last stage
// writes through STG, the intermediate stages live in the LDS line accessor
// `buf` (element i at buf(i)).  SRC_LDS: LDG reads the same LDS buffer, so the
// first stage also waits for every read before writing.  All threads of the
// block must call this (it synchronizes); threads with act == false only take
// part in the barriers.
template <typename T, int SIGN, bool SRC_LDS, int L, int NS, class LDG, class STG, class BUF>
__device__ __forceinline__ void line_fft_stage(LDG &ldg, STG &stg, BUF &buf, const C2<T> *__restrict__ tw, int jb,
                                               bool act)
{
    constexpr int R = (L / NS) >= 8 ? 8 : (L / NS);
    constexpr bool first = (NS == 1), last = (NS * R == L);
    C2<T> v[8];
    if (act) {
        if constexpr (first) {
            Stage<T, R, SIGN>::load(v, ldg, tw, L, NS, jb);
        } else {
            auto lds = [&](int i) { return buf(i); };
            Stage<T, R, SIGN>::load(v, lds, tw, L, NS, jb);
        }
        Stage<T, R, SIGN>::butterfly(v);
    }
    if (!first || SRC_LDS) __syncthreads();  // every LDS read of this stage is done
    if (act) {
        if constexpr (last) {
            Stage<T, R, SIGN>::store(v, stg, L, NS, jb);
        } else {
            auto sts = [&](int i, C2<T> x) { buf(i) = x; };
            Stage<T, R, SIGN>::store(v, sts, L, NS, jb);
        }
    }
    if constexpr (!last) {
        __syncthreads();  // stage output visible
        line_fft_stage<T, SIGN, SRC_LDS, L, NS * R>(ldg, stg, buf, tw, jb, act);
    }
}

// Full FFT of one line of L points: the first stage reads through LDG, the
// last stage writes through STG, the intermediate stages live in the LDS line
// accessor `buf` (element i at buf(i)).  SRC_LDS: LDG reads the same LDS
// buffer, so the first stage also waits for every read before writing.  All
// threads of the block must call this (it synchronizes); threads with
// act == false only take part in the barriers.
template <typename T, int SIGN, bool SRC_LDS, int L, class LDG, class STG, class BUF>
__device__ __forceinline__ void line_fft(LDG ldg, STG stg, BUF buf, const C2<T> *__restrict__ tw, int jb, bool act)
{
    line_fft_stage<T, SIGN, SRC_LDS, L, 1>(ldg, stg, buf, tw, jb, act);
}

template <typename TS, typename TC> struct CLoad;
template <> struct CLoad<double, double> {
    __device__ __forceinline__ static C2<double> ld(const double *p, long i)
    {
        const double2 x = reinterpret_cast<const double2 *>(p)[i];
        return {x.x, x.y};
    }
    __device__ __forceinline__ static void st(double *p, long i, C2<double> v)
    {
        reinterpret_cast<double2 *>(p)[i] = double2{v.x, v.y};
    }
};
template <typename TC> struct CLoadF {
    __device__ __forceinline__ static C2<TC> ld(const float *p, long i)
    {
        const float2 x = reinterpret_cast<const float2 *>(p)[i];
        return {(TC)x.x, (TC)x.y};
    }
    __device__ __forceinline__ static void st(float *p, long i, C2<TC> v)
    {
        reinterpret_cast<float2 *>(p)[i] = float2{(float)v.x, (float)v.y};
    }
};
template <> struct CLoad<float, float> : CLoadF<float> {};
template <> struct CLoad<float, double> : CLoadF<double> {};

// 1/x: correctly rounded in FP64; the hardware reciprocal (1 ulp) in FP32
__device__ __forceinline__ double recip(double x) { return 1.0 / x; }
__device__ __forceinline__ float recip(float x) { return __builtin_amdgcn_rcpf(x); }

// twiddles of the strided transforms staged in LDS (1) or read from the
// table in HBM / cache (0); tuning constant
#ifndef PDO_FFT_TW_LDS
#define PDO_FFT_TW_LDS 1
#endif

// the same for the x-line transforms; tuning constant
#ifndef PDO_FFT_X_TW_LDS
#define PDO_FFT_X_TW_LDS PDO_FFT_TW_LDS
#endif

// LDS rows of the strided transforms swizzled (1) or plain (0); tuning constant
#ifndef PDO_FFT_STRIDED_SWZ
#define PDO_FFT_STRIDED_SWZ 1
#endif

// XCD-aware tile order of a 2D grid of (line group, plane) tiles: workgroups
// are dispatched round-robin over the 8 XCDs in flattened order w, so XCD
// w % 8 gets the contiguous run of logical tiles below (a bijection for any
// grid).  Neighbouring line groups of a row then share one L2; with an odd
// row pitch (the (nx/2+1, ny, nz) spectra) a group's row segment straddles
// two 128-byte lines, each half read by a neighbour.
__device__ __forceinline__ void xcd_tile(unsigned &bx, unsigned &by)
{
    const unsigned gx = gridDim.x, nw = gx * gridDim.y, w = blockIdx.y * gx + blockIdx.x;
    const unsigned per = nw / 8, rem = nw % 8, xcd = w % 8, slot = w / 8;
    const unsigned lg = xcd < rem ? xcd * (per + 1) + slot : rem * (per + 1) + (xcd - rem) * per + slot;
    bx = lg % gx;
    by = lg / gx;
}

// LDS layout of an x line of L complex points.  An LDS access of 8-byte
// values is conflict-free when the 32 lanes of each half-wave fall in 32
// distinct slots (address mod 32).  The Stockham stages access a line
// contiguously (loads, the split/merge steps) and, in their stores, at
// 8 j + r and 64 (j / 8) + j % 8 + 8 r across the lanes j.
//   1: one pad element after every 8 (lines of 128 points or fewer, where a
//      half-wave spans several lines);
//   2: (L >= 256, a half-wave within one line) element i of 32-block b at
//      i ^ ((b & 7) | ((b >> 1) & 3) << 3): a permutation inside each block,
//      so contiguous runs stay conflict-free, and both store patterns spread
//      over all 32 slots.
// 0 is the plain layout.  Tuning constant.
#ifndef PDO_FFT_X_LAYOUT
#define PDO_FFT_X_LAYOUT 2
#endif
template <int L> __host__ __device__ constexpr int xslot(int i)
{
    if constexpr (PDO_FFT_X_LAYOUT == 2 && L >= 256) {
        const int b = i >> 5;
        return i ^ ((b & 7) | (((b >> 1) & 3) << 3));
    } else if constexpr (PDO_FFT_X_LAYOUT >= 1) {
        return i + (i >> 3);
    } else {
        return i;
    }
}
// line pitch (elements): past the last slot of element L (with L >= 256 a
// half-wave never spans two lines, so the lines need no relative offset)
template <int L> __host__ __device__ constexpr int xline_pitch()
{
    if constexpr (PDO_FFT_X_LAYOUT == 2 && L >= 256)
        return (L + 32) & ~31;
    else
        return xslot<L>(L) + 1;
}

// LDS bytes of an x-line workgroup: TXL lines and the staged twiddles (with
// split: also the L + 1 split/merge twiddles of the spectral-x kernels)
template <int L> static size_t xline_lds(int TXL, size_t ce, bool split = false)
{
    // with split, also the L + 1 wavenumbers (one value each, half a complex)
    return ((size_t)TXL * xline_pitch<L>() + (PDO_FFT_X_TW_LDS ? L + (split ? L + 1 + (L + 2) / 2 : 0) : 0)) * ce;
}

// the twiddle table of an x line (L values) staged in LDS after the tile of
// TXL lines; returns the LDS copy (or the table itself when staging is off).
// The first use is in the second Stockham stage, after a barrier.
template <typename TC, int L>
__device__ __forceinline__ const C2<TC> *x_twiddles(C2<TC> *tile, int TXL, const TC *twL)
{
    if constexpr (PDO_FFT_X_TW_LDS) {
        C2<TC> *twl = tile + (size_t)TXL * xline_pitch<L>();
        const C2<TC> *tw = (const C2<TC> *)twL;
        for (int i = threadIdx.x; i < L; i += blockDim.x) twl[i] = tw[i];
        return twl;
    } else {
        return (const C2<TC> *)twL;
    }
}

// the split/merge twiddles (L + 1 values) of the spectral-x kernels staged in
// LDS after the line twiddles; their first use follows a barrier
template <typename TC, int L>
__device__ __forceinline__ const C2<TC> *x_split_twiddles(C2<TC> *tile, int TXL, const TC *twN)
{
    if constexpr (PDO_FFT_X_TW_LDS) {
        C2<TC> *wl = tile + (size_t)TXL * xline_pitch<L>() + L;
        const C2<TC> *w = (const C2<TC> *)twN;
        for (int i = threadIdx.x; i <= L; i += blockDim.x) wl[i] = w[i];
        return wl;
    } else {
        return (const C2<TC> *)twN;
    }
}

// the modified wavenumbers k'(kx) (L + 1 values) of the spectral-x kernels
// staged in LDS, in the transform's arithmetic, after the split twiddles
template <typename TC, int L>
__device__ __forceinline__ const TC *x_wavenumbers(C2<TC> *tile, int TXL, const double *kp)
{
    if constexpr (PDO_FFT_X_TW_LDS) {
        TC *kl = (TC *)(tile + (size_t)TXL * xline_pitch<L>() + 2 * L + 1);
        for (int i = threadIdx.x; i <= L; i += blockDim.x) kl[i] = (TC)kp[i];
        return kl;
    } else {
        return nullptr;
    }
}

// Z_k = E_k + i O_k of the half-length inverse transform from the staged
// modes X_k (in place, one thread per pair (k, L-k)):
// E = (X_k + conj X_{L-k})/2, O = (X_k - conj X_{L-k}) conj(W^k)/2.  Only the
// real parts of the kx = 0 and kx = nx/2 modes enter (a Hermitian c2r);
// oddball != 0 drops kx = nx/2.
template <typename TC, int L, class BUF>
__device__ __forceinline__ void c2r_merge(BUF &buf, const C2<TC> *wN, int jb, int oddball)
{
    constexpr int L8 = L >> 3;
    for (int k = jb; k <= L / 2; k += L8) {
        const int kc = L - k;
        C2<TC> xk = buf(k), xc = buf(kc);
        if (k == 0) {
            xk.y = 0;
            xc.y = 0;
            if (oddball) xc.x = 0;
        }
        auto z = [&](C2<TC> a, C2<TC> b, int kk) {
            const C2<TC> ev = {(TC)0.5 * (a.x + b.x), (TC)0.5 * (a.y - b.y)};
            const C2<TC> df = {(TC)0.5 * (a.x - b.x), (TC)0.5 * (a.y + b.y)};
            const C2<TC> od = cmul(df, C2<TC>{wN[kk].x, -wN[kk].y});
            return C2<TC>{ev.x - od.y, ev.y + od.x};
        };
        const C2<TC> zk = z(xk, xc, k);
        const C2<TC> zc = z(xc, xk, kc);
        buf(k) = zk;
        if (k > 0 && kc != k) buf(kc) = zc;
    }
}

// X_k = E_k + W^k O_k of the real transform from the half-length one in buf,
// E = (Z_k + conj Z_{L-k})/2, O = (Z_k - conj Z_{L-k})/(2i)
template <typename TC, int L, class BUF>
__device__ __forceinline__ C2<TC> r2c_split(BUF &buf, const C2<TC> *wN, int k)
{
    const C2<TC> zk = buf(k == L ? 0 : k);
    const C2<TC> zc = buf(k == 0 ? 0 : L - k);
    const C2<TC> ev = {(TC)0.5 * (zk.x + zc.x), (TC)0.5 * (zk.y - zc.y)};
    const C2<TC> od = {(TC)0.5 * (zk.y + zc.y), (TC)-0.5 * (zk.x - zc.x)};
    return cadd(ev, cmul(wN[k], od));
}

// largest workgroups of the line transforms (threads); tuning constants
#ifndef PDO_FFT_STRIDED_THREADS
#define PDO_FFT_STRIDED_THREADS 1024
#endif
#ifndef PDO_FFT_X_THREADS
#define PDO_FFT_X_THREADS 256
#endif

// the fused forward-multiply-inverse pass (MODE 2) may use smaller
// workgroups than the single transforms; tuning constant
#ifndef PDO_FFT_FUSED_THREADS
#define PDO_FFT_FUSED_THREADS 1024
#endif

// lines per workgroup of the strided transforms: PDO_FFT_STRIDED_THREADS
// (PDO_FFT_FUSED_THREADS for MODE 2) threads, 8 points each, at most 64 KiB
// of LDS
template <int L, size_t CE, int MODE> constexpr int strided_fft_lines()
{
    int tx = (MODE == 2 ? PDO_FFT_FUSED_THREADS : PDO_FFT_STRIDED_THREADS) / (L / 8);
    if (tx < 1) tx = 1;
    while (tx > 1 && (size_t)tx * L * CE > 64 * 1024) tx >>= 1;
    return tx;
}

template <typename TC> struct Tw {
    const TC *x, *xn, *y, *z;
    explicit Tw(const PoissonPlanDev &pl)
    {
        const bool dbl = sizeof(TC) == 8;
        x = (const TC *)(dbl ? (const void *)pl.tw_d[0] : (const void *)pl.tw_f[0]);
        xn = (const TC *)(dbl ? (const void *)pl.twn_d : (const void *)pl.twn_f);
        y = (const TC *)(dbl ? (const void *)pl.tw_d[1] : (const void *)pl.tw_f[1]);
        z = (const TC *)(dbl ? (const void *)pl.tw_d[2] : (const void *)pl.tw_f[2]);
    }
};

}  // namespace pdo
