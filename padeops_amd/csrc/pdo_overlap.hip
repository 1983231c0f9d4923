// Compact operators on pencils of any length: overlapping segments.
//
// The register kernels of pdo_compact.hip cut a pencil into segments of 32
// rows, so they take n = 32 P only.  Here the P = ceil(n / m) segments still
// hold exactly m rows (32, or 16 for short pencils) in the registers of one
// lane, but overlap: segment s covers rows [start(s), start(s) + m) and stores
// the q0 or q0 + 1 rows up to the next start.  Rows that two segments share
// are solved by both from the same equations, so the partitioned solve is
// unchanged except that a segment takes its neighbours' values from rows
// inside them; every segment away from the ends keeps the same LU factors and
// spikes whatever n is.  Overlap costs (P m - n) / n in arithmetic and in
// loads that hit the cache, nothing in HBM traffic.
//
// These sizes ran on the one-lane-per-pencil kernel before: n rows in one
// serial chain, an FP64 scratch field in HBM, and x pencils read at a stride
// of n.  Measured, before -> after: a cd10 pass over 180 x 96 x 100 FP32
// values (14 MB in and out) along non-periodic x 276 -> 20 us, along z
// 276 -> 14 us; the three cd10 passes of 201 x 129 x 151 FP64 values 864 ->
// 93 us; the three cf90 passes of 300 x 161 x 200 FP64 values 1319 -> 181 us.
// The arithmetic stays FP64 for both storage types, as that kernel's was.
// The bound is memory (2 words per point); fields this small are served by
// the Infinity Cache, and what is left above it is the load-solve-store
// sequence of a few workgroups per CU.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "pdo_stencil.hpp"

namespace pdo {

namespace {

// first row of segment s: s smul / D, exact for the products met (below 2^15
// with D <= 32)
__device__ __forceinline__ int seg_start(const ApplyArgs &A, int s)
{
    return (int)(((unsigned long long)((unsigned)s * A.smul) * A.sdiv) >> 31);
}

// what segment s holds: its first row, the rows it stores, the local rows that
// the previous segment reads (lo, K of them) and those the next one reads (hi)
struct Seg {
    int r0, own, lo, hi;
};
template <int K> __device__ __forceinline__ Seg segment(const ApplyArgs &A, int s, int m)
{
    Seg g;
    const int last = A.P - 1, end = A.periodic ? A.n_sys : seg_start(A, last) + m;
    g.r0 = seg_start(A, s);
    g.own = (s < last ? seg_start(A, s + 1) : end) - g.r0;
    const int prev = s > 0 ? s - 1 : last;
    g.lo = m - ((prev < last ? seg_start(A, prev + 1) : end) - seg_start(A, prev));
    g.hi = g.own - K;
    return g;
}

// input row of window position r (a row relative to the pencil's start).
// Without periodicity the rows past the ends, which only enter values that
// closure rows replace, take any row of the pencil.
__device__ __forceinline__ int wrap_row(const ApplyArgs &A, int r, bool per)
{
    const int period = per ? A.n_sys : A.n_in, end = per ? A.n_read : A.n_in;
    return r < 0 ? r + period : (r >= end ? r - period : r);
}

// Tables of one segment type, m rows each: lower factors [m][K], inverse pivot
// and upper factors [m][1 + K], spikes [m][2K].  The two sweeps read arrays of
// their own: interleaved, the compiler widens the forward sweep's scalar loads
// over the backward sweep's factors and holds those in spilled registers.
template <int K, int M> constexpr int type_words() { return M * (K + 1 + K + 2 * K); }

template <int K, int M, int SB, typename PT> __device__ __forceinline__ void sweep(double (&d)[M], PT tb)
{
    PT up = tb + M * K;
#pragma unroll
    for (int j = 1; j < M; ++j) {
        d[j] -= tb[j * K] * d[j - 1];
        if (K == 2 && j >= 2) d[j] -= tb[j * K + 1] * d[j - 2];
        PDO_SCHED_FENCE(j, SB);
    }
#pragma unroll
    for (int j = M - 1; j >= 0; --j) {
        double v = d[j] * up[j * (1 + K)];
        if (j + 1 < M) v -= up[j * (1 + K) + 1] * d[j + 1];
        if (K == 2 && j + 2 < M) v -= up[j * (1 + K) + 2] * d[j + 2];
        d[j] = v;
        PDO_SCHED_FENCE(j, SB);
    }
}

// closure rows of the first (left: rows 0 .. nbl - 1) or the last segment's
// RHS, in the lanes where `mine`; ld(c) reads input column c.  They read their
// columns again (from the cache or LDS) rather than from the window, which is
// dead by then.  Lanes select instead of branching where `mine` varies: a
// branch here would split the block whose scheduling fences bound the table
// loads in flight.
template <int M, class LD>
__device__ __forceinline__ void end_rows(const ApplyArgs &A, double (&d)[M], bool left, bool mine, LD ld)
{
    const double *sp = A.tab_d + A.o_sp + (left ? 0 : NBMAX * WBMAX);
    const int col = left ? 0 : A.n_in - WBMAX;
    double x[WBMAX];
#pragma unroll
    for (int q = 0; q < WBMAX; ++q) x[q] = ld(col + q);
#pragma unroll
    for (int j = 0; j < NBMAX; ++j) {
        // right rows are stored from row m - nbr on; rows that are none read
        // the table's zeros or another row's weights, and are not taken
        const int i = left ? j : j - (NBMAX - A.nbr);
        const bool take = mine && (left ? j < A.nbl : i >= 0);
        double acc = 0;
#pragma unroll
        for (int q = 0; q < WBMAX; ++q) acc = fma(sp[(i < 0 ? 0 : i) * WBMAX + q], x[q], acc);
        double &dj = d[left ? j : M - NBMAX + j];
        dj = take ? acc : dj;
    }
}

// Solve the segment whose RHS is in d: local solve, exchange of the 2K rows
// that the neighbours read (red: [P][2K][pitch] values, lane pl of a pitch),
// and the spikes.  tb: this segment's tables (any address space), SB rows
// of them loaded ahead; s may vary between the lanes of a wave unless UNI.  All threads of the block take
// part.
template <int K, int M, bool UNI, int SB, typename PT>
__device__ __forceinline__ void ovl_solve(const ApplyArgs &A, double (&d)[M], PT tb, double *red, const double *gl, int pitch, int s,
                                          int pl, const Seg &g)
{
    constexpr int K2 = 2 * K;
    const int P = A.P;
    sweep<K, M, SB>(d, tb);
    // rows in registers cannot be indexed: each row in range is written under
    // its own condition, which costs less than selecting the values would
    double *rlo = red + (s * K2 - g.lo) * pitch + pl, *rhi = red + (s * K2 + K - g.hi) * pitch + pl;
#pragma unroll
    for (int j = 0; j < M; ++j) {
        if ((unsigned)(j - g.lo) < (unsigned)K) rlo[j * pitch] = d[j];
        if ((unsigned)(j - g.hi) < (unsigned)K) rhi[j * pitch] = d[j];
    }
    __syncthreads();
    double yl[2] = {0, 0}, yr[2] = {0, 0};
    auto reduce = [&](auto G) {
        int t = s + A.d0;
        t -= t >= P ? P : 0;
        for (int id = 0; id < A.nd; ++id) {
            const double *zp = red + t * K2 * pitch + pl;
            double z[K2];
#pragma unroll
            for (int c = 0; c < K2; ++c) z[c] = zp[c * pitch];
#pragma unroll
            for (int c = 0; c < K2; ++c) {
#pragma unroll
                for (int q = 0; q < K; ++q) {
                    yl[q] = fma(G[q * K2 + c], z[c], yl[q]);
                    yr[q] = fma(G[(K + q) * K2 + c], z[c], yr[q]);
                }
            }
            G += K2 * K2;
            t = t == P - 1 ? 0 : t + 1;
        }
    };
    const int go = A.guni ? 0 : s * A.nd * K2 * K2;
    if (!UNI && A.glds) reduce(gl + go);
    else reduce(A.tab_d + A.o_G + go);
    PT spk = tb + M * (2 * K + 1);
#pragma unroll
    for (int j = 0; j < M; ++j) {
#pragma unroll
        for (int q = 0; q < K; ++q) {
            d[j] = fma(-spk[j * K2 + q], yl[q], d[j]);
            d[j] = fma(-spk[j * K2 + K + q], yr[q], d[j]);
        }
        // the row is complete here, not inside the condition of its store,
        // where the compiler would move the sums and keep every spike until then
        asm volatile("" : "+v"(d[j]));
        PDO_SCHED_FENCE(j, SB);
    }
}

// ---------------------------------------------------------------------------
// strided pencils (y, z).  NPW = 64: one wave per segment (P <= 16), so rows,
// types and tables are scalar.  NPW = 32: two segments per wave (P <= 32);
// tables from LDS when the types differ (LT, no periodicity).  Lanes run over
// all na nb pencils of a y pass, not over those of one plane, so that a short
// contiguous index leaves no lane idle (A.flat); in a field of 4 GiB and more
// grid y is the plane.
// ---------------------------------------------------------------------------
// Tables a workgroup reads from LDS: the coupling rows (A.glds words) and, with
// LT, types 0, 1, 2 (or 3 alone).  Loaded to registers here, ahead of the field
// loads, so that one round trip to memory serves both; stage_write puts them
// in place.  Reading them where they are needed costs a dependent miss each.
constexpr int STAGE = 8;
template <int K, int M, bool LT> struct Staged {
    double v[STAGE];
    const double *src, *tab;
    int ng, nw;
    __device__ __forceinline__ double at(int i) const { return i < ng ? src[i] : tab[i - ng]; }
    __device__ __forceinline__ Staged(const ApplyArgs &A)
    {
        constexpr int TW = type_words<K, M>();
        src = A.tab_d + A.o_G;
        tab = A.tab_d + A.o_fac + (A.P == 1 ? 3 : 0) * TW;
        ng = A.glds;
        nw = ng + (LT ? (A.P == 1 ? 1 : 3) * TW : 0);
#pragma unroll
        for (int i = 0; i < STAGE; ++i) {
            const int e = threadIdx.x + i * blockDim.x;
            v[i] = e < nw ? at(e) : 0.0;
        }
    }
    __device__ __forceinline__ void write(double *lds) const
    {
#pragma unroll
        for (int i = 0; i < STAGE; ++i) {
            const int e = threadIdx.x + i * blockDim.x;
            if (e < nw) lds[e] = v[i];
        }
        for (int e = threadIdx.x + STAGE * blockDim.x; e < nw; e += blockDim.x) lds[e] = at(e);
    }
};

// scalar rows (UNI) read their tables through the scalar cache
struct NotStaged {
    __device__ __forceinline__ NotStaged(const ApplyArgs &) {}
    __device__ __forceinline__ void write(double *) const {}
};

template <int FAM, typename TS, int M, int NPW, bool LT, bool EPI, typename ARGS>
__global__ void __launch_bounds__(1024) k_ovl_strided(ARGS B)
{
    const ApplyArgs &A = pass_of(B);
    using F = Fam<FAM>;
    constexpr int K = F::K, R = F::R, W = M + 2 * R;
    constexpr bool UNI = NPW == 64;
    const int P = A.P;
    const int s = UNI ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : (int)threadIdx.x / NPW;
    const int pl = threadIdx.x % NPW;
    const unsigned id = blockIdx.x * NPW + pl;
    const unsigned na = (unsigned)A.na;
    const bool act = A.flat ? id < na * (unsigned)A.nb : id < na;
    const unsigned b = A.flat && act ? id / na : 0, a = act ? id - b * na : 0;
    const int ty = A.periodic ? 1 : (P == 1 ? 3 : (s == 0 ? 0 : (s == P - 1 ? 2 : 1)));
    const Seg g = segment<K>(A, s, M);
    const int r0 = g.r0, own = g.own;
    std::conditional_t<UNI, NotStaged, Staged<K, M, LT>> stage(A);
    const unsigned vi = (a + b * (unsigned)A.sb_in) * (unsigned)sizeof(TS);
    const char *fb = (const char *)A.f + (size_t)blockIdx.y * A.sb_in * sizeof(TS);
    TS win[W];
    const __amdgpu_buffer_rsrc_t rs = field_rsrc(A.f);
    const unsigned ss = (unsigned)A.se_in * (unsigned)sizeof(TS);
    // offset of row r0 - R (modulo 2^32), and how far the wrapped rows are off
    const unsigned vl = vi + (unsigned)(r0 - R) * ss;
    const unsigned turn = (unsigned)(A.periodic ? A.n_sys : A.n_in) * ss;
    const int end = A.periodic ? A.n_read : A.n_in;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        if constexpr (UNI) {
            const int r = wrap_row(A, r0 - R + w, A.periodic);
            win[w] = *(const TS *)(fb + (size_t)r * A.se_in * sizeof(TS) + vi);
        } else {
            // the whole offset in the lane's 32 bits, where a row before the
            // pencil's start wraps back into range
            const int r = r0 - R + w;
            const unsigned vo = vl + (unsigned)w * ss;
            win[w] = buf_ld<TS>(rs, r < 0 ? vo + turn : (r >= end ? vo - turn : vo), 0u);
        }
    }
    double d[M];
#pragma unroll
    for (int j = 0; j < M; ++j) d[j] = stencil_row<FAM, double>(win, j, A.c);
    if (!A.periodic) {
        auto ld = [&](int r) {
            return UNI ? (double)*(const TS *)(fb + (size_t)r * A.se_in * sizeof(TS) + vi)
                       : (double)buf_ld<TS>(rs, vi, (unsigned)r * ss);
        };
        if (!UNI || s == 0) end_rows<M>(A, d, true, s == 0, ld);
        if (!UNI || s == P - 1) end_rows<M>(A, d, false, s == P - 1, ld);
    }
    extern __shared__ double lds[];
    double *gl = lds + P * 2 * K * NPW, *tb = gl + A.glds;
    stage.write(gl);
    if constexpr (LT) {
        __syncthreads();
        ovl_solve<K, M, UNI, 2>(A, d, tb + (P == 1 ? 0 : ty) * type_words<K, M>(), lds, gl, NPW, s, pl, g);
    } else {
        ovl_solve<K, M, UNI, 8>(A, d, A.tab_d + A.o_fac + (UNI ? ty : 1) * type_words<K, M>(), lds, gl, NPW, s, pl, g);
    }
    if (!act) return;
    const unsigned vo = (a + b * (unsigned)A.sb_out) * (unsigned)sizeof(TS);
    char *ob = (char *)A.out + (size_t)blockIdx.y * A.sb_out * sizeof(TS);
    if constexpr (EPI) {
        // the operand's rows in chunks, read before the chunk's rows are
        // written (it may be the output)
        const char *xb = (const char *)A.aux + (size_t)blockIdx.y * A.sb_out * sizeof(TS);
        constexpr int CH = 8;
#pragma unroll
        for (int j0 = 0; j0 < M; j0 += CH) {
            double x[CH];
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                x[j] = 0.0;
                if (A.epi != 3 && j0 + j < own)
                    x[j] = (double)*(const TS *)(xb + (size_t)(r0 + j0 + j) * A.se_out * sizeof(TS) + vo);
            }
#pragma unroll
            for (int j = 0; j < CH; ++j) d[j0 + j] = A.epi == 1 ? x[j] + d[j0 + j] : x[j] - d[j0 + j];
        }
    }
    if constexpr (UNI) {
#pragma unroll
        for (int j = 0; j < M; ++j)
            if (j < own) *(TS *)(ob + (size_t)(r0 + j) * A.se_out * sizeof(TS) + vo) = (TS)d[j];
    } else {
        const __amdgpu_buffer_rsrc_t ro = field_rsrc(A.out);
        const unsigned so = (unsigned)A.se_out * (unsigned)sizeof(TS), vr = vo + (unsigned)r0 * so;
#pragma unroll
        for (int j = 0; j < M; ++j)
            if (j < own) buf_st((TS)d[j], ro, vr, (unsigned)j * so);
    }
    // periodic edge layouts repeat row 0 at row n_sys
    if (A.n_out > A.n_sys && s == 0) *(TS *)(ob + (size_t)A.n_sys * A.se_out * sizeof(TS) + vo) = (TS)d[0];
}

// ---------------------------------------------------------------------------
// contiguous pencils (x): TP whole pencils staged in LDS with coalesced loads
// of any alignment, lanes = (segment, pencil) with the pencil fastest.  The
// odd pitch LD sends the lanes of a half-wave, which read one row each of
// neighbouring pencils, to distinct banks.
// ---------------------------------------------------------------------------
template <int FAM, typename TS, int M, bool LT, bool EPI, typename ARGS>
__global__ void __launch_bounds__(512) k_ovl_x(ARGS B, int TP, int LD, unsigned magic)
{
    const ApplyArgs &A = pass_of(B);
    using F = Fam<FAM>;
    constexpr int K = F::K, R = F::R, W = M + 2 * R;
    const int P = A.P, n = A.n_sys, nt = TP * P;
    extern __shared__ double lds[];
    double *red = lds, *gl = red + P * 2 * K * TP, *tb = gl + A.glds;
    const Staged<K, M, LT> stage(A);
    TS *tile = (TS *)(tb + (LT ? (P == 1 ? 1 : 3) * type_words<K, M>() : 0));
    const int p = threadIdx.x % TP, s = threadIdx.x / TP;
    const long pen0 = (long)blockIdx.x * TP, left = A.na * A.nb - pen0;
    const int total = (int)(left < TP ? left : TP) * n;
    const TS *__restrict__ f = (const TS *)A.f + pen0 * n;
    // element e is row e % n of pencil e / n; e n < 2^32 makes the quotient by
    // the rounded-up reciprocal exact.  (Holding all n / P loads of a thread in
    // flight takes 225 instead of 124 registers and halves the waves of large
    // fields: 331 against 213-240 us for 384 x 320 x 640, 1 us gained on small ones.)
    const int pad = LD - n;  // 0 or 1
#pragma unroll 8
    for (int e = threadIdx.x; e < total; e += nt) {
        const int q = (int)__umulhi((unsigned)e, magic);
        tile[e + (q & -pad)] = f[e];
    }
    stage.write(gl);
    __syncthreads();
    const int ty = A.periodic ? 1 : (P == 1 ? 3 : (s == 0 ? 0 : (s == P - 1 ? 2 : 1)));
    const Seg g = segment<K>(A, s, M);
    const int r0 = g.r0, own = g.own;
    TS *line = tile + p * LD;
    TS win[W];
#pragma unroll
    for (int w = 0; w < W; ++w) {
        win[w] = line[wrap_row(A, r0 - R + w, !LT)];
    }
    double d[M];
#pragma unroll
    for (int j = 0; j < M; ++j) d[j] = stencil_row<FAM, double>(win, j, A.c);
    if constexpr (LT) {
        auto ld = [&](int r) { return (double)line[r]; };
        end_rows<M>(A, d, true, s == 0, ld);
        end_rows<M>(A, d, false, s == P - 1, ld);
        ovl_solve<K, M, false, 2>(A, d, tb + (P == 1 ? 0 : ty) * type_words<K, M>(), red, gl, TP, s, p, g);
    } else {
        ovl_solve<K, M, false, 8>(A, d, A.tab_d + A.o_fac + type_words<K, M>(), red, gl, TP, s, p, g);
    }
    // the exchange's barrier came after every read of the tile
#pragma unroll
    for (int j = 0; j < M; ++j)
        if (j < own) line[r0 + j] = (TS)d[j];
    __syncthreads();
    TS *__restrict__ out = (TS *)A.out + pen0 * n;
    if constexpr (!EPI) {
#pragma unroll 8
        for (int e = threadIdx.x; e < total; e += nt) {
            const int q = (int)__umulhi((unsigned)e, magic);
            out[e] = tile[e + (q & -pad)];
        }
        return;
    }
    TS *o = (TS *)A.out + pen0 * n;  // may be the operand
    const TS *aux = (const TS *)A.aux + (A.epi == 3 ? 0 : pen0 * n);
    for (int e0 = threadIdx.x; e0 < total; e0 += 4 * nt) {
        double x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = e0 + i * nt;
            x[i] = A.epi != 3 && e < total ? (double)aux[e] : 0.0;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = e0 + i * nt;
            if (e >= total) break;
            const int q = (int)__umulhi((unsigned)e, magic);
            const double y = (double)tile[e + (q & -pad)];
            o[e] = (TS)(A.epi == 1 ? x[i] + y : x[i] - y);
        }
    }
}

// the kernel for one pass or for several
template <class K1, class KB, class... X>
void go(K1 one, KB several, int count, dim3 grid, dim3 block, size_t lds, hipStream_t st, const ApplyBatch &B, X... x)
{
    if (count > 1) hipLaunchKernelGGL(several, grid, block, lds, st, B, x...);
    else hipLaunchKernelGGL(one, grid, block, lds, st, B.a[0], x...);
}

// f(EPI): the first derivatives have kernels with an epilogue operand
template <int FAM, class F> hipError_t with_epilogue(const ApplyArgs &A, F f)
{
    if constexpr (FAM == 0 || FAM == 2) {
        if (A.epi) {
            f(std::true_type{});
            return hipGetLastError();
        }
    }
    if (A.epi) return hipErrorInvalidValue;
    f(std::false_type{});
    return hipGetLastError();
}

// coupling rows staged in LDS up to 4 KiB: the ones of long pencils would
// cost a workgroup per CU (they come through the cache then)
template <int K> int staged_words(const ApplyArgs &A)
{
    const int words = (A.guni ? 1 : A.P) * A.nd * 4 * K * K;
    return words <= 512 ? words : 0;
}

template <int FAM, typename TS, int M> hipError_t strided_m(ApplyBatch &B, int count, hipStream_t st)
{
    constexpr int K = Fam<FAM>::K;
    const ApplyArgs &A = B.a[0];
    int glds = 0;
    for (int i = 0; i < count; i++) {
        B.a[i].glds = A.P > PMAX ? staged_words<K>(B.a[i]) : 0;
        glds = B.a[i].glds > glds ? B.a[i].glds : glds;
    }
    // pencils numbered through where 32-bit offsets reach the whole field
    const size_t nmax = (size_t)(A.n_in > A.n_out ? A.n_in : A.n_out);
    const size_t bytes = (size_t)A.na * A.nb * nmax * sizeof(TS);
    for (int i = 0; i < count; i++) B.a[i].flat = bytes < ((size_t)1 << 32) ? 1 : 0;
    const size_t pen = A.flat ? (size_t)A.na * A.nb : (size_t)A.na;
    if (!A.flat && (A.nb > 65535 || (size_t)A.na * sizeof(TS) >= ((size_t)1 << 32))) return hipErrorInvalidValue;
    if (A.P <= PMAX) {
        const dim3 grid((unsigned)((pen + 63) / 64), A.flat ? 1u : (unsigned)A.nb, (unsigned)count);
        const size_t red = (size_t)A.P * 2 * K * 64 * sizeof(double);
        return with_epilogue<FAM>(A, [&](auto e) {
            constexpr bool E = decltype(e)::value;
            go(k_ovl_strided<FAM, TS, M, 64, false, E, ApplyArgs>, k_ovl_strided<FAM, TS, M, 64, false, E, ApplyBatch>,
               count, grid, dim3(64 * A.P), red, st, B);
        });
    }
    if constexpr (M == MAXM && Fam<FAM>::SHIFT == 0) {
        if (!A.flat) return hipErrorInvalidValue;
        const dim3 grid((unsigned)((pen + 31) / 32), 1u, (unsigned)count);
        const size_t red = ((size_t)A.P * 2 * K * 32 + glds) * sizeof(double);
        const size_t tabs = sizeof(double) * 3 * type_words<K, M>();
        return with_epilogue<FAM>(A, [&](auto e) {
            constexpr bool E = decltype(e)::value;
            if (A.periodic)
                go(k_ovl_strided<FAM, TS, M, 32, false, E, ApplyArgs>,
                   k_ovl_strided<FAM, TS, M, 32, false, E, ApplyBatch>, count, grid, dim3(32 * A.P), red, st, B);
            else
                go(k_ovl_strided<FAM, TS, M, 32, true, E, ApplyArgs>,
                   k_ovl_strided<FAM, TS, M, 32, true, E, ApplyBatch>, count, grid, dim3(32 * A.P), red + tabs, st, B);
        });
    }
    return hipErrorInvalidValue;
}

template <int FAM, typename TS, int M> hipError_t x_m(ApplyBatch &B, int count, hipStream_t st)
{
    constexpr int K = Fam<FAM>::K;
    const ApplyArgs &A = B.a[0];
    int glds = 0;
    for (int i = 0; i < count; i++) {
        B.a[i].glds = staged_words<K>(B.a[i]);
        glds = B.a[i].glds > glds ? B.a[i].glds : glds;
    }
    const int n = A.n_sys, LD = n | 1;
    const size_t tabs = ((A.periodic ? 0 : (A.P == 1 ? 1 : 3) * type_words<K, M>()) + (size_t)glds) * sizeof(double);
    auto lds = [&](int tp) { return (size_t)tp * (LD * sizeof(TS) + A.P * 2 * K * sizeof(double)) + tabs; };
    // two workgroups on a CU (80 KiB each), at most 512 threads
    int TP = 32;
    while (TP > 8 && (TP * A.P > 512 || lds(TP) > 80 * 1024)) TP >>= 1;
    if (TP * A.P > 512 || lds(TP) > 160 * 1024) return hipErrorInvalidValue;
    const unsigned magic = (unsigned)(((unsigned long long)1 << 32) / n + 1);
    const dim3 grid((unsigned)((A.na * A.nb + TP - 1) / TP), 1u, (unsigned)count);
    return with_epilogue<FAM>(A, [&](auto e) {
        constexpr bool E = decltype(e)::value;
        if (A.periodic)
            go(k_ovl_x<FAM, TS, M, false, E, ApplyArgs>, k_ovl_x<FAM, TS, M, false, E, ApplyBatch>, count, grid,
               dim3(TP * A.P), lds(TP), st, B, TP, LD, magic);
        else
            go(k_ovl_x<FAM, TS, M, true, E, ApplyArgs>, k_ovl_x<FAM, TS, M, true, E, ApplyBatch>, count, grid,
               dim3(TP * A.P), lds(TP), st, B, TP, LD, magic);
    });
}

template <int FAM, typename TS> hipError_t launch_t(int shape, ApplyBatch &B, int count, hipStream_t st)
{
    const ApplyArgs &A = B.a[0];
    if (shape == SHAPE_OVL_STRIDED) return A.m == MAXM ? strided_m<FAM, TS, MAXM>(B, count, st) : strided_m<FAM, TS, MAXM / 2>(B, count, st);
    if constexpr (Fam<FAM>::SHIFT == 0) {
        if (shape == SHAPE_OVL_X) return A.m == MAXM ? x_m<FAM, TS, MAXM>(B, count, st) : x_m<FAM, TS, MAXM / 2>(B, count, st);
    }
    return hipErrorInvalidValue;
}

template <typename TS> hipError_t launch_f(int family, int shape, ApplyBatch &B, int count, hipStream_t st)
{
    switch (family) {
    case 0: return launch_t<0, TS>(shape, B, count, st);
    case 1: return launch_t<1, TS>(shape, B, count, st);
    case 2: return launch_t<2, TS>(shape, B, count, st);
    case 3: return launch_t<3, TS>(shape, B, count, st);
    case 4: return launch_t<4, TS>(shape, B, count, st);
    case 5: return launch_t<5, TS>(shape, B, count, st);
    case 6: return launch_t<6, TS>(shape, B, count, st);
    case 7: return launch_t<7, TS>(shape, B, count, st);
    case 8: return launch_t<8, TS>(shape, B, count, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_overlap(int family, int shape, bool dbl, ApplyBatch &B, int count, hipStream_t st)
{
    return dbl ? launch_f<double>(family, shape, B, count, st) : launch_f<float>(family, shape, B, count, st);
}

}  // namespace pdo
