// Device code the compact-operator kernels share: the families' stencils and
// the banded solve of one segment.
#pragma once

#include <hip/hip_runtime.h>

#include "pdo_kernels.hpp"

namespace pdo {

template <int FAM> struct Fam;
//                                  K  R  sigma shift center
#define PDO_FAM(ID, K_, R_, S_, H_, C_)                                                   \
    template <> struct Fam<ID> {                                                          \
        static constexpr int K = K_, R = R_, SIGMA = S_, SHIFT = H_;                      \
        static constexpr bool CENTER = C_;                                                \
    };
PDO_FAM(0, 1, 2, -1, 0, false)   // cd06 d1
PDO_FAM(1, 1, 2, +1, 0, true)    // cd06 d2, staggered d2
PDO_FAM(2, 2, 3, -1, 0, false)   // cd10 d1
PDO_FAM(3, 2, 3, +1, 0, true)    // cd10 d2
PDO_FAM(4, 2, 4, +1, 0, true)    // cf90
PDO_FAM(5, 1, 2, -1, +1, false)  // staggered ddz E2C
PDO_FAM(6, 1, 2, -1, -1, false)  // staggered ddz C2E
PDO_FAM(7, 1, 2, +1, +1, false)  // staggered interp E2C
PDO_FAM(8, 1, 2, +1, -1, false)  // staggered interp C2E
#undef PDO_FAM

// interior stencil of output row j; window index of input row (row0 + j + o)
// is j + R + o.
template <int FAM, typename T, typename TW, int W>
__device__ __forceinline__ T stencil_row(const TW (&win)[W], int j, const T *c)
{
    using F = Fam<FAM>;
    T acc = F::CENTER ? c[0] * (T)win[j + F::R] : T(0);
#pragma unroll
    for (int q = 1; q <= F::R; ++q) {
        const int hi = j + F::R + q + (F::SHIFT < 0 ? -1 : 0);
        const int lo = j + F::R - q + (F::SHIFT > 0 ? 1 : 0);
        const T pr = F::SIGMA > 0 ? (T)win[hi] + (T)win[lo] : (T)win[hi] - (T)win[lo];
        acc = fma(c[q], pr, acc);
    }
    return acc;
}

// local banded solve, in place, factors fac[j*5 + {l1,l2,inv,u1,u2}]
// Scheduling fence every SB rows: the row coefficients are uniform scalar
// loads; without a fence the scheduler hoists all of them (hundreds of
// values) and spills scalar registers into vector lanes.
#define PDO_SCHED_FENCE(j, SB) \
    if (((j) % (SB)) == (SB) - 1) __builtin_amdgcn_sched_barrier(0)

template <int K, int MM, bool EXACT, int SB = 8, typename T, typename PT>
__device__ __forceinline__ void local_solve(T (&d)[MM], PT fac, int m)
{
#pragma unroll
    for (int j = 1; j < MM; ++j) {
        if (EXACT || j < m) {
            T v = d[j] - fac[j * 5 + 0] * d[j - 1];
            if (K == 2 && j >= 2) v -= fac[j * 5 + 1] * d[j - 2];
            d[j] = v;
        }
        PDO_SCHED_FENCE(j, SB);
    }
#pragma unroll
    for (int j = MM - 1; j >= 0; --j) {
        if (EXACT || j < m) {
            T v = d[j] * fac[j * 5 + 2];
            if (j + 1 < MM && (EXACT || j + 1 < m)) v -= fac[j * 5 + 3] * d[j + 1];
            if (K == 2 && j + 2 < MM && (EXACT || j + 2 < m)) v -= fac[j * 5 + 4] * d[j + 2];
            d[j] = v;
        }
        PDO_SCHED_FENCE(j, SB);
    }
}

template <int K, int MM, bool EXACT, int SB = 8, typename T, typename PT>
__device__ __forceinline__ void apply_spikes(T (&d)[MM], PT spk, const T (&yl)[2], const T (&yr)[2], int m)
{
#pragma unroll
    for (int j = 0; j < MM; ++j) {
        if (EXACT || j < m) {
            T v = d[j];
#pragma unroll
            for (int q = 0; q < K; ++q) {
                v = fma(-spk[j * 4 + q], yl[q], v);
                v = fma(-spk[j * 4 + 2 + q], yr[q], v);
            }
            d[j] = v;
        }
        PDO_SCHED_FENCE(j, SB);
    }
}

// ---------------------------------------------------------------------------
// raw buffer access: a uniform resource over a field plus a per-lane and a
// scalar byte offset, so that rows of a strided pencil (scalar offsets
// row * stride) cost no vector ALU work.  Byte offsets are 32-bit: the host
// sends fields of 4 GiB or more elsewhere.
// ---------------------------------------------------------------------------
__device__ __forceinline__ __amdgpu_buffer_rsrc_t field_rsrc(const void *p)
{
    // stride 0, no range limit, 32-bit data format (raw dword access)
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, -1, 0x00020000);
}
template <typename T> __device__ __forceinline__ T buf_ld(__amdgpu_buffer_rsrc_t r, unsigned vo, unsigned so);
template <> __device__ __forceinline__ float buf_ld<float>(__amdgpu_buffer_rsrc_t r, unsigned vo, unsigned so)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)vo, (int)so, 0));
}
template <> __device__ __forceinline__ double buf_ld<double>(__amdgpu_buffer_rsrc_t r, unsigned vo, unsigned so)
{
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)vo, (int)so, 0));
}
__device__ __forceinline__ void buf_st(float v, __amdgpu_buffer_rsrc_t r, unsigned vo, unsigned so)
{
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, (int)vo, (int)so, 0);
}
__device__ __forceinline__ void buf_st(double v, __amdgpu_buffer_rsrc_t r, unsigned vo, unsigned so)
{
    using U2 = unsigned __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), r, (int)vo, (int)so, 0);
}

}  // namespace pdo
