// Device side of the closure network's evaluation, shared by the MLP's
// inference kernel and the closure's stress kernel.
//
// Each wave runs NT tiles of 16 samples through the network in the transposed
// form Z^T = W H^T: the weights are the MFMA A operand and the activations
// the B operand, so lane l = 16 g + r ends a 16-row output tile nt holding
// Z(16 nt + 4 g + i, sample r), i < 4.  A K = 32 operand (v_mfma_f32_16x16x32
// _bf16) takes eight features per lane; any assignment of features to its
// slots will do as long as the weights use the same one, so slots 4 h + i
// (h < 2) of step ks take the lane's own rows of tile 2 ks + h: an output
// tile pair is the next layer's operand and activations never leave the
// registers.  The BF16 weights of all four layers are staged in LDS once per
// (persistent) workgroup in fragment order; the biases, staged too, seed the
// accumulators.  BF16 rounding is the hardware's round-to-nearest-even
// conversion.  GELU is evaluated as z sigma(2 y) = z / (1 + 2^(-2 y log2 e)),
// y = sqrt(2/pi) (z + 0.044715 z^3), identical to 0.5 z (1 + tanh y); with
// the hardware exp2 and reciprocal it is within a few FP32 ulp of the tanhf
// form, far below the BF16 rounding of the activation.
//
// The 192 GELUs per sample bound it: 7 vector operations (2 of them
// transcendental, at a quarter of the rate) and 2 for the BF16 roundings,
// converted in pairs (one by one, with permutes to merge them, K = 16
// operands and the results in accumulation registers it took 1240 us for
// 16.8 M samples, now 1030).  Two tiles at a time halve the LDS reads of the
// weights and give the matrix cores and the vector unit independent work.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>

#include "pdo_mlp.hpp"

namespace pdo {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16v2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16v8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// two floats to BF16, the first in the low half
__device__ __forceinline__ unsigned pack2(float a, float b)
{
    return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){a, b}, bf16v2));
}

__device__ __forceinline__ float gelu_fast(float z)
{
    constexpr float c1 = (float)(-2.0 * 0.7978845608028654 * 1.4426950408889634);
    constexpr float c3 = (float)(-2.0 * 0.7978845608028654 * 1.4426950408889634 * 0.044715);
    const float a = z * __builtin_fmaf(z * z, c3, c1);
    return z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(a));
}

// BF16 pre-activations, GELU, BF16 activations of one output tile
__device__ __forceinline__ u32x2 hidden_act(f32x4 z)
{
    u32x2 o;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const unsigned p = pack2(z[2 * q], z[2 * q + 1]);
        o[q] = pack2(gelu_fast(__uint_as_float(p << 16)), gelu_fast(__uint_as_float(p & 0xffff0000u)));
    }
    return o;
}

// LDS of a workgroup: weights of layer 1 (4 fragments of K = 16), 2 and 3
// (4 x 2 fragments of K = 32 each), 4 (2 fragments), and the biases
struct MlpLds {
    u32x2 w1[4 * 64];
    u32x4 w[18 * 64];
    float b[3 * MLP_HID + MLP_OUT_PAD];
};

// every thread of the workgroup; a barrier must follow
__device__ __forceinline__ void mlp_stage(MlpLds &L, const unsigned short *__restrict__ Wb, const float *__restrict__ P)
{
    for (int i = threadIdx.x; i < 3 * MLP_HID + MLP_OUT_PAD; i += blockDim.x) {
        const int l = i / MLP_HID;
        const int off = l == 0 ? MLP_OFF_B1 : l == 1 ? MLP_OFF_B2 : l == 2 ? MLP_OFF_B3 : MLP_OFF_B4;
        L.b[i] = P[off + i - l * MLP_HID];
    }
    for (int i = threadIdx.x; i < 4 * 64; i += blockDim.x) {
        const int lane = i & 63;
        const unsigned short *q = Wb + MLP_OFF_W1 + (16 * (i >> 6) + (lane & 15)) * MLP_IN_PAD + 4 * (lane >> 4);
        L.w1[i] = (u32x2){q[0] | (unsigned)q[1] << 16, q[2] | (unsigned)q[3] << 16};
    }
    // fragment f of layers 2 .. 4: layer 2 (nt, ks) at 2 nt + ks, layer 3 at
    // 8 + 2 nt + ks, layer 4 at 16 + ks; slot 4 h + i holds
    // W(16 nt + r, 32 ks + 16 h + 4 g + i)
    for (int i = threadIdx.x; i < 18 * 64; i += blockDim.x) {
        const int lane = i & 63, f = i >> 6, nt = f < 16 ? (f & 7) >> 1 : 0, ks = f & 1;
        const int off = f < 8 ? MLP_OFF_W2 : f < 16 ? MLP_OFF_W3 : MLP_OFF_W4;
        const unsigned short *q = Wb + off + (16 * nt + (lane & 15)) * MLP_HID + 32 * ks + 4 * (lane >> 4);
        u32x4 v;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int p = 0; p < 2; ++p) v[2 * h + p] = q[16 * h + 2 * p] | (unsigned)q[16 * h + 2 * p + 1] << 16;
        L.w[i] = v;
    }
}

// the network on NT tiles: x[t] holds features 4 g .. 4 g + 3 of the lane's
// sample (BF16, zero beyond the tenth), y[t] its outputs 4 g .. 4 g + 3
template <int NT> __device__ __forceinline__ void mlp_eval(const MlpLds &L, const u32x2 (&x)[NT], f32x4 (&y)[NT])
{
    const int lane = threadIdx.x & 63, g = lane >> 4;
    auto bias = [&](int l, int nt) { return *(const f32x4 *)(L.b + l * MLP_HID + 16 * nt + 4 * g); };
    auto mma = [](u32x4 a, u32x2 b0, u32x2 b1, f32x4 c) {
        const u32x4 b = {b0[0], b0[1], b1[0], b1[1]};
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16v8, a), __builtin_bit_cast(bf16v8, b), c,
                                                       0, 0, 0);
    };
    u32x2 h[NT][4], k[NT][4];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
        const bf16x4 a = __builtin_bit_cast(bf16x4, L.w1[nt * 64 + lane]);
        const f32x4 b = bias(0, nt);
#pragma unroll
        for (int t = 0; t < NT; ++t)
            h[t][nt] = hidden_act(
                __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, __builtin_bit_cast(bf16x4, x[t]), b, 0, 0, 0));
    }
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
        const u32x4 a0 = L.w[(2 * nt) * 64 + lane], a1 = L.w[(2 * nt + 1) * 64 + lane];
        const f32x4 b = bias(1, nt);
#pragma unroll
        for (int t = 0; t < NT; ++t)
            k[t][nt] = hidden_act(mma(a1, h[t][2], h[t][3], mma(a0, h[t][0], h[t][1], b)));
    }
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
        const u32x4 a0 = L.w[(8 + 2 * nt) * 64 + lane], a1 = L.w[(9 + 2 * nt) * 64 + lane];
        const f32x4 b = bias(2, nt);
#pragma unroll
        for (int t = 0; t < NT; ++t)
            h[t][nt] = hidden_act(mma(a1, k[t][2], k[t][3], mma(a0, k[t][0], k[t][1], b)));
    }
    const u32x4 a0 = L.w[16 * 64 + lane], a1 = L.w[17 * 64 + lane];
    const f32x4 b = bias(3, 0);
#pragma unroll
    for (int t = 0; t < NT; ++t) y[t] = mma(a1, h[t][2], h[t][3], mma(a0, h[t][0], h[t][1], b));
}

// workgroups of a persistent kernel that are resident at once on the current
// device; the answer is kept per kernel and device
struct Resident {
    static constexpr int MAXDEV = 64;
    std::atomic<int> blocks[MAXDEV];
};
hipError_t resident_blocks(Resident &r, const void *kernel, int threads, int *blocks);

}  // namespace pdo
