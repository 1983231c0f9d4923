// Learned SGS closure: a pointwise MLP 10 -> 64 -> 64 -> 64 -> 6 (GELU on the
// hidden layers), trained and evaluated with hand-written gfx950 kernels:
// BF16 weights and activations, FP32 accumulation on the matrix cores
// (v_mfma_f32_16x16x16_bf16), FP32 master parameters updated by Adam.
//
// Training: a workgroup (4 waves) owns a tile of 64 samples and runs the whole
// network on it with every weight matrix staged in LDS; wave w owns rows 16w..16w+15
// of the activation tile.  The backward kernel forms per-workgroup weight
// gradients (the batch is the contraction dimension of dW = dZ^T H) that a
// second kernel sums in a fixed order, so training is deterministic.
#include <hip/hip_runtime.h>

#include "pdo_mlp_dev.hpp"

namespace pdo {

constexpr int TILE = 64;     // samples per workgroup
constexpr int HS = 64 + 8;   // LDS row pitch of activation tiles (bf16)

__device__ __forceinline__ unsigned short to_bf16(float x)
{
    unsigned u = __float_as_uint(x);
    u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
    return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float from_bf16(unsigned short b) { return __uint_as_float((unsigned)b << 16); }

__device__ __forceinline__ float gelu_f(float z)
{
    const float t = tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z));
    return 0.5f * z * (1.0f + t);
}
__device__ __forceinline__ float gelu_grad_f(float z)
{
    const float t = tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z));
    const float du = 0.7978845608028654f * (1.0f + 3.0f * 0.044715f * z * z);
    return 0.5f * (1.0f + t) + 0.5f * z * (1.0f - t * t) * du;
}

// One 16x16 output tile of this wave: D(m, n) += sum_k A(m, k) B(k, n),
// K a multiple of 16.  Operand layout of the 16x16x16 BF16 MFMA: lane l
// holds A(l % 16, 4 (l / 16) + i) and B(4 (l / 16) + i, l % 16), i < 4; the
// result D(4 (l / 16) + i, l % 16) lands in element i of lane l.
template <class AF, class BF>
__device__ __forceinline__ f32x4 mma16(AF a, BF b, int K, f32x4 acc)
{
    const int lane = threadIdx.x & 63;
    const int r = lane & 15, g = lane >> 4;
    for (int k0 = 0; k0 < K; k0 += 16) {
        bf16x4 av, bv;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            av[i] = (short)a(r, k0 + 4 * g + i);
            bv[i] = (short)b(k0 + 4 * g + i, r);
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, bv, acc, 0, 0, 0);
    }
    return acc;
}

struct Layers {
    int in[4] = {MLP_IN_PAD, MLP_HID, MLP_HID, MLP_HID};
    int out[4] = {MLP_HID, MLP_HID, MLP_HID, MLP_OUT_PAD};
    int w[4] = {MLP_OFF_W1, MLP_OFF_W2, MLP_OFF_W3, MLP_OFF_W4};
    int b[4] = {MLP_OFF_B1, MLP_OFF_B2, MLP_OFF_B3, MLP_OFF_B4};
};

// stage every weight matrix (BF16) of the network in LDS
__device__ void stage_weights(unsigned short *sW, const unsigned short *Wb)
{
    for (int i = threadIdx.x; i < MLP_NPARAM; i += blockDim.x) sW[i] = Wb[i];
}

// ---------------------------------------------------------------------------
// forward: X (B, 10) FP32 -> Y (B, 6) FP32; when cache != null the BF16 layer
// inputs H0 (B, 16), H1..H3 (B, 64) and pre-activations Z1..Z3 (B, 64) are
// kept for the backward pass
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_mlp_forward(const float *__restrict__ X, float *__restrict__ Y,
                                                    const unsigned short *__restrict__ Wb,
                                                    const float *__restrict__ P, long B, MlpCache cache)
{
    __shared__ unsigned short sW[MLP_NPARAM];
    __shared__ unsigned short sH[2][TILE * HS];
    const Layers L;
    const long row0 = (long)blockIdx.x * TILE;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    stage_weights(sW, Wb);
    for (int i = threadIdx.x; i < TILE * MLP_IN_PAD; i += blockDim.x) {
        const int m = i / MLP_IN_PAD, k = i % MLP_IN_PAD;
        const long s = row0 + m;
        const float x = (s < B && k < MLP_IN) ? X[s * MLP_IN + k] : 0.0f;
        const unsigned short hb = to_bf16(x);
        sH[0][m * HS + k] = hb;
        if (cache.H[0] && s < B) cache.H[0][s * MLP_IN_PAD + k] = hb;
    }
    __syncthreads();
    int cur = 0;
    for (int l = 0; l < 4; ++l) {
        const unsigned short *Wl = sW + L.w[l];
        const int K = L.in[l], N = L.out[l];
        const unsigned short *Hc = sH[cur];
        for (int nt = 0; nt < N / 16; ++nt) {
            f32x4 acc = {0, 0, 0, 0};
            acc = mma16([&](int m, int k) { return Hc[(16 * w + m) * HS + k]; },
                        [&](int k, int n) { return Wl[(16 * nt + n) * K + k]; }, K, acc);
            const int col = 16 * nt + r;
            const float bias = P[L.b[l] + col];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = 16 * w + 4 * g + i;
                const long s = row0 + m;
                const float z = acc[i] + bias;
                if (l < 3) {
                    const unsigned short zb = to_bf16(z);
                    const unsigned short hb = to_bf16(gelu_f(from_bf16(zb)));
                    sH[cur ^ 1][m * HS + col] = hb;
                    if (cache.Z[l] && s < B) {
                        cache.Z[l][s * MLP_HID + col] = zb;
                        cache.H[l + 1][s * MLP_HID + col] = hb;
                    }
                } else if (col < MLP_OUT && s < B) {
                    Y[s * MLP_OUT + col] = z;
                }
            }
        }
        __syncthreads();
        cur ^= 1;
    }
}

// ---------------------------------------------------------------------------
// inference forward (no cache): pdo_mlp_dev.hpp on samples in memory, NT
// tiles per wave at a time.  At most 128 registers, so that the matrix
// results stay in vector registers.
// ---------------------------------------------------------------------------
constexpr int INFER_WAVES = 4;  // waves per workgroup
// samples up to which a wave takes one tile, not two: as many tiles as the
// chip has SIMDs.  A launch lasts as long as one wave then: 1000 samples 5.1
// us with one tile and 6.6 with two, 16384 5.3 and 6.7; beyond, two tiles
// share the weights' LDS reads: 65536 10.7 and 9.4.
constexpr long ONE_TILE = 16 * 1024;

template <int NT>
__global__ void __launch_bounds__(64 * INFER_WAVES, 4)
k_mlp_infer(const float *__restrict__ X, float *__restrict__ Y, const unsigned short *__restrict__ Wb,
            const float *__restrict__ P, long B, long ngroups)
{
    __shared__ MlpLds L;
    mlp_stage(L, Wb, P);
    __syncthreads();
    const int lane = threadIdx.x & 63, g = lane >> 4;
    const long stride = (long)gridDim.x * INFER_WAVES;
    for (long t = (long)blockIdx.x * INFER_WAVES + (threadIdx.x >> 6); t < ngroups; t += stride) {
        // keeps the LDS weight reads inside the loop (hoisted, they would
        // occupy the registers the LDS placement is meant to free)
        asm volatile("" ::: "memory");
        u32x2 x[NT];
        f32x4 y[NT];
#pragma unroll
        for (int q = 0; q < NT; ++q) {
            const long s = 16 * (NT * t + q) + (lane & 15);  // this lane's sample
            f32x4 xv = {0, 0, 0, 0};
            if (s < B) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (4 * g + i < MLP_IN) xv[i] = X[s * MLP_IN + 4 * g + i];
            }
            x[q] = (u32x2){pack2(xv[0], xv[1]), pack2(xv[2], xv[3])};
        }
        mlp_eval<NT>(L, x, y);
#pragma unroll
        for (int q = 0; q < NT; ++q) {
            const long s = 16 * (NT * t + q) + (lane & 15);
            // outputs 4 g .. 4 g + 3 of sample s; 6 are used
            if (s < B && g < 2) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (4 * g + i < MLP_OUT) Y[s * MLP_OUT + 4 * g + i] = y[q][i];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// backward: per-workgroup gradient partials of the mean squared error
// loss = mean over B x 6 of (Y - T)^2, or of any loss whose gradient with
// respect to the outputs is dY; partial[blockIdx.x][MLP_NPARAM]
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_mlp_backward(const float *__restrict__ Y, const float *__restrict__ T,
                                                     const float *__restrict__ dY,
                                                     const unsigned short *__restrict__ Wb, long B,
                                                     MlpCache cache, float *__restrict__ partial)
{
    __shared__ unsigned short sW[MLP_NPARAM];
    __shared__ unsigned short sD[TILE * HS];   // dZ (BF16), [sample][feature]
    __shared__ float sDf[TILE * (64 + 1)];     // dZ (FP32) for the bias sums
    __shared__ unsigned short sH[TILE * HS];   // layer input H, [sample][feature]
    __shared__ unsigned short sZ[TILE * HS];   // pre-activation of the layer below
    const Layers L;
    const long row0 = (long)blockIdx.x * TILE;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    float *out = partial + (size_t)blockIdx.x * MLP_NPARAM;
    stage_weights(sW, Wb);
    const float scale = 2.0f / (float)(B * MLP_OUT);
    for (int i = threadIdx.x; i < TILE * MLP_OUT_PAD; i += blockDim.x) {
        const int m = i / MLP_OUT_PAD, n = i % MLP_OUT_PAD;
        const long s = row0 + m;
        // dL/dY: of the mean squared error against T, or given (dY)
        float d = 0.0f;
        if (s < B && n < MLP_OUT)
            d = dY ? dY[s * MLP_OUT + n] : scale * (Y[s * MLP_OUT + n] - T[s * MLP_OUT + n]);
        sDf[m * 65 + n] = d;
        sD[m * HS + n] = to_bf16(d);
    }
    for (int l = 3; l >= 0; --l) {
        const int K = L.in[l], N = L.out[l];
        const unsigned short *Wl = sW + L.w[l];
        // layer input H_l (and Z_l of the layer below, for the GELU derivative)
        const unsigned short *Hg = cache.H[l];
        const unsigned short *Zg = l > 0 ? cache.Z[l - 1] : nullptr;
        for (int i = threadIdx.x; i < TILE * K; i += blockDim.x) {
            const int m = i / K, k = i % K;
            const long s = row0 + m;
            sH[m * HS + k] = s < B ? Hg[s * K + k] : (unsigned short)0;
            if (Zg) sZ[m * HS + k] = s < B ? Zg[s * K + k] : (unsigned short)0;
        }
        __syncthreads();
        // bias gradient: column sums of dZ over the tile
        for (int n = threadIdx.x; n < N; n += blockDim.x) {
            float acc = 0.0f;
            for (int m = 0; m < TILE; ++m) acc += sDf[m * 65 + n];
            out[L.b[l] + n] = acc;
        }
        // weight gradient dW (N x K) = dZ^T (N x TILE) * H (TILE x K)
        for (int t = w; t < (N / 16) * (K / 16); t += 4) {
            const int mt = t / (K / 16), nt = t % (K / 16);
            f32x4 acc = {0, 0, 0, 0};
            acc = mma16([&](int m, int k) { return sD[k * HS + 16 * mt + m]; },
                        [&](int k, int n) { return sH[k * HS + 16 * nt + n]; }, TILE, acc);
#pragma unroll
            for (int i = 0; i < 4; ++i) out[L.w[l] + (16 * mt + 4 * g + i) * K + 16 * nt + r] = acc[i];
        }
        if (l == 0) break;
        // dH (TILE x K) = dZ (TILE x N) * W (N x K); dZ_below = dH * gelu'(Z)
        f32x4 dh[4];
        for (int nt = 0; nt < K / 16; ++nt) {
            f32x4 acc = {0, 0, 0, 0};
            dh[nt] = mma16([&](int m, int k) { return sD[(16 * w + m) * HS + k]; },
                           [&](int k, int n) { return Wl[k * K + 16 * nt + n]; }, N, acc);
        }
        __syncthreads();  // every read of sD / sDf for this layer is done
        for (int nt = 0; nt < K / 16; ++nt) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = 16 * w + 4 * g + i, col = 16 * nt + r;
                const float d = dh[nt][i] * gelu_grad_f(from_bf16(sZ[m * HS + col]));
                sDf[m * 65 + col] = d;
                sD[m * HS + col] = to_bf16(d);
            }
        }
        __syncthreads();
    }
}

// grads[p] = sum over the nblk partials, in block order
__global__ void __launch_bounds__(256) k_mlp_reduce(const float *__restrict__ partial, int nblk, float *grads)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= MLP_NPARAM) return;
    float acc = 0.0f;
    for (int b = 0; b < nblk; ++b) acc += partial[(size_t)b * MLP_NPARAM + p];
    grads[p] = acc;
}

// Adam on the FP32 master parameters, then the BF16 copy used by the kernels
__global__ void __launch_bounds__(256) k_mlp_adam(float *P, float *M, float *V, const float *grads,
                                                 unsigned short *Wb, float lr, float b1, float b2, float eps,
                                                 float c1, float c2)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= MLP_NPARAM) return;
    const float gr = grads[p];
    const float m = b1 * M[p] + (1.0f - b1) * gr;
    const float v = b2 * V[p] + (1.0f - b2) * gr * gr;
    M[p] = m;
    V[p] = v;
    const float np = P[p] - lr * (m / c1) / (sqrtf(v / c2) + eps);
    P[p] = np;
    Wb[p] = to_bf16(np);
}

__global__ void k_mlp_to_bf16(const float *P, unsigned short *Wb)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < MLP_NPARAM) Wb[p] = to_bf16(P[p]);
}

hipError_t resident_blocks(Resident &r, const void *kernel, int threads, int *blocks)
{
    int dev = 0, ncu = 0, per_cu = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const bool kept = dev >= 0 && dev < Resident::MAXDEV;
    if (kept && (*blocks = r.blocks[dev].load(std::memory_order_relaxed)) > 0) return hipSuccess;
    e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, 0);
    if (e != hipSuccess) return e;
    *blocks = ncu * (per_cu > 0 ? per_cu : 1);
    if (kept) r.blocks[dev].store(*blocks, std::memory_order_relaxed);
    return hipSuccess;
}

static unsigned nblocks(long B) { return (unsigned)((B + TILE - 1) / TILE); }

template <int NT>
static hipError_t launch_infer(const float *X, float *Y, const unsigned short *Wb, const float *P, long B, long blocks,
                               hipStream_t st)
{
    const long ngroups = (B + 16 * NT - 1) / (16 * NT);
    const long need = (ngroups + INFER_WAVES - 1) / INFER_WAVES;
    hipLaunchKernelGGL(k_mlp_infer<NT>, dim3((unsigned)(need < blocks ? need : blocks)), dim3(64 * INFER_WAVES), 0, st,
                       X, Y, Wb, P, B, ngroups);
    return hipGetLastError();
}

hipError_t launch_mlp_forward(const float *X, float *Y, const unsigned short *Wb, const float *P, long B,
                              const MlpCache &cache, hipStream_t st)
{
    if (B <= 0) return hipSuccess;
    if (!cache.H[0]) {
        // inference: as many persistent workgroups as are resident at once
        static Resident resident;
        int res = 0;
        const hipError_t e = resident_blocks(resident, (const void *)k_mlp_infer<2>, 64 * INFER_WAVES, &res);
        if (e != hipSuccess) return e;
        return B <= ONE_TILE ? launch_infer<1>(X, Y, Wb, P, B, res, st) : launch_infer<2>(X, Y, Wb, P, B, res, st);
    }
    hipLaunchKernelGGL(k_mlp_forward, dim3(nblocks(B)), dim3(256), 0, st, X, Y, Wb, P, B, cache);
    return hipGetLastError();
}

hipError_t launch_mlp_backward(const float *Y, const float *T, const float *dY, const unsigned short *Wb, long B,
                               const MlpCache &cache, float *partial, float *grads, hipStream_t st)
{
    if (B <= 0) return hipSuccess;
    const unsigned nb = nblocks(B);
    hipLaunchKernelGGL(k_mlp_backward, dim3(nb), dim3(256), 0, st, Y, T, dY, Wb, B, cache, partial);
    hipLaunchKernelGGL(k_mlp_reduce, dim3((MLP_NPARAM + 255) / 256), dim3(256), 0, st, partial, (int)nb, grads);
    return hipGetLastError();
}

hipError_t launch_mlp_adam(float *P, float *M, float *V, const float *grads, unsigned short *Wb, float lr, float b1,
                           float b2, float eps, float c1, float c2, hipStream_t st)
{
    hipLaunchKernelGGL(k_mlp_adam, dim3((MLP_NPARAM + 255) / 256), dim3(256), 0, st, P, M, V, grads, Wb, lr, b1, b2,
                       eps, c1, c2);
    return hipGetLastError();
}

hipError_t launch_mlp_to_bf16(const float *P, unsigned short *Wb, hipStream_t st)
{
    hipLaunchKernelGGL(k_mlp_to_bf16, dim3((MLP_NPARAM + 255) / 256), dim3(256), 0, st, P, Wb);
    return hipGetLastError();
}

}  // namespace pdo
