// Device functions of the eddy-viscosity models.
#pragma once

#include <hip/hip_runtime.h>

namespace pdo {

// S_ij (11 12 13 22 23 33) of the gradient d (eddyViscosity.F90:8-16)
template <typename TC> __device__ __forceinline__ void strain(const TC (&d)[9], TC (&s)[6])
{
    s[0] = d[0];
    s[3] = d[4];
    s[5] = d[8];
    s[1] = (TC)0.5 * (d[1] + d[3]);
    s[2] = (TC)0.5 * (d[2] + d[6]);
    s[4] = (TC)0.5 * (d[5] + d[7]);
}

// the model kernel: 0 Smagorinsky |S|, 1 sigma, 2 AMD (cx, cy, cz)
template <typename TC>
__device__ __forceinline__ TC sgs_viscosity(const TC (&d)[9], const TC (&s)[6], int model, TC cx, TC cy, TC cz)
{
    if (model == 0) {
        TC q = s[0] * s[0];
        q += (TC)2 * (s[1] * s[1]);
        q += (TC)2 * (s[2] * s[2]);
        q += s[3] * s[3];
        q += (TC)2 * (s[4] * s[4]);
        q += s[5] * s[5];
        return sqrt((TC)2 * q);
    } else if (model == 1) {
        // sigma.F90:46-96: singular values of the gradient from the
        // invariants of G = A^T A, nu = s3 (s1 - s2) (s2 - s3) / s1^2,
        // in FP64 for every storage type: the closed-form cubic roots
        // lose about half their digits to cancellation
        using TD = double;
        TD e[9];
#pragma unroll
        for (int c = 0; c < 9; ++c) e[c] = (TD)d[c];
        const TD G11 = e[0] * e[0] + e[3] * e[3] + e[6] * e[6];
        const TD G12 = e[0] * e[1] + e[3] * e[4] + e[6] * e[7];
        const TD G13 = e[0] * e[2] + e[3] * e[5] + e[6] * e[8];
        const TD G22 = e[1] * e[1] + e[4] * e[4] + e[7] * e[7];
        const TD G23 = e[1] * e[2] + e[4] * e[5] + e[7] * e[8];
        const TD G33 = e[2] * e[2] + e[5] * e[5] + e[8] * e[8];
        const TD I1 = G11 + G22 + G33, I1sq = I1 * I1, I1cu = I1sq * I1;
        TD I2 = -G11 * G11 - G22 * G22 - G33 * G33;
        I2 = I2 - (TD)2 * G12 * G12 - (TD)2 * G13 * G13;
        I2 = I2 - (TD)2 * G23 * G23;
        I2 = (TD)0.5 * (I2 + I1sq);
        TD I3 = G11 * (G22 * G33 - G23 * G23);
        I3 = I3 + G12 * (G13 * G23 - G12 * G33);
        I3 = I3 + G13 * (G12 * G23 - G22 * G13);
        TD a1 = I1sq / (TD)9 - I2 / (TD)3;
        a1 = a1 > (TD)0 ? a1 : (TD)0;
        const TD a2 = I1cu / (TD)27 - I1 * I2 / (TD)6 + I3 / (TD)2;
        const TD a1s = sqrt(a1);
        TD ca = a2 / (a1 * a1s + (TD)1e-13);
        ca = ca < (TD)1 ? ca : (TD)1;
        ca = ca > (TD)-1 ? ca : (TD)-1;
        const TD a3 = acos(ca) / (TD)3;
        constexpr TD pi3 = 1.04719755119659774615;
        TD s1sq = I1 / (TD)3 + (TD)2 * a1s * cos(a3);
        s1sq = s1sq > (TD)0 ? s1sq : (TD)0;
        const TD s1 = sqrt(s1sq);
        TD s2 = (TD)-2 * a1s * cos(pi3 + a3) + I1 / (TD)3;
        s2 = sqrt(s2 > (TD)0 ? s2 : (TD)0);
        TD s3 = (TD)-2 * a1s * cos(pi3 - a3) + I1 / (TD)3;
        s3 = sqrt(s3 > (TD)0 ? s3 : (TD)0);
        return (TC)(s3 * (s1 - s2) * (s2 - s3) / (s1sq + (TD)1e-15));
    } else {
        // AMD.F90:43-70: -(C grad u_i . C grad u_j) S_ij / (grad u : grad u)
        auto row = [&](int i, int j) {
            return (d[3 * i] * cx) * (d[3 * j] * cx) + (d[3 * i + 1] * cy) * (d[3 * j + 1] * cy) +
                   (d[3 * i + 2] * cz) * (d[3 * j + 2] * cz);
        };
        TC num = row(0, 0) * s[0];
        num += row(1, 1) * s[3];
        num += row(2, 2) * s[5];
        num += (TC)2 * row(0, 1) * s[1];
        num += (TC)2 * row(0, 2) * s[2];
        num += (TC)2 * row(1, 2) * s[4];
        TC den = 0;
#pragma unroll
        for (int c = 0; c < 9; ++c) den += d[c] * d[c];
        const TC v = -num / (den + (TC)1e-32);
        return v > (TC)0 ? v : (TC)0;
    }
}

}  // namespace pdo
