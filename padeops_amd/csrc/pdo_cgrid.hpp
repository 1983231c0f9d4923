// cgrid compressible right-hand side (pdo_cgrid.cpp) and its pointwise
// kernels (pdo_cgrid.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/padeops_hip.h"

namespace pdo {

enum CgOp {
    CG_PRIMITIVE,   // in W; out prim (7 fields); c: gam - 1, 1 / Rgas
    CG_STRAIN,      // in g (9 fields); out strain-rate magnitude, dilatation
    CG_MUSTAR,      // in X, Y, Z, rho; out; c: Cmu, dx^6, dy^6, dz^6
    CG_BULKSTAR,    // in X, Y, Z, grad rho (3), g, dil, rho; out; c: Cbeta, dx, dy, dz, dx^4, dy^4, dz^4
    CG_KAPSTAR,     // in X, Y, Z, grad e (3), prim; out; c: Ckap, gam, dx, dy, dz, dx^4, dy^4, dz^4
    CG_FLUXES,      // in W, prim, g, star (3), grad e (3); out mu/bulk/kap (3), tau (6), q (3), fluxes (12: 4
                    // per direction); i0 inviscid; c: mu_ref, T_ref, n, Cp, Pr, dT/de
    CG_COPY,        // out = in
};

struct CgArgs {
    const void *in[8] = {};
    void *out[4] = {};
    long n = 0;  // points per field
    int i0 = 0;
    double c[8] = {};
};

hipError_t launch_cgrid(bool dbl, CgOp op, const CgArgs &a, hipStream_t st);

// of the derivatives and filters objects (pdo_dispatch.cpp): independent
// passes along direction d (0, 1, 2), several per launch for small fields
struct DerivTask {
    const void *f;
    void *out;
    int bc1, bcn;
    int sub = 0;  // 2: out -= df, 3: out = -df
};
// order 1 or 2, at most 8 tasks; work holds one field (null without sub)
int derivatives_many(pdo_derivatives h, int d, int order, int prec, const DerivTask *t, int count, void *work,
                     hipStream_t st);
// whether one pass along d can apply the filter twice
bool filters_twice(pdo_filters h, int d, int prec);
// at most 3 fields, the filter applied `times` (1, or 2 where filters_twice) times
int filters_many(pdo_filters h, int d, int prec, const void *const *f, void *const *ff, int count, int times, int bc1,
                 int bcn, hipStream_t st);

}  // namespace pdo
