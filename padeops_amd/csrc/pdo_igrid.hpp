// Pointwise kernels of the igrid pieces (pdo_igrid.hip).  mode: 0 FP64,
// 1 FP32, 2 FP32 storage with FP64 arithmetic (as the spectral objects).
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/padeops_hip.h"

namespace pdo {

// plane 0 of a spectrum of nplane complex values per plane: zero, except the
// mean mode, which is set to v
hipError_t launch_surface_plane(int mode, void *f, long nplane, double v, hipStream_t st);
// f[k nplane] += v (the real part of the mean mode of each of nz planes of
// a spectrum with nplane complex values per plane)
hipError_t launch_mean_add(int mode, void *f, long nplane, int nz, double v, hipStream_t st);
// subgrid terms of one set of points: nu from the gradients g (9 components n
// apart) and the model constant (cplane per plane of nxy points, or cglobal),
// and tau = -2 nu S: on cells 11, 12, 22, 33; on edges 13, 23
hipError_t launch_sgs_tau(int mode, bool edges, const void *g, void *nu, void *tau, long n, long nxy, int model,
                          const double (&camd)[3], const double *cplane, double cglobal, hipStream_t st);
// edges, nu given: nu = max(nu, 0) with clip, and tau
hipError_t launch_edge_tau(int mode, bool clip, const void *g, void *nu, void *tau, long n, hipStream_t st);
// divergence of the stress from its spectra: u -= i k1 t11 + i k2 t12 + z13,
// v -= i k1 t12 + i k2 t22 + z23 (cells), w -= z33 + i k1 t13 + i k2 t23
// (edges); complex, cells ncell values, edges nedge
struct StressSpectra {
    const void *t11, *t12, *t22, *z13, *z23, *z33, *t13, *t23;
};
hipError_t launch_stress_div(int mode, void *u, void *v, void *w, const StressSpectra &S, const double *k1,
                             const double *k2, int nxh, int ny, long ncell, long nedge, hipStream_t st);

// rhs[c] += s[c] (c = 0, 1; null: nothing) + invRe (-(k1^2 + k2^2) f[c] + d2[c])
// (invRe 0: nothing), c = 0, 1 on cells, 2 on edges; complex
struct RhsTerms {
    void *rhs[3];
    const void *s[3], *f[3], *d2[3];
};
hipError_t launch_rhs_terms(int mode, const RhsTerms &T, const double *k1, const double *k2, int nxh, int ny,
                            long ncell, long nedge, double invRe, hipStream_t st);
// out[c] = (coef[0] x[0][c] + ... + coef[nterms-1] x[nterms-1][c], left to
// right) g1[kx] g2[ky], components c = 0, 1 on cells, 2 on edges; complex
struct StageTerms {
    void *out[3];
    const void *x[5][3];
    double coef[5];
    int nterms;
};
hipError_t launch_stage(int mode, const StageTerms &T, const double *g1, const double *g2, int nxh, int ny, long ncell,
                        long nedge, hipStream_t st);
// partial[b] = max over block b of |u|/dx + |v|/dy + |w|/dz (nblocks blocks)
hipError_t launch_cfl(int mode, const void *u, const void *v, const void *w, long n, double idx, double idy,
                      double idz, double *partial, int nblocks, hipStream_t st);

// Moeng wall model (wallmodel.F90:33-86, 106-134, 162-199 unstratified):
// sums of sqrt(u^2 + v^2) and u over the first cell plane (nxy points of u,
// v) in nb blocks, then wm = {Uspmn, ustar, WallMFactor, Umn} with
// Uspmn = sum / nxy, ustar = Uspmn kappa / lg (lg = log(dz / 2 / z0)),
// WallMFactor = -ustar^2 / (Uspmn + 1e-13), and on the bottom edge plane of
// tauE (13 at 0, 23 at nE) tau13 = WallMFactor u, tau23 = WallMFactor v.
// part holds 2 nb doubles; the sums run in a fixed order.
hipError_t launch_wall_model(int mode, const void *u, const void *v, void *tauE, long nxy, long nE, double *part,
                             int nb, double kappa, double lg, double *wm, hipStream_t st);
// whether a Pade6stagg object is periodic (pdo_pade6.cpp)
bool pade6stagg_periodic(pdo_pade6stagg h);
// independent pdo_pade6stagg_apply calls on complex (n1, n2) lines, those of
// one kind sharing launches for small fields (at most 8)
struct StaggTask {
    int kind, bot, top;
    const void *in;
    void *out;
};
int pade6stagg_many(pdo_pade6stagg h, const StaggTask *t, int count, int prec, int n1, int n2, hipStream_t st);

struct BandLimit;
// interp_PrimitiveVars and compute_duidxj of dealiased spectra in one go: the
// physical fields, their gradients and the second derivatives; I.uE etc. as
// in those, with u, v, w the physical velocity too.  The gradient spectra
// (duidxjChat, duidxjEhat) are work here and do not come back.
int igrid_fields(pdo_duidxj h, int prec, const pdo_interp_fields &I, const pdo_duidxj_fields &D, void *u, void *v,
                 void *w, const BandLimit &bl, hipStream_t st);

struct HitForcingArgs {
    int nxh, ny, nz, nwaves;
    double kmin, kmax, eps, normfact, dz;
    unsigned long long seed, draw;
    const double *k3;  // device: GetWaveNums(nz, dz)
};
// HIT_shell_forcing on the spectra (uhat, vhat: nz planes; what: nz+1)
hipError_t launch_hit_forcing(int mode, const void *uhat, const void *vhat, const void *what, void *urhs, void *vrhs,
                              void *wrhs, const HitForcingArgs &F, hipStream_t st);

}  // namespace pdo
