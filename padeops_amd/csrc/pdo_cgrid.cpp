// The cgrid compressible right-hand side for one species of ideal gas on one
// GPU (src/compressible/cgrid.F90): get_primitive :763-797, getRHS :822-894
// with getRHS_x/y/z :896-1056, getLAD :1058-1257 (artificial shear and bulk
// viscosity and conductivity), filter :1259-1336, get_tau :1360-1404, get_q
// :1406-1452.  Derivatives and filters are the library's derivatives /
// filters objects (derivatives%ddx.., filters%filterx..), so the compact
// solves of the collocated drop-in carry the work; the rest are pointwise
// kernels (pdo_cgrid.hip).  All fields live in device memory for the life of
// the object.
#include <algorithm>
#include <cmath>
#include <vector>

#include "../../include/padeops_hip.h"
#include "pdo_cgrid.hpp"
#include "pdo_ops.hpp"

namespace pdo {

// work field indices (each n words of the storage type)
enum {
    F_PRIM = 0,            // rho u v w e p T
    F_G = F_PRIM + 7,      // du_i/dx_j at 3 i + j
    F_MU = F_G + 9,        // mu, bulk, kap (physical + artificial)
    F_TAU = F_MU + 3,      // xx xy xz yy yz zz
    F_Q = F_TAU + 6,       // qx qy qz
    F_STAR = F_Q + 3,      // mustar, bulkstar, kapstar
    F_DE = F_STAR + 3,     // gradient of e
    // of the artificial coefficients alone: the fluxes overlie them
    F_DRHO = F_DE + 3,     // gradient of rho
    F_FUNC = F_DRHO + 3,   // strain-rate magnitude
    F_DIL = F_FUNC + 1,    // dilatation
    F_PASS = F_DIL + 1,    // fields of the coefficients formed together
    F_FLUX = F_DRHO        // momentum and energy fluxes, four per direction
};
// of each coefficient formed at a time: a second derivative, the fourth
// derivatives along x, y, z, and two filter buffers
enum { P_T1 = 0, P_D4 = P_T1 + 1, P_FIL = P_D4 + 3, P_COUNT = P_FIL + 2 };

struct CgridObject {
    pdo_cgrid_params p{};
    int prec = PDO_F64;
    size_t W = 8;
    long n = 0;
    pdo_derivatives der = nullptr;
    pdo_filters fil = nullptr, gfil = nullptr;
    int together = 1;  // artificial coefficients formed at a time: 1 or 3
    void *buf = nullptr;
    ~CgridObject()
    {
        if (der) pdo_derivatives_destroy(der);
        if (fil) pdo_filters_destroy(fil);
        if (gfil) pdo_filters_destroy(gfil);
        if (buf) (void)hipFree(buf);
    }
    void *f(int i) { return (char *)buf + (size_t)i * n * W; }
    // of the q-th coefficient of those formed together
    void *pass(int q, int i) { return f(F_PASS + q * P_COUNT + i); }
    // 46 fields, 57 with the three coefficients together
    int fields() const { return std::max(F_PASS + together * P_COUNT, F_FLUX + 12); }
};

}  // namespace pdo

struct pdo_cgrid_s : public pdo::CgridObject {};

using namespace pdo;

namespace {

#define PDO_TRY(x)                   \
    do {                             \
        if (int r_ = (x)) return r_; \
    } while (0)

int cg(pdo_cgrid h, CgOp op, const CgArgs &a, hipStream_t st)
{
    hipError_t e = launch_cgrid(h->W == 8, op, a, st);
    return e == hipSuccess ? 0 : hip_fail(e, "cgrid kernel");
}

const int *bc_of(pdo_cgrid h, int d) { return d == 0 ? h->p.x_bc : (d == 1 ? h->p.y_bc : h->p.z_bc); }

// the fourth derivatives along each direction (two second-derivative passes)
// of count functions f
int fourth(pdo_cgrid h, const void *const *f, int count, hipStream_t st)
{
    for (int d = 0; d < 3; d++) {
        const int *b = bc_of(h, d);
        DerivTask t[3];
        for (int q = 0; q < count; q++) t[q] = {f[q], h->pass(q, P_T1), b[0], b[1]};
        PDO_TRY(derivatives_many(h->der, d, 2, h->prec, t, count, nullptr, st));
        for (int q = 0; q < count; q++) t[q] = {h->pass(q, P_T1), h->pass(q, P_D4 + d), b[0], b[1]};
        PDO_TRY(derivatives_many(h->der, d, 2, h->prec, t, count, nullptr, st));
    }
    return 0;
}

// filter (cgrid.F90:1259-1336): numtimes passes along y, then x, then z, in
// place on each of arr[0 .. count), through two buffers each.  Two
// applications along a direction go together where the filter can.
int filter3(pdo_cgrid h, pdo_filters fl, void *const *arr, int count, int numtimes, hipStream_t st)
{
    const int order[3] = {1, 0, 2};
    int total = 0;
    for (int d : order) total += filters_twice(fl, d, h->prec) ? (numtimes + 1) / 2 : numtimes;
    void *cur[3];
    for (int k = 0; k < count; k++) cur[k] = arr[k];
    int pass = 0, buf = 0;
    for (int d : order) {
        const int *b = bc_of(h, d);
        const bool two = filters_twice(fl, d, h->prec);
        for (int left = numtimes; left > 0; pass++) {
            const int times = two && left > 1 ? 2 : 1;
            // out of place: the last pass writes arr unless it also reads it
            const bool home = pass == total - 1 && cur[0] != arr[0];
            void *dst[3];
            for (int k = 0; k < count; k++) dst[k] = home ? arr[k] : h->pass(k, P_FIL + buf);
            PDO_TRY(filters_many(fl, d, h->prec, cur, dst, count, times, b[0], b[1], st));
            for (int k = 0; k < count; k++) cur[k] = dst[k];
            buf ^= 1;
            left -= times;
        }
    }
    for (int k = 0; k < count; k++) {
        if (cur[k] == arr[k]) continue;
        CgArgs a;
        a.in[0] = cur[k];
        a.out[0] = arr[k];
        a.n = h->n;
        PDO_TRY(cg(h, CG_COPY, a, st));
    }
    return 0;
}

// getLAD (cgrid.F90:1058-1257), one species: the filtered artificial shear
// and bulk viscosity and conductivity into F_STAR
int lad(pdo_cgrid h, hipStream_t st)
{
    const pdo_cgrid_params &p = h->p;
    const double dx = p.dx, dy = p.dy, dz = p.dz;
    const double dx2 = dx * dx, dy2 = dy * dy, dz2 = dz * dz;
    const double dx4 = dx2 * dx2, dy4 = dy2 * dy2, dz4 = dz2 * dz2;
    const long n = h->n;
    CgArgs a;
    a.in[0] = h->f(F_G);
    a.out[0] = h->f(F_FUNC);
    a.out[1] = h->f(F_DIL);
    a.n = n;
    PDO_TRY(cg(h, CG_STRAIN, a, st));
    const void *const func[3] = {h->f(F_FUNC), h->f(F_DIL), h->f(F_PRIM + 4)};
    // coefficient k, the q-th of those formed together
    auto star = [&](int k, int q) -> int {
        CgArgs c;
        for (int d = 0; d < 3; d++) c.in[d] = h->pass(q, P_D4 + d);
        c.out[0] = h->f(F_STAR + k);
        c.n = n;
        if (k == 0) {
            c.in[3] = h->f(F_PRIM);
            const double v[4] = {p.Cmu, dx4 * dx2, dy4 * dy2, dz4 * dz2};
            for (int i = 0; i < 4; i++) c.c[i] = v[i];
            return cg(h, CG_MUSTAR, c, st);
        }
        if (k == 1) {
            c.in[3] = h->f(F_DRHO);
            c.in[4] = h->f(F_G);
            c.in[5] = h->f(F_DIL);
            c.in[6] = h->f(F_PRIM);
            const double v[7] = {p.Cbeta, dx, dy, dz, dx4, dy4, dz4};
            for (int i = 0; i < 7; i++) c.c[i] = v[i];
            return cg(h, CG_BULKSTAR, c, st);
        }
        c.in[3] = h->f(F_DE);
        c.in[4] = h->f(F_PRIM);
        const double v[8] = {p.Ckap, p.gam, dx, dy, dz, dx4, dy4, dz4};
        for (int i = 0; i < 8; i++) c.c[i] = v[i];
        return cg(h, CG_KAPSTAR, c, st);
    };
    // small fields: the three coefficients' passes share launches; others:
    // one coefficient after the other, so that a pass finds what the last one
    // wrote in the Infinity Cache
    const int step = h->together;
    for (int k = 0; k < 3; k += step) {
        PDO_TRY(fourth(h, func + k, step, st));
        void *s[3];
        for (int q = 0; q < step; q++) {
            PDO_TRY(star(k + q, q));
            s[q] = h->f(F_STAR + k + q);
        }
        PDO_TRY(filter3(h, h->gfil, s, step, 2, st));
    }
    return 0;
}

}  // namespace

extern "C" {

int pdo_cgrid_init(pdo_cgrid *out, const pdo_cgrid_params *p, int prec)
{
    if (!out || !p) { set_error("invalid argument"); return PDO_ERR_ARG; }
    *out = nullptr;
    if (prec_mode(prec) < 0) { set_error("unknown precision mode"); return PDO_ERR_ARG; }
    if (p->nx < 1 || p->ny < 1 || p->nz < 1 || !(p->dx > 0) || !(p->dy > 0) || !(p->dz > 0)) {
        set_error("cgrid: sizes and spacings must be positive");
        return PDO_ERR_ARG;
    }
    if (!(p->gam > 1) || !(p->Rgas > 0) || (!p->inviscid && (!(p->T_ref > 0) || !(p->Pr > 0)))) {
        set_error("cgrid: need gam > 1, Rgas > 0 and, when viscous, T_ref > 0 and Pr > 0");
        return PDO_ERR_ARG;
    }
    auto *h = new pdo_cgrid_s();
    h->p = *p;
    h->prec = prec;
    h->W = prec == PDO_F64 ? 8 : 4;
    h->n = (long)p->nx * p->ny * p->nz;
    int st = pdo_derivatives_init(&h->der, p->nx, p->ny, p->nz, p->dx, p->dy, p->dz, p->periodic, p->derivative);
    if (!st) st = pdo_filters_init(&h->fil, p->nx, p->ny, p->nz, p->periodic, p->filter);
    const int gauss[3] = {2, 2, 2};
    if (!st) st = pdo_filters_init(&h->gfil, p->nx, p->ny, p->nz, p->periodic, gauss);
    if (st) { delete h; return st; }
    h->together = small_field(h->n, prec) ? 3 : 1;
    hipError_t e = hipMalloc(&h->buf, (size_t)h->fields() * h->n * h->W);
    if (e != hipSuccess) { delete h; return hip_fail(e, "hipMalloc(cgrid work)"); }
    *out = h;
    return 0;
}

int pdo_cgrid_rhs(pdo_cgrid h, int prec, const void *Wc, void *rhs, void *stream)
{
    if (!h || !Wc || !rhs) { set_error("invalid argument"); return PDO_ERR_ARG; }
    if (prec != h->prec) { set_error("cgrid: the object's work buffers were sized for another precision"); return PDO_ERR_ARG; }
    hipStream_t st = (hipStream_t)stream;
    const pdo_cgrid_params &p = h->p;
    const long n = h->n;
    // get_primitive
    {
        CgArgs a;
        a.in[0] = Wc;
        a.out[0] = h->f(F_PRIM);
        a.n = n;
        a.c[0] = p.gam - 1.0;
        a.c[1] = 1.0 / p.Rgas;
        PDO_TRY(cg(h, CG_PRIMITIVE, a, st));
    }
    // gradients (cgrid.F90:446-480) of u, v, w, rho and e: antisymmetric ends
    // for u along x, v along y and w along z
    for (int d = 0; d < 3; d++) {
        const int *b = bc_of(h, d);
        DerivTask t[5];
        for (int c = 0; c < 3; c++) {
            const int sg = c == d ? -1 : 1;
            t[c] = {h->f(F_PRIM + 1 + c), h->f(F_G + 3 * c + d), sg * b[0], sg * b[1]};
        }
        t[3] = {h->f(F_PRIM), h->f(F_DRHO + d), b[0], b[1]};
        t[4] = {h->f(F_PRIM + 4), h->f(F_DE + d), b[0], b[1]};
        PDO_TRY(derivatives_many(h->der, d, 1, h->prec, t, 5, nullptr, st));
    }
    PDO_TRY(lad(h, st));
    // transport properties, tau, q and the fluxes along every direction
    {
        CgArgs a;
        a.in[0] = Wc;
        a.in[1] = h->f(F_PRIM);
        a.in[2] = h->f(F_G);
        a.in[3] = h->f(F_STAR);
        a.in[4] = h->f(F_DE);
        a.out[0] = h->f(F_MU);
        a.out[1] = h->f(F_TAU);
        a.out[2] = h->f(F_Q);
        a.out[3] = h->f(F_FLUX);
        a.n = n;
        a.i0 = p.inviscid;
        a.c[0] = p.mu_ref;
        a.c[1] = p.T_ref;
        a.c[2] = p.visc_n;
        a.c[3] = p.gam * p.Rgas * (1.0 / (p.gam - 1.0));
        a.c[4] = p.Pr;
        a.c[5] = (p.gam - 1.0) * (1.0 / p.Rgas);
        PDO_TRY(cg(h, CG_FLUXES, a, st));
    }
    // rhs = -sum_d d/dx_d (fluxes along d): symmetric ends for the momentum
    // along d, antisymmetric for the others
    for (int d = 0; d < 3; d++) {
        const int *b = bc_of(h, d);
        DerivTask t[5];
        for (int c = 0; c < 5; c++) {
            const int sg = c == 1 + d ? 1 : -1;
            // the mass flux is the momentum
            const void *f = c == 0 ? (const char *)Wc + (size_t)(1 + d) * n * h->W : h->f(F_FLUX + 4 * d + c - 1);
            t[c] = {f, (char *)rhs + (size_t)c * n * h->W, sg * b[0], sg * b[1], d == 0 ? 3 : 2};
        }
        PDO_TRY(derivatives_many(h->der, d, 1, h->prec, t, 5, h->f(F_STAR), st));
    }
    return 0;
}

int pdo_cgrid_filter(pdo_cgrid h, int prec, void *arr, int numtimes, int gaussian, void *stream)
{
    if (!h || !arr || numtimes < 1) { set_error("invalid argument"); return PDO_ERR_ARG; }
    if (prec != h->prec) { set_error("cgrid: the object's work buffers were sized for another precision"); return PDO_ERR_ARG; }
    return filter3(h, gaussian ? h->gfil : h->fil, &arr, 1, numtimes, (hipStream_t)stream);
}

int pdo_cgrid_field(pdo_cgrid h, int which, const void **ptr)
{
    if (!h || !ptr || which < 0 || which > 12) { set_error("invalid argument"); return PDO_ERR_ARG; }
    static const int base[13] = {F_PRIM,     F_PRIM + 1, F_PRIM + 2, F_PRIM + 3, F_PRIM + 4, F_PRIM + 5, F_PRIM + 6,
                                 F_MU,       F_MU + 1,   F_MU + 2,   F_G,        F_TAU,      F_Q};
    *ptr = h->f(base[which]);
    return 0;
}

int pdo_cgrid_destroy(pdo_cgrid h)
{
    delete h;
    return 0;
}

}  // extern "C"
