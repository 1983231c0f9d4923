// Compact-operator objects and the C ABI of cd06 / cd10 / cf90 / cd06stagg.
#include "pdo_ops.hpp"

#include <cstdint>
#include <algorithm>
#include <cstring>
#include <vector>

#include "../../include/padeops_hip.h"

namespace pdo {

static thread_local std::string g_err;
void set_error(const std::string &msg) { g_err = msg; }
const char *last_error() { return g_err.c_str(); }

int hip_fail(hipError_t e, const char *what)
{
    set_error(std::string(what) + ": " + hipGetErrorString(e));
    return PDO_ERR_HIP;
}

Variant::~Variant()
{
    if (mem) (void)hipFree(mem);
}

std::vector<double> TabSet::pack()
{
    const SpikeTables &t = tab;
    std::vector<double> all;
    o_fac = 0; all.insert(all.end(), t.fac.begin(), t.fac.end());
    o_spk = (int)all.size(); all.insert(all.end(), t.spk.begin(), t.spk.end());
    o_lhs = (int)all.size(); all.insert(all.end(), t.lhs.begin(), t.lhs.end());
    o_G = (int)all.size(); all.insert(all.end(), t.G.begin(), t.G.end());
    o_sp = (int)all.size(); all.insert(all.end(), t.sp.begin(), t.sp.end());
    return all;
}

// every table of the variant in one device buffer, by one copy: the FP64
// tables, then the FP32 copies of the partitioned ones
int Variant::upload()
{
    std::vector<double> a = fast.pack(), g, o;
    const bool single = !fast.tab.general;
    if (single) g = gen.pack();
    if (ovl.P > 0) {
        // per segment type: lower factors, pivots and upper factors, spikes
        const int K = ovl.K, m = ovl.m;
        for (int ty = 0; ty < 4; ty++) {
            const double *F = &ovl.fac[ty * m * 5], *S = &ovl.spk[ty * m * 4];
            for (int j = 0; j < m; j++) o.insert(o.end(), F + j * 5, F + j * 5 + K);
            for (int j = 0; j < m; j++) o.insert(o.end(), F + j * 5 + 2, F + j * 5 + 3 + K);
            for (int j = 0; j < m; j++) {
                o.insert(o.end(), S + j * 4, S + j * 4 + K);
                o.insert(o.end(), S + j * 4 + 2, S + j * 4 + 2 + K);
            }
        }
        ov_G = (int)o.size(); o.insert(o.end(), ovl.G.begin(), ovl.G.end());
        ov_sp = (int)o.size(); o.insert(o.end(), ovl.sp.begin(), ovl.sp.end());
    }
    // each set starts on a 256-byte boundary, as allocations of its own would
    auto up = [](size_t words) { return (words + 31) & ~(size_t)31; };
    const size_t wa = up(a.size()), wg = up(g.size()), wo = up(o.size()), wf = up((a.size() + 1) / 2);
    std::vector<double> host(wa + wg + wo + wf, 0.0);
    std::copy(a.begin(), a.end(), host.begin());
    std::copy(g.begin(), g.end(), host.begin() + wa);
    std::copy(o.begin(), o.end(), host.begin() + wa + wg);
    const std::vector<float> f(a.begin(), a.end());
    std::memcpy(host.data() + wa + wg + wo, f.data(), f.size() * sizeof(float));
    hipError_t e = hipMalloc(&mem, host.size() * sizeof(double));
    if (e != hipSuccess) return hip_fail(e, "hipMalloc(tables)");
    e = hipMemcpy(mem, host.data(), host.size() * sizeof(double), hipMemcpyHostToDevice);
    if (e != hipSuccess) return hip_fail(e, "hipMemcpy(tables)");
    double *d = (double *)mem;
    fast.d_tab = d;
    fast.f_tab = (float *)(d + wa + wg + wo);
    fast.ready = true;
    if (single) {
        gen.d_tab = d + wa;
        gen.ready = true;
    }
    d_ovl = d + wa + wg;
    return 0;
}

static int build_desc(const OpObject &o, int kind, int bc1, int bcn, SystemDesc &s)
{
    if (o.scheme == SCHEME_CF90 && kind == KIND_FILTER + 1000) {
        // complex filter3: RHS closures of (bc1, bcn), LHS of the (0,0) system
        // (cf90.F90:1245-1248)
        SystemDesc nn;
        int st = build_cf90(nn, o.n, false, 0, 0);
        if (st) return st;
        st = build_cf90(s, o.n, false, bc1, bcn);
        if (st) return st;
        s.lhs = nn.lhs;
        return 0;
    }
    switch (o.scheme) {
    case SCHEME_CD06: return build_cd06(s, kind, o.n, o.dx, o.periodic, o.bc1, o.bcn);
    case SCHEME_CD10: return build_cd10(s, kind, o.n, o.dx, o.periodic, o.periodic ? 0 : bc1, o.periodic ? 0 : bcn);
    case SCHEME_CF90: return build_cf90(s, o.n, o.periodic, o.periodic ? 0 : bc1, o.periodic ? 0 : bcn);
    case SCHEME_CD06STAGG:
        if (o.periodic) {
            // the collocated first derivatives exist only in the non-periodic
            // object (cd06stagg.F90:883-925 read its Tri tables)
            if (kind == KIND_STG_D1_C2C || kind == KIND_STG_D1_E2E) return PDO_ERR_UNSUP;
            return build_stagg_periodic(s, kind, o.n, o.dx);
        }
        return build_stagg_nonperiodic(s, kind, o.n, o.dx, o.flags);
    }
    return PDO_ERR_ARG;
}

Variant *OpObject::find_variant(int kind, int b1, int bn)
{
    if (periodic) b1 = bn = 0;
    const int key = kind * 100 + (b1 + 1) * 10 + (bn + 1);
    std::lock_guard<std::mutex> lk(mu);
    auto it = variants.find(key);
    return it == variants.end() ? nullptr : it->second.get();
}

int OpObject::variant(int kind, int b1, int bn, Variant **out)
{
    if (periodic) b1 = bn = 0;  // periodic systems ignore the boundary flags
    const int key = kind * 100 + (b1 + 1) * 10 + (bn + 1);
    std::lock_guard<std::mutex> lk(mu);
    auto it = variants.find(key);
    if (it != variants.end()) { *out = it->second.get(); return 0; }
    auto v = std::make_unique<Variant>();
    int st = build_desc(*this, kind, b1, bn, v->sys);
    if (st) {
        if (st == PDO_ERR_UNSUP) set_error("operator variant not implemented by the reference");
        return st;
    }
    st = build_spike(v->sys, v->fast.tab);
    if (st) { set_error("failed to build the partitioned-solve tables"); return PDO_ERR_ARG; }
    // the single-segment tables of the general kernel and those of the
    // overlapping segments too (a few KB), so that every shape the variant
    // can take is ready once the variant exists
    if (!v->fast.tab.general && build_spike(v->sys, v->gen.tab, true)) {
        set_error("failed to build tables");
        return PDO_ERR_ARG;
    }
    build_overlap(v->sys, v->ovl);
    if ((st = v->upload())) return st;
    *out = v.get();
    variants[key] = std::move(v);
    return 0;
}

int prec_mode(int prec)
{
    switch (prec) {
    case PDO_F64: return MODE_F64;
    case PDO_F32_REFINE: return MODE_F32R;
    case PDO_F32_STORE: return MODE_F32S;
    case PDO_F32: return MODE_F32;
    }
    return -1;
}

// whether the overlapping-segment kernels take a call
static bool overlap_fits(const Variant &v, int dir, long na, long nb, size_t word)
{
    const SystemDesc &s = v.sys;
    const OverlapTables &o = v.ovl;
    const FamShape f = family_shape(s.family);
    if (o.P <= 0) return false;
    if (dir == 1) {
        if (f.shift != 0 || s.n_in != s.n_sys || s.n_out != s.n_sys) return false;
        // at least 8 pencils fit a workgroup's LDS, with the exchange values and tables
        const size_t pen = (size_t)(s.n_sys | 1) * word + (size_t)o.P * 2 * o.K * 8;
        return 8 * pen + (s.periodic ? 0 : 3 * (size_t)o.m * 9 * 8) + 4 * 1024 <= 160 * 1024 &&
               (size_t)na * nb < ((size_t)1 << 31);
    }
    if (o.P > PMAX && (f.shift != 0 || o.m != MAXM)) return false;
    // pencils are addressed by 32-bit byte offsets within the field, or
    // within one plane of a larger one
    const size_t nmax = (size_t)std::max(std::max(s.n_in, s.n_out), s.n_sys + 1);
    const size_t lim = (size_t)1 << 32;
    if ((size_t)na * nb * nmax * word < lim) return true;
    if (o.P > PMAX) return false;
    return dir == 3 ? (size_t)na * nb * word < lim : ((size_t)na * word < lim && nb <= 65535);
}

// Validate one apply call and fill its launch arguments; *empty is set when
// there is nothing to do (na or nb zero).
static int prepare(OpObject *op, int kind, int bc1, int bcn, int dir, int prec, const void *f, void *out, long na,
                   long nb, int epi, const void *aux, int force_shape, bool several, ApplyArgs &A, int &shape, int &mode,
                   int &family, size_t &scratch_elems, bool *empty, bool noalloc = false)
{
    *empty = false;
    if (!op || !f || !out || na < 0 || nb < 0 || dir < 1 || dir > 3) {
        set_error("invalid argument");
        return PDO_ERR_ARG;
    }
    mode = prec_mode(prec);
    if (mode < 0) { set_error("unknown precision mode"); return PDO_ERR_ARG; }
    if ((epi == 1 || epi == 2) && !aux) { set_error("epilogue without operand"); return PDO_ERR_ARG; }
    if (na == 0 || nb == 0) { *empty = true; return 0; }
    Variant *v = nullptr;
    int st = 0;
    if (noalloc) {
        // building a variant uploads its tables (device allocations)
        if (!(v = op->find_variant(kind, bc1, bcn))) {
            set_error("operator variant not built yet: one call of the allocating entry point with this handle, "
                      "kind and boundary flags builds it");
            return PDO_ERR_ARG;
        }
    } else if ((st = op->variant(kind, bc1, bcn, &v))) {
        return st;
    }
    const SystemDesc &s = v->sys;
    long A_na, A_nb;
    if (dir == 1) { A_na = na; A_nb = nb; shape = SHAPE_X; }
    else if (dir == 2) { A_na = na; A_nb = nb; shape = SHAPE_STRIDED; }
    else { A_na = na * nb; A_nb = 1; shape = SHAPE_STRIDED; }
    // non-periodic x pencils and sizes outside the register path use the
    // single-pencil kernel
    // the x kernel stages whole pencils in LDS with 16-byte accesses: periodic
    // collocated systems, n a power of two, aligned buffers
    auto aligned = [](const void *p) { return p == nullptr || ((uintptr_t)p & 15) == 0; };
    if (shape == SHAPE_X && ((s.n_in & (s.n_in - 1)) != 0 || !aligned(f) || !aligned(out) || !aligned(aux)))
        shape = SHAPE_GENERAL;
    if (v->fast.tab.general || (shape == SHAPE_X && (!s.periodic || s.family >= FAM_STG_E2C_A)) ||
        force_shape == SHAPE_GENERAL)
        shape = SHAPE_GENERAL;
    // the strided kernel addresses a field with 32-bit byte offsets
    const size_t word = (mode == MODE_F64) ? 8 : 4;
    const size_t nmax = (size_t)std::max(std::max(s.n_in, s.n_out), s.n_sys + 1);
    if (shape == SHAPE_STRIDED && (size_t)na * (size_t)nb * nmax * word >= ((size_t)1 << 32)) shape = SHAPE_GENERAL;
    // the register path's non-periodic kernels take no epilogue operand, and
    // an extra row in the last segment only in the tridiagonal families
    if (shape == SHAPE_STRIDED && !s.periodic && (epi || (v->fast.tab.xr && family_shape(s.family).K != 1)))
        shape = SHAPE_GENERAL;
    // only the first derivatives of cd06 and cd10 have epilogues there
    const bool epi_ok = !epi || s.family == FAM_CD06_D1 || s.family == FAM_CD10_D1;
    // sizes and ends without a register kernel of their own: overlapping
    // segments, where they fit (n >= 16, at most 512 rows, 1024 of the
    // collocated operators), else one lane per pencil
    scratch_elems = (shape == SHAPE_GENERAL) ? (size_t)s.n_sys * (size_t)(na * nb) : 0;
    if (shape == SHAPE_GENERAL && force_shape != SHAPE_GENERAL && epi_ok &&
        overlap_fits(*v, dir, na, nb, word))
        shape = dir == 1 ? SHAPE_OVL_X : SHAPE_OVL_STRIDED;
    // FP32 + refinement without periodicity: the refined kernels carry two
    // solves and closure rows in up to 149 registers and scratch, the
    // overlapping segments one FP64 solve (512 x 512 x 256 FP32, along z: cd10
    // 287 -> 160 us, cf90 298 -> 163, 257-row staggered systems 231 -> 174,
    // cd06 131 -> 134; 512^3: cd06 317 -> 258).  FP64 passes stay (cd10 216
    // against 257 us), and so do periodic ones (cd10 150 against 166).
    if (shape == SHAPE_STRIDED && !s.periodic && mode == MODE_F32R && v->ovl.P <= PMAX &&
        overlap_fits(*v, dir, na, nb, word))
        shape = SHAPE_OVL_STRIDED;
    // several refined pentadiagonal passes over a small field: the register
    // kernels have no launch of several passes (can_batch)
    if (several && (shape == SHAPE_STRIDED || shape == SHAPE_X) && mode == MODE_F32R &&
        !can_batch(family_shape(s.family).K, mode) && v->ovl.P <= PMAX && epi_ok &&
        small_field(s.n_sys * na * nb, prec) && overlap_fits(*v, dir, na, nb, word))
        shape = dir == 1 ? SHAPE_OVL_X : SHAPE_OVL_STRIDED;
    TabSet *ts = &v->fast;
    if (shape == SHAPE_GENERAL && !v->fast.tab.general) {
        // built with the variant
        if (!v->gen.ready) { set_error("single-segment tables missing"); return PDO_ERR_ARG; }
        ts = &v->gen;
    }
    const SpikeTables &t = ts->tab;
    std::memset(&A, 0, sizeof(A));
    family = s.family;
    A.f = f; A.out = out; A.aux = aux; A.epi = epi;
    A.periodic = s.periodic ? 1 : 0;
    A.n_sys = s.n_sys; A.n_in = s.n_in; A.n_out = s.n_out;
    A.n_read = (s.family == FAM_STG_E2C_A || s.family == FAM_STG_E2C_S) ? s.n_sys + 1 : s.n_sys;
    A.m = t.m; A.P = t.P; A.xr = t.xr; A.nbl = t.nbl; A.nbr = t.nbr; A.wb = t.wb;
    A.D32 = t.D32; A.D64 = t.D64; A.D32R = t.D32R; A.D32C = t.D32C;
    A.lgn = 0;
    while ((1 << A.lgn) < s.n_in) A.lgn++;
    A.tab_d = ts->d_tab; A.tab_f = ts->f_tab;
    A.o_fac = ts->o_fac; A.o_spk = ts->o_spk; A.o_lhs = ts->o_lhs; A.o_G = ts->o_G; A.o_sp = ts->o_sp;
    for (int q = 0; q < 5; q++) A.c[q] = s.c[q];
    for (int q = 0; q < 5; q++) A.band[q] = s.lhs[s.n_sys / 2][q];
    A.na = A_na; A.nb = A_nb;
    if (dir == 1) {
        // f(n, na, nb): pencil (a,b) at (a + na*b)*n
        A.sa_in = s.n_in; A.sb_in = (long)s.n_in * na; A.se_in = 1;
        A.sa_out = s.n_out; A.sb_out = (long)s.n_out * na; A.se_out = 1;
    } else if (dir == 2) {
        // f(na, n, nb)
        A.sa_in = 1; A.sb_in = na * (long)s.n_in; A.se_in = na;
        A.sa_out = 1; A.sb_out = na * (long)s.n_out; A.se_out = na;
    } else {
        // f(na, nb, n): the (na, nb) plane is one contiguous pencil index
        A.sa_in = 1; A.sb_in = 0; A.se_in = na * nb;
        A.sa_out = 1; A.sb_out = 0; A.se_out = na * nb;
    }
    if (shape == SHAPE_OVL_X || shape == SHAPE_OVL_STRIDED) {
        const OverlapTables &o = v->ovl;
        A.m = o.m; A.P = o.P; A.xr = 0; A.nbl = o.nbl; A.nbr = o.nbr;
        A.nd = o.nd; A.d0 = o.d0; A.guni = o.guni;
        const int steps = s.periodic ? o.P : std::max(o.P - 1, 1);
        A.smul = s.periodic ? s.n_sys : (o.P > 1 ? s.n_sys - o.m : 0);
        A.sdiv = steps > 1 ? (1u << 31) / steps + 1 : 1u << 31;
        A.tab_d = v->d_ovl; A.tab_f = nullptr;
        A.o_fac = 0; A.o_G = v->ov_G; A.o_sp = v->ov_sp;
    }
    return 0;
}

// launch of prepared calls; `work` serves the general kernel
static hipError_t launch(int family, int shape, int mode, ApplyBatch &B, int count, double *work, hipStream_t stream)
{
    if (shape == SHAPE_OVL_X || shape == SHAPE_OVL_STRIDED)
        return launch_overlap(family, shape, mode == MODE_F64, B, count, stream);
    return launch_compact(family, shape, mode, B, count, work, stream);
}

// whether a shape has kernels for several passes
static bool may_join(int shape, int mode, int family)
{
    if (shape == SHAPE_OVL_X || shape == SHAPE_OVL_STRIDED) return true;
    return shape != SHAPE_GENERAL && can_batch(family_shape(family).K, mode);
}

bool small_field(long points, int prec)
{
    return prec == PDO_F64 ? points * 8 <= (long)SMALL_F64 : points * 4 <= (long)SMALL_F32;
}

int apply_many(const ApplyTask *tasks, int count, int dir, int prec, long na, long nb, hipStream_t stream)
{
    ApplyBatch B;
    int held = 0, shape0 = 0, mode0 = 0, family0 = 0;
    auto flush = [&]() -> int {
        if (!held) return 0;
        const hipError_t e = launch(family0, shape0, mode0, B, held, nullptr, stream);
        held = 0;
        return e == hipSuccess ? 0 : hip_fail(e, "kernel launch");
    };
    for (int i = 0; i < count; i++) {
        const ApplyTask &t = tasks[i];
        ApplyArgs A;
        int shape = 0, mode = 0, family = 0;
        size_t scratch_elems = 0;
        bool empty = false;
        int st = prepare(t.op, t.kind, t.bc1, t.bcn, dir, prec, t.f, t.out, na, nb, t.epi, t.aux, t.force_shape,
                         count > 1, A, shape, mode, family, scratch_elems, &empty);
        if (st) return st;
        if (empty) continue;
        // one launch serves passes whose grid, workgroup and kernel agree
        const ApplyArgs &F = B.a[0];
        const bool join = held > 0 && held < MAX_BATCH && may_join(shape, mode, family) && shape == shape0 && mode == mode0 && family == family0 &&
                          small_field(A.n_sys * na * nb, prec) && A.periodic == F.periodic &&
                          A.n_sys == F.n_sys && A.n_in == F.n_in && A.n_out == F.n_out && A.m == F.m && A.P == F.P &&
                          A.xr == F.xr && (A.epi != 0) == (F.epi != 0);
        if (!join && (st = flush())) return st;
        if (shape == SHAPE_GENERAL) {
            // the general kernel's work area is stream-ordered memory of this
            // pass alone: no host synchronisation, and no sharing between
            // launches that run concurrently on different streams
            double *scratch = nullptr;
            hipError_t e = hipMallocAsync((void **)&scratch, scratch_elems * sizeof(double), stream);
            if (e != hipSuccess) return hip_fail(e, "hipMallocAsync(general-kernel work area)");
            B.a[0] = A;
            e = launch(family, shape, mode, B, 1, scratch, stream);
            const hipError_t ef = hipFreeAsync(scratch, stream);
            if (e == hipSuccess) e = ef;
            if (e != hipSuccess) return hip_fail(e, "kernel launch");
            continue;
        }
        B.a[held++] = A;
        shape0 = shape; mode0 = mode; family0 = family;
    }
    return flush();
}

int apply(OpObject *op, int kind, int bc1, int bcn, int dir, int prec, const void *f, void *out, long na, long nb,
          hipStream_t stream, int epi, const void *aux, int force_shape)
{
    const ApplyTask t{op, kind, bc1, bcn, f, out, epi, aux, force_shape};
    return apply_many(&t, 1, dir, prec, na, nb, stream);
}

int apply_noalloc(OpObject *op, int kind, int bc1, int bcn, int dir, int prec, const void *f, void *out, long na,
                  long nb, hipStream_t stream, double *work, size_t work_elems)
{
    if (!op || !f || !out || na < 0 || nb < 0 || dir < 1 || dir > 3 || prec_mode(prec) < 0) {
        set_error("invalid argument");
        return PDO_ERR_ARG;
    }
    if (op->scheme == SCHEME_CD10 || op->scheme == SCHEME_CF90) {
        // cd10.F90:2042-2058, cf90.F90:1036-1052: GracefulExit(..., 324)
        if (bc1 < -1 || bc1 > 1 || bcn < -1 || bcn > 1) {
            set_error("Incorrect boundary specification for bc1/bcn (should be 0, 1 or -1)");
            return 324;
        }
    } else {
        bc1 = bcn = 0;  // cd06 and cd06stagg objects take their ends from init
    }
    if (op->n == 1) {
        // one-point objects: derivatives are zero, the filter is the identity
        const size_t w = (prec == PDO_F64) ? 8 : 4;
        hipError_t e = (kind == KIND_FILTER)
                           ? hipMemcpyAsync(out, f, (size_t)(na * nb) * w, hipMemcpyDeviceToDevice, stream)
                           : launch_zero_words(out, na * nb * (long)(w / 4), stream);
        return e == hipSuccess ? 0 : hip_fail(e, "one-point operator");
    }
    ApplyArgs A;
    int shape = 0, mode = 0, family = 0;
    size_t scratch_elems = 0;
    bool empty = false;
    int st = prepare(op, kind, bc1, bcn, dir, prec, f, out, na, nb, 0, nullptr, -1, false, A, shape, mode, family,
                     scratch_elems, &empty, true);
    if (st || empty) return st;
    // the limit is the entry point's contract for every call outside the fixed
    // register kernels, whichever kernel serves it
    if (scratch_elems > work_elems) {
        set_error("input too large for the fixed work area of the allocation-free entry point (" +
                  std::to_string(scratch_elems) + " > " + std::to_string(work_elems) + " FP64 words)");
        return PDO_ERR_ARG;
    }
    ApplyBatch B;
    B.a[0] = A;
    const hipError_t e = launch(family, shape, mode, B, 1, shape == SHAPE_GENERAL ? work : nullptr, stream);
    if (e != hipSuccess) return hip_fail(e, "kernel launch");
    return 0;
}

}  // namespace pdo

using namespace pdo;

extern "C" {

const char *pdo_last_error(void) { return pdo::last_error(); }

int pdo_device_count(int *count)
{
    int c = 0;
    hipError_t e = hipGetDeviceCount(&c);
    if (count) *count = (e == hipSuccess) ? c : 0;
    if (e == hipErrorNoDevice || (e == hipSuccess && c == 0)) {
        set_error("no HIP device");
        return PDO_ERR_NOGPU;
    }
    if (e != hipSuccess) return hip_fail(e, "hipGetDeviceCount");
    return 0;
}

int pdo_sync(void *stream)
{
    hipError_t e = hipStreamSynchronize((hipStream_t)stream);
    return e == hipSuccess ? 0 : hip_fail(e, "hipStreamSynchronize");
}

int pdo_malloc(void **ptr, size_t bytes)
{
    hipError_t e = hipMalloc(ptr, bytes);
    return e == hipSuccess ? 0 : hip_fail(e, "hipMalloc");
}

int pdo_free(void *ptr)
{
    hipError_t e = hipFree(ptr);
    return e == hipSuccess ? 0 : hip_fail(e, "hipFree");
}

int pdo_memcpy_h2d(void *dst, const void *src, size_t bytes)
{
    hipError_t e = hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice);
    return e == hipSuccess ? 0 : hip_fail(e, "hipMemcpy");
}

int pdo_memcpy_d2h(void *dst, const void *src, size_t bytes)
{
    hipError_t e = hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
    return e == hipSuccess ? 0 : hip_fail(e, "hipMemcpy");
}

int pdo_memcpy_d2d(void *dst, const void *src, size_t bytes, void *stream)
{
    if (dst == src || bytes == 0) return 0;
    hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, (hipStream_t)stream);
    return e == hipSuccess ? 0 : hip_fail(e, "hipMemcpyAsync");
}

static int make_op(pdo_op *h, int scheme, int n, double dx, int periodic, int bc1, int bcn)
{
    if (!h) { set_error("null handle"); return PDO_ERR_ARG; }
    *h = nullptr;
    auto *o = new pdo_op_s();
    o->scheme = scheme; o->n = n; o->dx = dx; o->periodic = periodic != 0; o->bc1 = bc1; o->bcn = bcn;
    *h = o;
    return 0;
}

// ---- cd06 -----------------------------------------------------------------
int pdo_cd06_init(pdo_op *h, int n, double dx, int periodic, int bc1, int bcn)
{
    // cd06.F90:129-207: periodic n>=6 (ierr 3), non-periodic n>=8 (ierr 2), n==1 allowed
    if (n != 1 && periodic && n < 6) return 3;
    if (n != 1 && !periodic && n < 8) return 2;
    return make_op(h, SCHEME_CD06, n, dx, periodic, bc1, bcn);
}

static int zero_fill(const pdo_op h, int prec, void *df, long count, hipStream_t st)
{
    // a fill kernel rather than a memset node, so the call can be graph-captured
    const long words = count * ((prec == PDO_F64) ? 2 : 1);
    hipError_t e = launch_zero_words(df, words, st);
    (void)h;
    return e == hipSuccess ? 0 : hip_fail(e, "zero fill");
}

static int copy_fill(int prec, void *dst, const void *src, long count, hipStream_t st)
{
    const size_t w = (prec == PDO_F64) ? 8 : 4;
    hipError_t e = hipMemcpyAsync(dst, src, (size_t)count * w, hipMemcpyDeviceToDevice, st);
    return e == hipSuccess ? 0 : hip_fail(e, "hipMemcpyAsync");
}

#define PDO_N1_DERIV(h, prec, df, na, nb, st)                                   \
    if (!(h)) { set_error("null handle"); return PDO_ERR_ARG; }                 \
    if ((h)->n == 1) return zero_fill(h, prec, df, (long)(na) * (nb), st);

int pdo_cd06_dd1(pdo_op h, int prec, const void *f, void *df, int na, int nb, void *stream)
{
    PDO_N1_DERIV(h, prec, df, na, nb, (hipStream_t)stream)
    return apply(h, KIND_D1, 0, 0, 1, prec, f, df, na, nb, (hipStream_t)stream);
}
int pdo_cd06_dd2(pdo_op h, int prec, const void *f, void *df, int na, int nb, void *stream)
{
    PDO_N1_DERIV(h, prec, df, na, nb, (hipStream_t)stream)
    return apply(h, KIND_D1, 0, 0, 2, prec, f, df, na, nb, (hipStream_t)stream);
}
int pdo_cd06_dd3(pdo_op h, int prec, const void *f, void *df, int na, int nb, void *stream)
{
    PDO_N1_DERIV(h, prec, df, na, nb, (hipStream_t)stream)
    return apply(h, KIND_D1, 0, 0, 3, prec, f, df, na, nb, (hipStream_t)stream);
}
int pdo_cd06_d2d1(pdo_op h, int prec, const void *f, void *df, int na, int nb, void *stream)
{
    PDO_N1_DERIV(h, prec, df, na, nb, (hipStream_t)stream)
    return apply(h, KIND_D2, 0, 0, 1, prec, f, df, na, nb, (hipStream_t)stream);
}
int pdo_cd06_d2d2(pdo_op h, int prec, const void *f, void *df, int na, int nb, void *stream)
{
    PDO_N1_DERIV(h, prec, df, na, nb, (hipStream_t)stream)
    return apply(h, KIND_D2, 0, 0, 2, prec, f, df, na, nb, (hipStream_t)stream);
}
int pdo_cd06_d2d3(pdo_op h, int prec, const void *f, void *df, int na, int nb, void *stream)
{
    PDO_N1_DERIV(h, prec, df, na, nb, (hipStream_t)stream)
    return apply(h, KIND_D2, 0, 0, 3, prec, f, df, na, nb, (hipStream_t)stream);
}

// ---- cd10 -----------------------------------------------------------------
int pdo_cd10_init(pdo_op *h, int n, double dx, int periodic, int bc1, int bcn)
{
    if (n != 1 && n < 8) return 2;  // cd10.F90:216-224
    return make_op(h, SCHEME_CD10, n, dx, periodic, bc1, bcn);
}

static int check_bc(int bc1, int bcn)
{
    // cd10.F90:2042-2058, cf90.F90:1036-1052: GracefulExit(..., 324)
    if (bc1 < -1 || bc1 > 1 || bcn < -1 || bcn > 1) {
        set_error("Incorrect boundary specification for bc1/bcn (should be 0, 1 or -1)");
        return 324;
    }
    return 0;
}

#define PDO_CD10(NAME, KIND, DIR)                                                                          \
    int NAME(pdo_op h, int prec, const void *f, void *df, int na, int nb, int bc1, int bcn, void *stream) \
    {                                                                                                      \
        PDO_N1_DERIV(h, prec, df, na, nb, (hipStream_t)stream)                                             \
        if (int e = check_bc(bc1, bcn)) return e;                                                         \
        return apply(h, KIND, bc1, bcn, DIR, prec, f, df, na, nb, (hipStream_t)stream);                  \
    }
PDO_CD10(pdo_cd10_dd1, KIND_D1, 1)
PDO_CD10(pdo_cd10_dd2, KIND_D1, 2)
PDO_CD10(pdo_cd10_dd3, KIND_D1, 3)
PDO_CD10(pdo_cd10_d2d1, KIND_D2, 1)
PDO_CD10(pdo_cd10_d2d2, KIND_D2, 2)
PDO_CD10(pdo_cd10_d2d3, KIND_D2, 3)
#undef PDO_CD10

// ---- cf90 -----------------------------------------------------------------
int pdo_cf90_init(pdo_op *h, int n, int periodic)
{
    if (n != 1 && n < 10) return 7;  // cf90.F90:123-131,147-170
    return make_op(h, SCHEME_CF90, n, 1.0, periodic, 0, 0);
}

#define PDO_CF90(NAME, DIR)                                                                                  \
    int NAME(pdo_op h, int prec, const void *f, void *fil, int na, int nb, int bc1, int bcn, void *stream) \
    {                                                                                                        \
        if (!h) { set_error("null handle"); return PDO_ERR_ARG; }                                            \
        if (h->n == 1) return copy_fill(prec, fil, f, (long)na * nb, (hipStream_t)stream);                   \
        if (int e = check_bc(bc1, bcn)) return e;                                                           \
        return apply(h, KIND_FILTER, bc1, bcn, DIR, prec, f, fil, na, nb, (hipStream_t)stream);             \
    }
PDO_CF90(pdo_cf90_filter1, 1)
PDO_CF90(pdo_cf90_filter2, 2)
PDO_CF90(pdo_cf90_filter3, 3)
#undef PDO_CF90

int pdo_cf90_filter3_cmplx(pdo_op h, int prec, const void *f, void *fil, int na, int nb, int bc1, int bcn,
                           void *stream)
{
    if (!h) { set_error("null handle"); return PDO_ERR_ARG; }
    if (h->n == 1) return copy_fill(prec, fil, f, 2L * na * nb, (hipStream_t)stream);
    if (h->periodic) {
        // cf90.F90:1246-1248 solves with penta_nn, which a periodic object never allocates
        set_error("complex filter3 needs a non-periodic cf90 object");
        return PDO_ERR_UNSUP;
    }
    // the RHS uses (bc1,bcn) but the solve always uses the (0,0) system
    // (cf90.F90:1246-1248): expressed as an epilogue-free two-variant apply
    // is not possible, so the mixed case uses its own variant key.
    if (bc1 == 0 && bcn == 0)
        return apply(h, KIND_FILTER, 0, 0, 3, prec, f, fil, 2L * na, nb, (hipStream_t)stream);
    return apply(h, KIND_FILTER + 1000, bc1, bcn, 3, prec, f, fil, 2L * na, nb, (hipStream_t)stream);
}

// ---- cd06stagg --------------------------------------------------------------
int pdo_cd06stagg_init_periodic(pdo_op *h, int n, double dz)
{
    if (n <= 4) {
        set_error("CD06_stagg requires at least 4 points");  // cd06stagg.F90:181-183
        return 21;
    }
    return make_op(h, SCHEME_CD06STAGG, n, dz, 1, 0, 0);
}

int pdo_cd06stagg_init(pdo_op *h, int n, double dz, int isTopEven, int isBotEven, int isTopSided, int isBotSided)
{
    if (n <= 4) {
        set_error("CD06_stagg requires at least 4 points");  // cd06stagg.F90:216-218
        return 21;
    }
    if (n < 8) {
        set_error("non-periodic cd06stagg needs n >= 8 here (closure rows span 8 points)");
        return PDO_ERR_UNSUP;
    }
    int st = make_op(h, SCHEME_CD06STAGG, n, dz, 0, 0, 0);
    if (st) return st;
    (*h)->flags = (isTopEven ? 1 : 0) | (isBotEven ? 2 : 0) | (isTopSided ? 4 : 0) | (isBotSided ? 8 : 0);
    return 0;
}

#define PDO_STG(NAME, KIND)                                                                                   \
    int NAME(pdo_op h, int prec, const void *fi, void *fo, int n1, int n2, int is_complex, void *stream)    \
    {                                                                                                         \
        if (!h) { set_error("null handle"); return PDO_ERR_ARG; }                                             \
        return apply(h, KIND, 0, 0, 3, prec, fi, fo, (long)n1 * (is_complex ? 2 : 1), n2, (hipStream_t)stream); \
    }
PDO_STG(pdo_cd06stagg_ddz_E2C, KIND_STG_D1_E2C)
PDO_STG(pdo_cd06stagg_ddz_C2E, KIND_STG_D1_C2E)
PDO_STG(pdo_cd06stagg_d2dz2_C2C, KIND_STG_D2_C2C)
PDO_STG(pdo_cd06stagg_d2dz2_E2E, KIND_STG_D2_E2E)
PDO_STG(pdo_cd06stagg_interpz_E2C, KIND_STG_IN_E2C)
PDO_STG(pdo_cd06stagg_interpz_C2E, KIND_STG_IN_C2E)
PDO_STG(pdo_cd06stagg_ddz_C2C, KIND_STG_D1_C2C)
PDO_STG(pdo_cd06stagg_ddz_E2E, KIND_STG_D1_E2E)
#undef PDO_STG

int pdo_op_destroy(pdo_op h)
{
    delete h;
    return 0;
}

int pdo_op_dims(pdo_op h, int kind, int *n_sys, int *n_in)
{
    if (!h) return PDO_ERR_ARG;
    SystemDesc s;
    int st = build_desc(*h, kind, 0, 0, s);
    if (st) return st;
    if (n_sys) *n_sys = s.n_sys;
    if (n_in) *n_in = s.n_in;
    return 0;
}

int pdo_op_dense(pdo_op h, int kind, int bc1, int bcn, double *A, double *B)
{
    if (!h || !A || !B) return PDO_ERR_ARG;
    SystemDesc s;
    int st = build_desc(*h, kind, h->periodic ? 0 : bc1, h->periodic ? 0 : bcn, s);
    if (st) return st;
    dense(s, A, B);
    return 0;
}

int pdo_op_partition(pdo_op h, int kind, int bc1, int bcn, int *m, int *P)
{
    if (!h) return PDO_ERR_ARG;
    SystemDesc s;
    int st = build_desc(*h, kind, h->periodic ? 0 : bc1, h->periodic ? 0 : bcn, s);
    if (st) return st;
    SpikeTables t;
    st = build_spike(s, t);
    if (st) return PDO_ERR_ARG;
    if (m) *m = t.m;
    if (P) *P = t.P;
    return 0;
}

int pdo_op_tables(pdo_op h, int kind, int bc1, int bcn, int general, int *meta, double *fac, double *spk,
                  double *G, double *sp)
{
    if (!h || !meta) return PDO_ERR_ARG;
    SystemDesc s;
    int st = build_desc(*h, kind, h->periodic ? 0 : bc1, h->periodic ? 0 : bcn, s);
    if (st) return st;
    SpikeTables t;
    if (build_spike(s, t, general != 0)) return PDO_ERR_ARG;
    meta[0] = t.m; meta[1] = t.P; meta[2] = t.K; meta[3] = t.nbl; meta[4] = t.nbr; meta[5] = t.xr;
    if (fac) std::memcpy(fac, t.fac.data(), t.fac.size() * sizeof(double));
    if (spk) std::memcpy(spk, t.spk.data(), t.spk.size() * sizeof(double));
    if (G) std::memcpy(G, t.G.data(), t.G.size() * sizeof(double));
    if (sp) std::memcpy(sp, t.sp.data(), t.sp.size() * sizeof(double));
    return 0;
}

int pdo_op_overlap_tables(pdo_op h, int kind, int bc1, int bcn, int *meta, double *fac, double *spk, double *G,
                          double *sp)
{
    if (!h || !meta) return PDO_ERR_ARG;
    SystemDesc s;
    int st = build_desc(*h, kind, h->periodic ? 0 : bc1, h->periodic ? 0 : bcn, s);
    if (st) return st;
    OverlapTables t;
    build_overlap(s, t);
    const int m[9] = {t.m, t.P, t.K, t.nbl, t.nbr, t.q0, t.nd, t.d0, t.guni};
    std::copy(m, m + 9, meta);
    if (fac) std::copy(t.fac.begin(), t.fac.end(), fac);
    if (spk) std::copy(t.spk.begin(), t.spk.end(), spk);
    if (G) std::copy(t.G.begin(), t.G.end(), G);
    if (sp) std::copy(t.sp.begin(), t.sp.end(), sp);
    return 0;
}

}  // extern "C"
