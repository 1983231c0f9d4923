// Operator objects behind the C ABI: one object per reference derivative /
// filter object, holding lazily built device tables for each (kind, bc1, bcn)
// variant it is applied with.
#pragma once

#include <hip/hip_runtime.h>

#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "pdo_system.hpp"

namespace pdo {

void set_error(const std::string &msg);
int hip_fail(hipError_t e, const char *what);

// one set of tables in device memory: fac | spk | lhs | G | sp
struct TabSet {
    SpikeTables tab;
    double *d_tab = nullptr;  // device: FP64 tables
    float *f_tab = nullptr;   // device: FP32 copies
    int o_fac = 0, o_spk = 0, o_lhs = 0, o_G = 0, o_sp = 0;
    bool ready = false;
    std::vector<double> pack();  // the set's tables in order, and its offsets
};

struct Variant {
    SystemDesc sys;
    TabSet fast;   // partitioned tables (general == true when n does not fit)
    TabSet gen;    // single-segment tables of the general kernel, where fast is not general itself
    OverlapTables ovl;         // overlapping segments (P == 0: not for this system)
    const double *d_ovl = nullptr;
    int ov_G = 0, ov_sp = 0;
    void *mem = nullptr;       // device memory of every table above
    int upload();
    ~Variant();
};

struct OpObject {
    int scheme = 0;
    int n = 0;
    double dx = 1.0;
    bool periodic = true;
    int bc1 = 0, bcn = 0;
    int flags = 0;  // cd06stagg non-periodic: bit 0 isTopEven, 1 isBotEven, 2 isTopSided, 3 isBotSided
    std::map<int, std::unique_ptr<Variant>> variants;
    std::mutex mu;
    // build (or fetch) a variant; returns status (0 ok)
    int variant(int kind, int bc1, int bcn, Variant **out);
    // an already built variant, or nullptr (builds nothing)
    Variant *find_variant(int kind, int bc1, int bcn);
};

// Apply one variant along dir (1 x, 2 y, 3 z) of a field whose pencil count
// is na*nb, optionally fused with an epilogue: epi 1 out = aux + y,
// epi 2 out = aux - y, epi 3 out = -y.
int apply(OpObject *op, int kind, int bc1, int bcn, int dir, int prec, const void *f, void *out, long na, long nb,
          hipStream_t stream, int epi = 0, const void *aux = nullptr, int force_shape = -1);

// Independent passes along one direction of fields of one shape (no output
// read by another), in order but for those that share a launch: see
// small_field.
struct ApplyTask {
    OpObject *op;
    int kind, bc1, bcn;
    const void *f;
    void *out;
    int epi = 0;
    const void *aux = nullptr;
    int force_shape = -1;
};
int apply_many(const ApplyTask *tasks, int count, int dir, int prec, long na, long nb, hipStream_t stream);

// whether passes over fields of this size share launches: a launch of one pass
// over a small field leaves most of the chip idle for its latency.  A cgrid
// RHS in launches of one pass and of up to MAX_BATCH (us): FP64 64^3 471 ->
// 192, 128^3 1107 -> 810, 160^3 2118 -> 1744, 192^3 3249 -> 3004 (54 MiB per
// field; beyond, passes over one field after the other find it in the Infinity
// Cache); FP32 + refine 96^3 716 -> 369, 128^3 853 -> 675, 160^3 1417 -> 1295
// and 192^3 1893 -> 2102 (27 MiB; several pentadiagonal passes run on
// overlapping segments).
constexpr size_t SMALL_F64 = 64u << 20, SMALL_F32 = 16u << 20;  // bytes per field
bool small_field(long points, int prec);

// apply() without any device allocation, for pdo_op_apply_noalloc: the
// variant must already be built, and the general kernel's work area is
// `work` (work_elems FP64 words); larger inputs are rejected
int apply_noalloc(OpObject *op, int kind, int bc1, int bcn, int dir, int prec, const void *f, void *out, long na,
                  long nb, hipStream_t stream, double *work, size_t work_elems);

int prec_mode(int prec);

}  // namespace pdo

struct pdo_op_s : public pdo::OpObject {};
