// Explicit symmetric filters (Gaussian, least squares): launch arguments;
// the elementwise sums of the operators module.
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/padeops_hip.h"

namespace pdo {

constexpr int EXPL_R = 4;   // stencil half-width
constexpr int EXPL_NB = 4;  // closure rows per end (non-periodic)
constexpr int EXPL_WB = 8;  // closure weights per row

// Passed by value: the coefficients travel in the kernel arguments.
struct ExplicitArgs {
    int n, na, nb, dir, periodic;
    double c[EXPL_R + 1];                 // c0, c1..c4 of the symmetric stencil
    double left[EXPL_NB * EXPL_WB];       // rows 0..3 against points 0..7
    double right[EXPL_NB * EXPL_WB];      // rows n-4..n-1 against points n-8..n-1
};

// up to three fields of one call (grid z)
struct ExplicitFields {
    const void *f[3];
    void *out[3];
};

// the filter applied `times` (1, or 2 where explicit_twice) times to each field
hipError_t launch_explicit(bool dbl, const ExplicitArgs &E, const ExplicitFields &F, int count, hipStream_t st,
                           int times);
bool explicit_twice(const ExplicitArgs &E);
// the filter along dir, `times` times (1, or 2 where xfilter_can_twice), on
// each of count (at most 3) fields
bool xfilter_can_twice(pdo_xfilter h, int dir);
int xfilter_many(pdo_xfilter h, int dir, int prec, const ExplicitFields &F, int count, int times, long na, long nb,
                 int bc1, int bcn, hipStream_t st);
// out = a + s b, elementwise over n values (FP64 arithmetic)
hipError_t launch_axpy(bool dbl, void *out, const void *a, const void *b, double s, long n, hipStream_t st);

}  // namespace pdo
