// Queries of the apply planner shared by the library's translation units
// (internal to libpadeops_hip).
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/padeops_hip.h"

namespace pade {

// Whether pade_op_apply(op, oper, axis, f, f, na, nb, bc1, bcn, s) -- output
// over its input, FP64 -- is exact: true when the apply runs on the
// partitioned kernels, where a workgroup holds every partition of its
// pencils and all of a pencil is loaded and consumed before any of it is
// stored.  The one-lane-per-pencil path (which keeps intermediates in its
// output), the bounded cd06 second derivative and edge outputs answer false.
bool apply_in_place_ok(pade_op_t op, int oper, int axis, int na, int nb, int bc1, int bcn);

// One operator along one axis of several FP64 device fields (at most six;
// each with its own boundary codes), `times` (1 or 2) times each: out =
// op^times(f), or with acc out = alpha op^times(f) + beta out.  One launch
// where the fields share a partitioned kernel: a field of a small grid
// leaves most of the chip idle, and a repeated operator keeps its
// intermediate in registers; else one apply per field and repetition, with
// `tmp` (a field, needed for times = 2) as the intermediate.  Outputs must
// not overlap any input of the call.
//
// A stage (Runge-Kutta, low storage) may end an accumulating apply: with r =
// alpha op(f) + beta out, Q = dt r + A Q and W += B Q for every field; `out`
// then holds r or its old values, as the kernels serve it.
struct BatchField {
    const double *f;
    double *out;
    int bc1, bcn;
    double *Q = nullptr, *W = nullptr;   // of the stage
};
struct Stage {
    double dt, A, B;
};
int apply_fields(pade_op_t op, int oper, int axis, int nf, const BatchField *flds, int na, int nb, int times, bool acc,
                 double alpha, double beta, double *tmp, hipStream_t s, const Stage *stage = nullptr);

}  // namespace pade
