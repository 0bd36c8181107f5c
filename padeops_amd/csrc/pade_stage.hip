// The accumulating apply along z finished by a Runge-Kutta stage: the last
// flux derivative of a right-hand side.  The sum would otherwise be written,
// then read back by the stage: six fields move per equation instead of eight.
// Bound by memory: five equations of 512^3 points, 6 x 1 GiB each, in 5.95 ms
// (5.4 TB/s).
#include "pade_spike.h"

namespace pade {

template <int M, bool UNE>
static hipError_t stage_m(const ApplyArgs<double> &a, hipStream_t s)
{
    return a.periodic ? launch_kernel<double, M, 2, false, 0, false, kStage, UNE, 1, kMaxFields>(a, 1, s)
                      : launch_kernel<double, M, 2, false, 0, true, kStage, UNE, 1, kMaxFields>(a, 1, s);
}

hipError_t launch_stage(const ApplyArgs<double> &a, int M, bool uneven, hipStream_t s)
{
    if (a.P < 1 || a.P > kMaxPartitions || (uneven && !uneven_layout_ok(a, M))) return hipErrorInvalidValue;
    switch (M) {
    case 16: return uneven ? stage_m<16, true>(a, s) : stage_m<16, false>(a, s);
    case 24: return uneven ? stage_m<24, true>(a, s) : hipErrorInvalidValue;
    case 32: return uneven ? stage_m<32, true>(a, s) : stage_m<32, false>(a, s);
    case 40: return uneven ? stage_m<40, true>(a, s) : hipErrorInvalidValue;
    case 48: return uneven ? stage_m<48, true>(a, s) : hipErrorInvalidValue;
    case 64: return uneven ? stage_m<64, true>(a, s) : stage_m<64, false>(a, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace pade
