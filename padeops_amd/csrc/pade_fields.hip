// The forward partitioned solve of several FP64 fields in one launch: even
// partitions, and the dispatch.
#include "pade_fields_launch.h"

namespace pade {

hipError_t launch_fields(const ApplyArgs<double> &a, int M, int PW, int GW, bool uneven, int mode, hipStream_t s)
{
    if (GW < 1 || GW > 8 || (mode != 0 && mode != 1)) return hipErrorInvalidValue;
    if (uneven) {
        if (!uneven_layout_ok(a, M) || PW != (a.P > kMaxPartitions ? 4 : 2)) return hipErrorInvalidValue;
        return M == 40 || M == 48 || PW == 4 ? fields_uneven_b(a, M, mode, s) : fields_uneven_a(a, M, mode, s);
    }
    if (a.P < 1 || a.P > kMaxPartitions || (a.P + PW - 1) / PW > 8) return hipErrorInvalidValue;
    if (PW == 2) {
        switch (M) {
        case 16: return fields_m<16, 2, false>(a, mode, s);
        case 32: return fields_m<32, 2, false>(a, mode, s);
        case 64: return fields_m<64, 2, false>(a, mode, s);
        default: return hipErrorInvalidValue;
        }
    }
    if (PW != 8 || mode != 1 || a.P > 8) return hipErrorInvalidValue;
    switch (M) {
    case 32: return launch_spike_t<double, 32, 8, false, 1, false, 1, kMaxFields>(a, GW, s);
    case 48: return launch_spike_t<double, 48, 8, false, 1, false, 1, kMaxFields>(a, GW, s);
    case 64: return launch_spike_t<double, 64, 8, false, 1, false, 1, kMaxFields>(a, GW, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace pade
