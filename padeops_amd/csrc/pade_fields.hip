// The forward partitioned solve of several FP64 fields in one launch.
#include "pade_spike.h"

namespace pade {

template <int M>
static hipError_t fields_m(const ApplyArgs<double> &a, int mode, hipStream_t s)
{
    return mode == 0 ? launch_spike_t<double, M, 2, false, 0, false, 1, kMaxFields>(a, 1, s)
                     : launch_spike_t<double, M, 2, false, 1, false, 1, kMaxFields>(a, 1, s);
}

hipError_t launch_fields(const ApplyArgs<double> &a, int M, int PW, int GW, int mode, hipStream_t s)
{
    if (a.P < 1 || a.P > kMaxPartitions || (a.P + PW - 1) / PW > 8 || GW < 1 || GW > 8) return hipErrorInvalidValue;
    if (mode != 0 && mode != 1) return hipErrorInvalidValue;
    if (PW == 2) {
        switch (M) {
        case 16: return fields_m<16>(a, mode, s);
        case 32: return fields_m<32>(a, mode, s);
        case 64: return fields_m<64>(a, mode, s);
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
