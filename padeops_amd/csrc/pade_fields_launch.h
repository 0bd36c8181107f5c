// Dispatch of a partitioned solve of several FP64 fields; one translation unit
// per group of partition sizes instantiates it.
#pragma once

#include "pade_spike.h"

namespace pade {

template <int M, int PW, bool UNE>
hipError_t fields_m(const ApplyArgs<double> &a, int mode, hipStream_t s)
{
    return mode == 0 ? launch_spike_t<double, M, PW, false, 0, UNE, 1, kMaxFields>(a, 1, s)
                     : launch_spike_t<double, M, PW, false, 1, UNE, 1, kMaxFields>(a, 1, s);
}

// uneven partitions of 16, 24, 32 and 64 slots; of 40 and 48, and more than
// sixteen of 64
hipError_t fields_uneven_a(const ApplyArgs<double> &a, int M, int mode, hipStream_t s);
hipError_t fields_uneven_b(const ApplyArgs<double> &a, int M, int mode, hipStream_t s);

}  // namespace pade
