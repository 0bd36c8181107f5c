// Dispatch of a partitioned solve over uneven partitions; one translation
// unit per element type instantiates it.
#pragma once

#include "pade_spike.h"

namespace pade {

template <typename T, int M, int PW = 2>
static hipError_t launch_uneven_m(const ApplyArgs<T> &a, bool adj, int mode, hipStream_t s)
{
    if (!adj) {
        if (mode == 2) return launch_spike_t<T, M, PW, false, 2, true>(a, 1, s);
        return mode == 0 ? launch_spike_t<T, M, PW, false, 0, true>(a, 1, s)
                         : launch_spike_t<T, M, PW, false, 1, true>(a, 1, s);
    }
    if (mode == 2) return hipErrorInvalidValue;
    return mode == 0 ? launch_spike_t<T, M, PW, true, 0, true>(a, 1, s)
                     : launch_spike_t<T, M, PW, true, 1, true>(a, 1, s);
}

// 40 and 48 slots, in translation units of their own
template <typename T>
hipError_t launch_uneven_mid(const ApplyArgs<T> &a, int M, bool adj, int mode, hipStream_t s);

// more than sixteen partitions of 64 slots, four per wave (two would need nine
// or more waves of 256 registers in a workgroup, and a CU holds eight): 16
// neighbouring pencils per strided row, one whole line in FP64.  Bound by
// each wave's own chain, its reduced system of up to 21 partitions included:
// 1025 points, 256 x 128 pencils, FP64 cd10 x / y / z 240 / 176 / 179 us (2.2 /
// 3.0 / 3.0 TB/s), 3780 / 2494 / 2450 with one lane per pencil.  In
// translation units of their own
template <typename T>
hipError_t launch_uneven_long(const ApplyArgs<T> &a, bool adj, int mode, hipStream_t s);

template <typename T>
hipError_t launch_uneven(const ApplyArgs<T> &a, int M, bool adj, int mode, hipStream_t s)
{
    if (!uneven_layout_ok(a, M)) return hipErrorInvalidValue;
    switch (M) {
    case 16: return launch_uneven_m<T, 16>(a, adj, mode, s);
    case 24: return launch_uneven_m<T, 24>(a, adj, mode, s);
    case 32: return launch_uneven_m<T, 32>(a, adj, mode, s);
    case 40:
    case 48: return launch_uneven_mid<T>(a, M, adj, mode, s);
    case 64:
        return a.P > kMaxPartitions ? launch_uneven_long<T>(a, adj, mode, s)
                                    : launch_uneven_m<T, 64>(a, adj, mode, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace pade
