// Dispatch of a partitioned solve over uneven partitions; one translation
// unit per element type instantiates it.
#pragma once

#include "pade_spike.h"

namespace pade {

template <typename T, int M>
static hipError_t launch_uneven_m(const ApplyArgs<T> &a, bool adj, int mode, hipStream_t s)
{
    if (!adj) {
        if (mode == 2) return launch_spike_t<T, M, 2, false, 2, true>(a, 1, s);
        return mode == 0 ? launch_spike_t<T, M, 2, false, 0, true>(a, 1, s)
                         : launch_spike_t<T, M, 2, false, 1, true>(a, 1, s);
    }
    if (mode == 2) return hipErrorInvalidValue;
    return mode == 0 ? launch_spike_t<T, M, 2, true, 0, true>(a, 1, s)
                     : launch_spike_t<T, M, 2, true, 1, true>(a, 1, s);
}

// 40 and 48 slots, in translation units of their own
template <typename T>
hipError_t launch_uneven_mid(const ApplyArgs<T> &a, int M, bool adj, int mode, hipStream_t s);

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
    case 64: return launch_uneven_m<T, 64>(a, adj, mode, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace pade
