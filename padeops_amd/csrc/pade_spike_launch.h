// Dispatch of a partitioned solve to its kernel (partition size, partitions
// per wave, mode); one translation unit per element type instantiates it.
#pragma once

#include "pade_spike.h"

namespace pade {

template <typename T, int M, int PW>
static hipError_t launch_spike_mp(const ApplyArgs<T> &a, bool adj, int mode, hipStream_t s)
{
    if (!adj) {
        if (mode == 2) return launch_spike_t<T, M, PW, false, 2>(a, 1, s);
        return mode == 0 ? launch_spike_t<T, M, PW, false, 0>(a, 1, s) : launch_spike_t<T, M, PW, false, 1>(a, 1, s);
    }
    if (mode == 2) return hipErrorInvalidValue;
    return mode == 0 ? launch_spike_t<T, M, PW, true, 0>(a, 1, s) : launch_spike_t<T, M, PW, true, 1>(a, 1, s);
}

template <typename T>
hipError_t launch_spike(const ApplyArgs<T> &a, int M, int PW, int GW, bool adj, int mode, hipStream_t s)
{
    if (a.P < 1 || a.P > kMaxPartitions || (a.P + PW - 1) / PW > 8) return hipErrorInvalidValue;
    if (GW < 1 || GW > 8) return hipErrorInvalidValue;
    if (PW == 1) {
        switch (M) {
        case 16: return launch_spike_mp<T, 16, 1>(a, adj, mode, s);
        case 32: return launch_spike_mp<T, 32, 1>(a, adj, mode, s);
        case 64: return launch_spike_mp<T, 64, 1>(a, adj, mode, s);
        default: return hipErrorInvalidValue;
        }
    }
    if (PW == 2) {
        switch (M) {
        case 16: return launch_spike_mp<T, 16, 2>(a, adj, mode, s);
        case 32: return launch_spike_mp<T, 32, 2>(a, adj, mode, s);
        case 64: return launch_spike_mp<T, 64, 2>(a, adj, mode, s);
        default: return hipErrorInvalidValue;
        }
    }
    // whole pencils per wave: x pencils only (strided rows of 8 pencils
    // would split every load into 64-byte pieces), P <= 8
    if (PW == 8 && mode == 1 && a.P <= 8) {
        switch (M) {
        case 32:
            return adj ? launch_spike_t<T, 32, 8, true, 1>(a, GW, s) : launch_spike_t<T, 32, 8, false, 1>(a, GW, s);
        case 48:
            if constexpr (sizeof(T) == 8)       // (periodic: no adjoint form)
                return adj ? hipErrorInvalidValue : launch_spike_t<T, 48, 8, false, 1>(a, GW, s);
            return hipErrorInvalidValue;
        case 64:
            return adj ? launch_spike_t<T, 64, 8, true, 1>(a, GW, s) : launch_spike_t<T, 64, 8, false, 1>(a, GW, s);
        default: return hipErrorInvalidValue;
        }
    }
    // four partitions of 16 pencils per wave on strided rows (one 128-byte
    // line of FP64 per partition row)
    if (PW == 4 && mode == 0) {
        switch (M) {
        case 32: return adj ? launch_spike_t<T, 32, 4, true, 0>(a, 1, s) : launch_spike_t<T, 32, 4, false, 0>(a, 1, s);
        case 64: return adj ? launch_spike_t<T, 64, 4, true, 0>(a, 1, s) : launch_spike_t<T, 64, 4, false, 0>(a, 1, s);
        default: return hipErrorInvalidValue;
        }
    }
    return hipErrorInvalidValue;
}

}  // namespace pade
