// Dispatch of the operator-applied-twice kernels (REP = 2 of spike_apply): the
// first solve's values stay in registers, their halos go through LDS, and the
// field moves through memory once instead of twice.  With twice the arithmetic
// and 146 instead of 118 registers (FP64, M = 32: three waves per SIMD instead
// of four) the second chain of sweeps and exchange is not hidden behind the
// memory: strided rows at 512^3 take 701 us per field (3.1 TB/s) as two
// periodic cd10 applies in one launch, a bounded cd06 second derivative of 256
// points along y 250 us (4.3 TB/s).  Two launches are slower still: bounded
// cd06 second derivatives in 64 rows or slots, plain, accumulating and adjoint
// on each axis, 1.10-1.67 times as long, the kernels that spill (44-48
// bytes of scratch as whole pencils, 48-116 uneven and bounded) among them; alone 400
// points along x, accumulating, tie (0.98).  A 384 x 384 x 256 RK3 step with
// its gradient, twelve bounded cd06 second derivatives in it, 17.61 -> 16.95
// ms; the compressible step's fourth derivatives and filter pairs are noted
// with its right-hand side.  One translation unit per group of partition sizes
// instantiates them.
#pragma once

#include "pade_spike.h"

namespace pade {

template <int M, int PW, bool UNE>
hipError_t launch_twice_m(const ApplyArgs<double> &a, int GW, bool adj, int mode, hipStream_t s)
{
    if constexpr (PW == 2) {
        if (mode == 0)
            return adj ? launch_spike_t<double, M, 2, true, 0, UNE, 2>(a, 1, s)
                       : launch_spike_t<double, M, 2, false, 0, UNE, 2>(a, 1, s);
    }
    if (mode != 1 || (PW != 2 && adj)) return hipErrorInvalidValue;
    if constexpr (PW == 2) {
        if (adj) return launch_spike_t<double, M, 2, true, 1, UNE, 2>(a, 1, s);
    }
    return launch_spike_t<double, M, PW, false, 1, UNE, 2>(a, GW, s);
}

// instantiated in pade_twice_*.hip
hipError_t launch_twice_16(const ApplyArgs<double> &a, bool uneven, bool adj, int mode, hipStream_t s);
hipError_t launch_twice_24(const ApplyArgs<double> &a, bool adj, int mode, hipStream_t s);
hipError_t launch_twice_32(const ApplyArgs<double> &a, int PW, int GW, bool adj, int mode, hipStream_t s);
hipError_t launch_twice_32u(const ApplyArgs<double> &a, bool adj, int mode, hipStream_t s);
hipError_t launch_twice_mid(const ApplyArgs<double> &a, int M, int PW, int GW, bool uneven, bool adj, int mode,
                            hipStream_t s);
hipError_t launch_twice_64(const ApplyArgs<double> &a, int PW, int GW, bool adj, int mode, hipStream_t s);
hipError_t launch_twice_64u(const ApplyArgs<double> &a, bool adj, int mode, hipStream_t s);

}  // namespace pade
