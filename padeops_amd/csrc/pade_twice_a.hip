// The operator applied twice: 16-, 24- and 32-row partitions, and the dispatch.
#include "pade_twice_launch.h"

namespace pade {

hipError_t launch_twice_16(const ApplyArgs<double> &a, bool uneven, bool adj, int mode, hipStream_t s)
{
    return uneven ? launch_twice_m<16, 2, true>(a, 1, adj, mode, s) : launch_twice_m<16, 2, false>(a, 1, adj, mode, s);
}

hipError_t launch_twice_32(const ApplyArgs<double> &a, int PW, int GW, bool adj, int mode, hipStream_t s)
{
    if (PW == 8) return launch_twice_m<32, 8, false>(a, GW, adj, mode, s);
    return launch_twice_m<32, 2, false>(a, GW, adj, mode, s);
}

hipError_t launch_twice(const ApplyArgs<double> &a, int M, int PW, int GW, bool uneven, bool adj, int mode,
                        hipStream_t s)
{
    if (a.P < 1 || a.P > kMaxPartitions || (a.P + PW - 1) / PW > 8) return hipErrorInvalidValue;
    if ((PW != 2 && PW != 8) || (PW == 8 && (uneven || mode != 1 || a.P > 8))) return hipErrorInvalidValue;
    if (uneven && !uneven_layout_ok(a, M)) return hipErrorInvalidValue;
    switch (M) {
    case 16: return PW == 2 ? launch_twice_16(a, uneven, adj, mode, s) : hipErrorInvalidValue;
    case 24: return uneven ? launch_twice_24(a, adj, mode, s) : hipErrorInvalidValue;
    case 32: return uneven ? launch_twice_32u(a, adj, mode, s) : launch_twice_32(a, PW, GW, adj, mode, s);
    case 40:
    case 48: return launch_twice_mid(a, M, PW, GW, uneven, adj, mode, s);
    case 64: return uneven ? launch_twice_64u(a, adj, mode, s) : launch_twice_64(a, PW, GW, adj, mode, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace pade
