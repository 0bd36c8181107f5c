// The operator applied twice: uneven partitions of 40 and 48 slots, and whole
// pencils of 48-row partitions.
#include "pade_twice_launch.h"

namespace pade {

hipError_t launch_twice_mid(const ApplyArgs<double> &a, int M, int PW, int GW, bool uneven, bool adj, int mode,
                            hipStream_t s)
{
    if (PW == 8) return M == 48 && !uneven ? launch_twice_m<48, 8, false>(a, GW, adj, mode, s) : hipErrorInvalidValue;
    if (!uneven) return hipErrorInvalidValue;
    return M == 40 ? launch_twice_m<40, 2, true>(a, 1, adj, mode, s) : launch_twice_m<48, 2, true>(a, 1, adj, mode, s);
}

}  // namespace pade
