// The operator applied twice: 64-row partitions.
#include "pade_twice_launch.h"

namespace pade {

hipError_t launch_twice_64(const ApplyArgs<double> &a, int PW, int GW, bool adj, int mode, hipStream_t s)
{
    if (PW == 8) return launch_twice_m<64, 8, false>(a, GW, adj, mode, s);
    return launch_twice_m<64, 2, false>(a, GW, adj, mode, s);
}

}  // namespace pade
