// FP32 instantiations of the partitioned solve over uneven partitions
// of 40 and 48 slots.
#include "pade_uneven_launch.h"

namespace pade {

template <>
hipError_t launch_uneven_mid<float>(const ApplyArgs<float> &a, int M, bool adj, int mode, hipStream_t s)
{
    return M == 40 ? launch_uneven_m<float, 40>(a, adj, mode, s) : launch_uneven_m<float, 48>(a, adj, mode, s);
}

}  // namespace pade
