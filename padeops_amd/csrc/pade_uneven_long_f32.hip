// FP32 instantiations of the partitioned solve over more than sixteen uneven
// partitions.
#include "pade_uneven_launch.h"

namespace pade {

template <>
hipError_t launch_uneven_long<float>(const ApplyArgs<float> &a, bool adj, int mode, hipStream_t s)
{
    return launch_uneven_m<float, 64, 4>(a, adj, mode, s);
}

}  // namespace pade
