// FP64 instantiations of the partitioned solve over more than sixteen uneven
// partitions.
#include "pade_uneven_launch.h"

namespace pade {

template <>
hipError_t launch_uneven_long<double>(const ApplyArgs<double> &a, bool adj, int mode, hipStream_t s)
{
    return launch_uneven_m<double, 64, 4>(a, adj, mode, s);
}

}  // namespace pade
