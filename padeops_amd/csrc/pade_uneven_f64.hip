// FP64 instantiations of the partitioned solve over uneven partitions
// (pade_spike.h).
#include "pade_uneven_launch.h"

namespace pade {

template hipError_t launch_uneven<double>(const ApplyArgs<double> &, int, bool, int, hipStream_t);

}  // namespace pade
