// FP32 instantiations of the partitioned solve over uneven partitions
// (pade_spike.h).
#include "pade_uneven_launch.h"

namespace pade {

template hipError_t launch_uneven<float>(const ApplyArgs<float> &, int, bool, int, hipStream_t);

}  // namespace pade
