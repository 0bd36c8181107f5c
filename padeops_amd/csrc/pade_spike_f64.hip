// FP64 instantiations of the partitioned solve (pade_spike.h).
#include "pade_spike_launch.h"

namespace pade {

template hipError_t launch_spike<double>(const ApplyArgs<double> &, int, int, int, bool, int, hipStream_t);

}  // namespace pade
