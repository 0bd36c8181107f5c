// FP32 instantiations of the partitioned solve (pade_spike.h).
#include "pade_spike_launch.h"

namespace pade {

template hipError_t launch_spike<float>(const ApplyArgs<float> &, int, int, int, bool, int, hipStream_t);

}  // namespace pade
