// The operator applied twice: uneven partitions of 24, 32 and 64 slots.
#include "pade_twice_launch.h"

namespace pade {

hipError_t launch_twice_24(const ApplyArgs<double> &a, bool adj, int mode, hipStream_t s)
{
    return launch_twice_m<24, 2, true>(a, 1, adj, mode, s);
}

hipError_t launch_twice_32u(const ApplyArgs<double> &a, bool adj, int mode, hipStream_t s)
{
    return launch_twice_m<32, 2, true>(a, 1, adj, mode, s);
}

hipError_t launch_twice_64u(const ApplyArgs<double> &a, bool adj, int mode, hipStream_t s)
{
    return launch_twice_m<64, 2, true>(a, 1, adj, mode, s);
}

}  // namespace pade
