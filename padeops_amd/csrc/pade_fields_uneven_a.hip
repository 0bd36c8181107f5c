// Several fields over uneven partitions of 16, 24, 32 and 64 slots.
#include "pade_fields_launch.h"

namespace pade {

hipError_t fields_uneven_a(const ApplyArgs<double> &a, int M, int mode, hipStream_t s)
{
    switch (M) {
    case 16: return fields_m<16, 2, true>(a, mode, s);
    case 24: return fields_m<24, 2, true>(a, mode, s);
    case 32: return fields_m<32, 2, true>(a, mode, s);
    case 64: return fields_m<64, 2, true>(a, mode, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace pade
