// Several fields over uneven partitions of 40 and 48 slots, and over more than
// sixteen of 64, four per wave.
#include "pade_fields_launch.h"

namespace pade {

hipError_t fields_uneven_b(const ApplyArgs<double> &a, int M, int mode, hipStream_t s)
{
    switch (M) {
    case 40: return fields_m<40, 2, true>(a, mode, s);
    case 48: return fields_m<48, 2, true>(a, mode, s);
    case 64: return fields_m<64, 4, true>(a, mode, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace pade
