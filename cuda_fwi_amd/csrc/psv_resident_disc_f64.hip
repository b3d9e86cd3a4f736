// psv_resident_disc_f64.hip -- the resident loops of the exact gradient (FP64): replay and
// reverse.
#include "psv_resident.inc"

namespace psv {

template <>
const void* resident_kernel_discrete<double>(int order, int mode, int shape, int* threads)
{
#define PSV_KERNEL(I, NW, R, RE, US, FWD, ADJ) \
    if (shape == I) { \
        *threads = NW * 64; \
        return kernel_of<double, kReplay, kReverse, NW, R, RE>(order, mode); \
    }
    PSV_RESIDENT_F64(PSV_KERNEL)
    return nullptr;
}

}  // namespace psv
