// psv_resident_disc_f32.hip -- the resident loops of the exact gradient (FP32): replay and
// reverse. The largest shape has none: the five gradients of its cells do not fit in LDS.
#include "psv_resident.inc"

namespace psv {

template <>
const void* resident_kernel_discrete<float>(int order, int mode, int shape, int* threads)
{
#define PSV_KERNEL(I, NW, R, RE, US, FWD, ADJ) \
    if (shape == I) { \
        *threads = NW * 64; \
        return kernel_of<float, kReplay, kReverse, NW, R, RE>(order, mode); \
    }
    PSV_RESIDENT_F32(PSV_KERNEL)
    return nullptr;
}

}  // namespace psv
