// psv_resident_disc_f32x2.hip -- the resident loops of the exact gradient (compensated FP32): replay and
// reverse.
#include "psv_resident.inc"

namespace psv {

template <>
const void* resident_kernel_discrete<dfloat>(int order, int mode, int shape, int* threads)
{
#define PSV_KERNEL(I, NW, R, RE, US, FWD, ADJ) \
    if (shape == I) { \
        *threads = NW * 64; \
        return kernel_of<dfloat, kReplay, kReverse, NW, R, RE>(order, mode); \
    }
    PSV_RESIDENT_F32X2(PSV_KERNEL)
    return nullptr;
}

}  // namespace psv
