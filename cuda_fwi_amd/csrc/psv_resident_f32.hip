// psv_resident_f32.hip -- the resident time loop in FP32.
#include "psv_resident.inc"
#include "psv_resident_launch.inc"

namespace psv {

template <>
int resident_shapes<float>(const ResShape** out)
{
#define PSV_SHAPE(I, NW, R, RE, US, FWD, ADJ) {NW, R, RE, US, FWD, ADJ},
    static const ResShape shapes[] = {PSV_RESIDENT_F32(PSV_SHAPE)};
    *out = shapes;
    return (int)(sizeof shapes / sizeof shapes[0]);
}

template <>
const void* resident_kernel<float>(int order, int mode, int shape, int* threads)
{
#define PSV_KERNEL(I, NW, R, RE, US, FWD, ADJ) \
    if (shape == I) { \
        *threads = NW * 64; \
        return kernel_of<float, kForward, kAdjoint, NW, R, RE>(order, mode); \
    }
    PSV_RESIDENT_F32(PSV_KERNEL)
    return nullptr;
}

template hipError_t resident_capacity<float>(int, int, int, int*);
template hipError_t launch_resident<float>(const ResidentParams<float>&, int, int, int, hipStream_t);

}  // namespace psv
