// psv_resident_f64.hip -- the resident time loop in FP64.
#include "psv_resident.inc"
#include "psv_resident_launch.inc"

namespace psv {

template <>
int resident_shapes<double>(const ResShape** out)
{
#define PSV_SHAPE(I, NW, R, RE, US, FWD, ADJ) {NW, R, RE, US, FWD, ADJ},
    static const ResShape shapes[] = {PSV_RESIDENT_F64(PSV_SHAPE)};
    *out = shapes;
    return (int)(sizeof shapes / sizeof shapes[0]);
}

template <>
const void* resident_kernel<double>(int order, int mode, int shape, int* threads)
{
#define PSV_KERNEL(I, NW, R, RE, US, FWD, ADJ) \
    if (shape == I) { \
        *threads = NW * 64; \
        return kernel_of<double, kForward, kAdjoint, NW, R, RE>(order, mode); \
    }
    PSV_RESIDENT_F64(PSV_KERNEL)
    return nullptr;
}

template hipError_t resident_capacity<double>(int, int, int, int*);
template hipError_t launch_resident<double>(const ResidentParams<double>&, int, int, int, hipStream_t);

}  // namespace psv
