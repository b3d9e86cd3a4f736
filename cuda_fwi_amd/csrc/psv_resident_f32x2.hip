// psv_resident_f32x2.hip -- the resident time loop in compensated FP32.  FP32 with FMA
// contraction has none: what the compiler fuses depends on the code around it, so another
// kernel would give other roundings than the split step's.
#include "psv_resident.inc"
#include "psv_resident_launch.inc"

namespace psv {

template <>
int resident_shapes<dfloat>(const ResShape** out)
{
#define PSV_SHAPE(I, NW, R, RE, US, FWD, ADJ) {NW, R, RE, US, FWD, ADJ},
    static const ResShape shapes[] = {PSV_RESIDENT_F32X2(PSV_SHAPE)};
    *out = shapes;
    return (int)(sizeof shapes / sizeof shapes[0]);
}

template <>
const void* resident_kernel<dfloat>(int order, int mode, int shape, int* threads)
{
#define PSV_KERNEL(I, NW, R, RE, US, FWD, ADJ) \
    if (shape == I) { \
        *threads = NW * 64; \
        return kernel_of<dfloat, kForward, kAdjoint, NW, R, RE>(order, mode); \
    }
    PSV_RESIDENT_F32X2(PSV_KERNEL)
    return nullptr;
}

template hipError_t resident_capacity<dfloat>(int, int, int, int*);
template hipError_t launch_resident<dfloat>(const ResidentParams<dfloat>&, int, int, int, hipStream_t);

template <>
int resident_shapes<ffloat>(const ResShape** out)
{
    *out = nullptr;
    return 0;
}

template <>
hipError_t resident_capacity<ffloat>(int, int, int, int*)
{
    return hipErrorInvalidValue;
}

template <>
hipError_t launch_resident<ffloat>(const ResidentParams<ffloat>&, int, int, int, hipStream_t)
{
    return hipErrorInvalidValue;
}

}  // namespace psv
