// psv_resident_f32x2.hip -- the resident time loop in compensated FP32.  FP32 with FMA
// contraction has none: what the compiler fuses depends on the code around it, so another
// kernel would give other roundings than the split step's.
#include "psv_resident.inc"

namespace psv {

namespace {

const ResShape kShapes[] = {{8, 2, 2, 12.5}, {12, 2, 2, 17}, {12, 3, 2, 20.5}};

template <>
const void* kernel_of<dfloat>(int order, int mode, int shape, int* threads)
{
    if (shape >= 0 && shape < 3) *threads = kShapes[shape].waves * 64;
    if (shape == 0) return resident_kernel<dfloat, 8, 2, 2>(order, mode);
    if (shape == 1) return resident_kernel<dfloat, 12, 2, 2>(order, mode);
    if (shape == 2) return resident_kernel<dfloat, 12, 3, 2>(order, mode);
    return nullptr;
}

}  // namespace

template <>
int resident_shapes<dfloat>(const ResShape** out)
{
    *out = kShapes;
    return 3;
}

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

template hipError_t resident_capacity<dfloat>(int, int, int, int*);
template hipError_t launch_resident<dfloat>(const ResidentParams<dfloat>&, int, int, int, hipStream_t);

}  // namespace psv
