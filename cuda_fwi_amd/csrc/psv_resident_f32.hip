// psv_resident_f32.hip -- the resident time loop in FP32.
#include "psv_resident.inc"

namespace psv {

namespace {

const ResShape kShapes[] = {{8, 2, 2}, {16, 4, 3}, {16, 7, 4}};

template <>
const void* kernel_of<float>(int order, int mode, int shape, int* threads)
{
    if (shape >= 0 && shape < 3) *threads = kShapes[shape].waves * 64;
    if (shape == 0) return resident_kernel<float, 8, 2, 2>(order, mode);
    if (shape == 1) return resident_kernel<float, 16, 4, 3>(order, mode);
    if (shape == 2) return resident_kernel<float, 16, 7, 4>(order, mode);
    return nullptr;
}

}  // namespace

template <>
int resident_shapes<float>(const ResShape** out)
{
    *out = kShapes;
    return 3;
}

template hipError_t resident_capacity<float>(int, int, int, int*);
template hipError_t launch_resident<float>(const ResidentParams<float>&, int, int, int, hipStream_t);

}  // namespace psv
