// psv_resident_f32.hip -- the resident time loop in FP32.
#include "psv_resident.inc"

namespace psv {

namespace {

const ResShape kShapes[] = {{8, 2, 2, 3.8}, {12, 4, 3, 5.2}, {16, 4, 3, 5.8}, {12, 6, 4, 6.6}, {12, 9, 5, 12.5}};

template <>
const void* kernel_of<float>(int order, int mode, int shape, int* threads)
{
    if (shape >= 0 && shape < 5) *threads = kShapes[shape].waves * 64;
    if (shape == 0) return resident_kernel<float, 8, 2, 2>(order, mode);
    if (shape == 1) return resident_kernel<float, 12, 4, 3>(order, mode);
    if (shape == 2) return resident_kernel<float, 16, 4, 3>(order, mode);
    if (shape == 3) return resident_kernel<float, 12, 6, 4>(order, mode);
    if (shape == 4) return resident_kernel<float, 12, 9, 5>(order, mode);
    return nullptr;
}

}  // namespace

template <>
int resident_shapes<float>(const ResShape** out)
{
    *out = kShapes;
    return 5;
}

template hipError_t resident_capacity<float>(int, int, int, int*);
template hipError_t launch_resident<float>(const ResidentParams<float>&, int, int, int, hipStream_t);

}  // namespace psv
