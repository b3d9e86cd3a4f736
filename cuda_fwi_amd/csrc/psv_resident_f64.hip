// psv_resident_f64.hip -- the resident time loop in FP64.
#include "psv_resident.inc"

namespace psv {

namespace {

const ResShape kShapes[] = {{8, 2, 2}, {16, 3, 2}};

template <>
const void* kernel_of<double>(int order, int mode, int shape, int* threads)
{
    if (shape >= 0 && shape < 2) *threads = kShapes[shape].waves * 64;
    if (shape == 0) return resident_kernel<double, 8, 2, 2>(order, mode);
    if (shape == 1) return resident_kernel<double, 16, 3, 2>(order, mode);
    return nullptr;
}

}  // namespace

template <>
int resident_shapes<double>(const ResShape** out)
{
    *out = kShapes;
    return 2;
}

template hipError_t resident_capacity<double>(int, int, int, int*);
template hipError_t launch_resident<double>(const ResidentParams<double>&, int, int, int, hipStream_t);

}  // namespace psv
