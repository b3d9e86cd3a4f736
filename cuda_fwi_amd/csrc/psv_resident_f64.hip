// psv_resident_f64.hip -- the resident time loop in FP64.
#include "psv_resident.inc"

namespace psv {

namespace {

const ResShape kShapes[] = {{8, 2, 2, 5.6}, {12, 2, 2, 7.2}, {8, 4, 3, 7.6}, {12, 3, 2, 8.8}, {12, 4, 3, 14.5}};

template <>
const void* kernel_of<double>(int order, int mode, int shape, int* threads)
{
    if (shape >= 0 && shape < 5) *threads = kShapes[shape].waves * 64;
    if (shape == 0) return resident_kernel<double, 8, 2, 2>(order, mode);
    if (shape == 1) return resident_kernel<double, 12, 2, 2>(order, mode);
    if (shape == 2) return resident_kernel<double, 8, 4, 3>(order, mode);
    if (shape == 3) return resident_kernel<double, 12, 3, 2>(order, mode);
    if (shape == 4) return resident_kernel<double, 12, 4, 3>(order, mode);
    return nullptr;
}

}  // namespace

template <>
int resident_shapes<double>(const ResShape** out)
{
    *out = kShapes;
    return 5;
}

template hipError_t resident_capacity<double>(int, int, int, int*);
template hipError_t launch_resident<double>(const ResidentParams<double>&, int, int, int, hipStream_t);

}  // namespace psv
