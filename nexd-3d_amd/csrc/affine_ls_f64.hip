// affine_kernel instantiations, FP64, low-storage RK4, every block shape.
#include "affine_impl.hpp"

template void nexd::launch_affine<double, true, 0>(int, bool, bool, const nexd::StageArgs<double> &, hipStream_t);
template void nexd::launch_affine<double, true, 1>(int, bool, bool, const nexd::StageArgs<double> &, hipStream_t);
template void nexd::launch_affine<double, true, 2>(int, bool, bool, const nexd::StageArgs<double> &, hipStream_t);
