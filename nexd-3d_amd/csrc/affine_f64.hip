// affine_kernel instantiations, FP64, TVD schemes, the largest blocks.
#include "affine_impl.hpp"

template void nexd::launch_affine<double, false, 0>(int, bool, bool, const nexd::StageArgs<double> &, hipStream_t);
