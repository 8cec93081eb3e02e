// affine_kernel instantiations, FP64, TVD schemes, half of the elements per block.
#include "affine_impl.hpp"

template void nexd::launch_affine<double, false, 1>(int, bool, bool, const nexd::StageArgs<double> &, hipStream_t);
