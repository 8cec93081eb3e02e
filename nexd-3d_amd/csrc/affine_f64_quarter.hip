// affine_kernel instantiations, FP64, TVD schemes, a quarter of the elements per block.
#include "affine_impl.hpp"

template void nexd::launch_affine<double, false, 2>(int, bool, bool, const nexd::StageArgs<double> &, hipStream_t);
