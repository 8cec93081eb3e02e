// affine_kernel instantiations, block shape 1: two blocks per CU (the autotuner's alternative to shape 0).
#include "affine_impl.hpp"

template void nexd::launch_affine<float, false, 1>(int, bool, bool, const nexd::StageArgs<float> &, hipStream_t);
