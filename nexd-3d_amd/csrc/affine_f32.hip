// affine_kernel instantiations, block shape 0: four blocks per CU.
#include "affine_impl.hpp"

template void nexd::launch_affine<float, false, 0>(int, bool, bool, const nexd::StageArgs<float> &, hipStream_t);
