// Definition of launch_affine (stage_launch.hpp), included only by the
// affine_*.hip translation units that instantiate it.
#pragma once
#include "stage_launch.hpp"

namespace nexd {

template <typename R, bool LS, int VAR, int ORDER, bool ATT, bool PML>
void launch_affine_one(const StageArgs<R> &a, hipStream_t s) {
    using S = AffShape<ORDER, ATT, PML, R, VAR>;
    const dim3 grid((unsigned)((a.nlist + S::EB - 1) / S::EB) * (unsigned)a.nshot), block(S::NTHR);
    if (grid.x == 0) return;
    // TVD RK2 has kernels of its own per stage; with attenuation or PML they
    // recompute, which the caller decides (recompute_rk2)
    const int rc = ATT || PML ? a.recompute : (a.scheme == 2 ? a.irk : 0);
    if constexpr (LS) hipLaunchKernelGGL((affine_kernel<ORDER, ATT, PML, R, true, VAR, 0>), grid, block, 0, s, a);
    else if (rc == 1) hipLaunchKernelGGL((affine_kernel<ORDER, ATT, PML, R, false, VAR, 1>), grid, block, 0, s, a);
    else if (rc == 2) hipLaunchKernelGGL((affine_kernel<ORDER, ATT, PML, R, false, VAR, 2>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((affine_kernel<ORDER, ATT, PML, R, false, VAR, 0>), grid, block, 0, s, a);
}

template <typename R, bool LS, int VAR, int ORDER>
void launch_affine_order(bool att, bool pml, const StageArgs<R> &a, hipStream_t s) {
    if (att && pml) launch_affine_one<R, LS, VAR, ORDER, true, true>(a, s);
    else if (att) launch_affine_one<R, LS, VAR, ORDER, true, false>(a, s);
    else if (pml) launch_affine_one<R, LS, VAR, ORDER, false, true>(a, s);
    else launch_affine_one<R, LS, VAR, ORDER, false, false>(a, s);
}

template <typename R, bool LS, int VAR>
void launch_affine(int order, bool att, bool pml, const StageArgs<R> &a, hipStream_t s) {
    switch (order) {
        case 2: launch_affine_order<R, LS, VAR, 2>(att, pml, a, s); break;
        case 3: launch_affine_order<R, LS, VAR, 3>(att, pml, a, s); break;
        case 4: launch_affine_order<R, LS, VAR, 4>(att, pml, a, s); break;
        default: launch_affine_order<R, LS, VAR, 5>(att, pml, a, s); break;
    }
}

}  // namespace nexd
