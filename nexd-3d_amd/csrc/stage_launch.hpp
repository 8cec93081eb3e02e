// Launchers of the stage kernel, one per (real type, scheme class).  Each
// is compiled in its own translation unit (stage_*.hip), so the kernel's
// instantiations build in parallel and only once for the single-shot and
// the batched path.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "affine_kernels.hpp"
#include "plain_kernels.hpp"

namespace nexd {

// Launches stage_kernel<order, att, pml, R, LS, VAR> for a.nlist elements
// and a.nshot shots on stream s (nothing for an empty list).  LS selects the
// low-storage RK4 instantiation, VAR the block shape (FP32 TVD only has
// VAR 1).
template <typename R, bool LS, int VAR>
void launch_stage(int order, bool att, bool pml, const StageArgs<R> &a, hipStream_t s);

constexpr int kAffMinOrder = 2;

// Launches affine_kernel<order, att, pml, R, LS, VAR> (straight-sided meshes;
// FP32 has the TVD schemes only) for a.nlist elements and a.nshot shots on
// stream s.
template <typename R, bool LS, int VAR>
void launch_affine(int order, bool att, bool pml, const StageArgs<R> &a, hipStream_t s);
extern template void launch_affine<float, false, 0>(int, bool, bool, const StageArgs<float> &, hipStream_t);
extern template void launch_affine<float, false, 1>(int, bool, bool, const StageArgs<float> &, hipStream_t);
extern template void launch_affine<double, false, 0>(int, bool, bool, const StageArgs<double> &, hipStream_t);
extern template void launch_affine<double, false, 1>(int, bool, bool, const StageArgs<double> &, hipStream_t);
extern template void launch_affine<double, false, 2>(int, bool, bool, const StageArgs<double> &, hipStream_t);
extern template void launch_affine<double, true, 0>(int, bool, bool, const StageArgs<double> &, hipStream_t);
extern template void launch_affine<double, true, 1>(int, bool, bool, const StageArgs<double> &, hipStream_t);
extern template void launch_affine<double, true, 2>(int, bool, bool, const StageArgs<double> &, hipStream_t);

// Whether a run uses the recomputing RK2 kernels (stage_kernel, RC): TVD RK2
// with memory variables or with PML auxiliaries whose update takes the last
// element's fluxes (compat).
constexpr bool recompute_rk2(int scheme, bool att, bool pml, bool pml_compat) {
    return scheme == 2 && (att || pml) && (!pml || pml_compat);
}

// the block shapes the autotuner chooses from, for a real type and scheme
template <typename R>
constexpr int stage_variants(bool ls) { return (sizeof(R) == 4 && !ls) ? 2 : 1; }

// An affine kernel's elements per block, and (FP64) the matrix instructions of
// its busiest wave.
struct AffineBlock {
    int eb, work;
};
template <typename R>
inline AffineBlock affine_block(int order, bool att, bool pml, int var) {
    auto pick = [&](auto ord) {
        constexpr int O = decltype(ord)::value;
        auto shape = [&](auto v) {
            constexpr int V = decltype(v)::value;
            auto one = [](auto s) { return AffineBlock{decltype(s)::EB, decltype(s)::RW * decltype(s)::CW * decltype(s)::KT}; };
            if (att && pml) return one(AffShape<O, true, true, R, V>{});
            if (att) return one(AffShape<O, true, false, R, V>{});
            if (pml) return one(AffShape<O, false, true, R, V>{});
            return one(AffShape<O, false, false, R, V>{});
        };
        if constexpr (sizeof(R) == 8)
            if (var == 2) return shape(std::integral_constant<int, 2>{});
        return var == 1 ? shape(std::integral_constant<int, 1>{}) : shape(std::integral_constant<int, 0>{});
    };
    switch (order) {
        case 2: return pick(std::integral_constant<int, 2>{});
        case 3: return pick(std::integral_constant<int, 3>{});
        case 4: return pick(std::integral_constant<int, 4>{});
        default: return pick(std::integral_constant<int, 5>{});
    }
}

// The FP64 affine shape of a launch of n elements (over all shots).  A small
// launch leaves the chip idle either way, and what is left is one block's
// chain of phases, shorter with fewer elements; with many blocks small ones
// fill the matrix instruction's 16 columns worse.  512 blocks run at once, two
// on each of 256 CUs; a launch with more of the largest takes those.
//   PML (bound by its loads): the smallest blocks that all run at once.
//   Else the least of (blocks on a CU) x (matrix instructions of a wave) + 50 a
//   round of 512 blocks, the smaller block where that is equal.
// us a step of RK2, largest block, half, quarter (* taken): N = 2, 3,072 tets
// 34.0, 35.5, 30.8*; N = 3, 162 tets 32.9, 26.6, 23.9*, 3,072 tets 42.9, 42.2*,
// 44.3, 7,986 tets 79*, 77, 83; N = 4, 162 tets 36, 33, 31*, 750 tets 39.4, 36.8*, 40.8,
// 1,764 tets 45.7*, 52.9, 63.4; N = 5, 162 tets 45, 35, 29*, 3,072 tets 104*,
// 113, 120; with PML N = 2, 3,072 tets 88, 78*, 77, N = 3, 1,764 tets 98, 86*, 90.
inline int affine_shape_f64(int order, bool att, bool pml, long n) {
    int best = 0;
    long cost = 0;
    for (int var = 0; var < 3; ++var) {
        const AffineBlock b = affine_block<double>(order, att, pml, var);
        const long nb = (n + b.eb - 1) / b.eb, rounds = (nb + 511) / 512;
        if (var == 0 && rounds > 1) return 0;
        const long c = pml ? (rounds > 1 ? 1 + var : 0) : (nb + 255) / 256 * b.work + 50 * rounds;
        if (var == 0 || c <= cost) { best = var; cost = c; }
    }
    return best;
}

// the FP64 affine kernel of a launch: its scheme and shape
inline void launch_affine_f64(int order, bool att, bool pml, const StageArgs<double> &a, hipStream_t s) {
    const int var = affine_shape_f64(order, att, pml, (long)a.nlist * a.nshot);
    if (a.scheme == 4) {
        if (var == 2) launch_affine<double, true, 2>(order, att, pml, a, s);
        else if (var == 1) launch_affine<double, true, 1>(order, att, pml, a, s);
        else launch_affine<double, true, 0>(order, att, pml, a, s);
    } else {
        if (var == 2) launch_affine<double, false, 2>(order, att, pml, a, s);
        else if (var == 1) launch_affine<double, false, 1>(order, att, pml, a, s);
        else launch_affine<double, false, 0>(order, att, pml, a, s);
    }
}

// elements per block of an instantiation (block counts of the energy partials)
template <typename R>
inline int stage_eb(int order, bool att, bool pml, int var = 0) {
    auto pick = [&](auto ord) {
        constexpr int O = decltype(ord)::value;
        if (var == 1) {
            if (att && pml) return Shape<O, true, true, R, 1>::EB;
            if (att) return Shape<O, true, false, R, 1>::EB;
            if (pml) return Shape<O, false, true, R, 1>::EB;
            return Shape<O, false, false, R, 1>::EB;
        }
        if (att && pml) return Shape<O, true, true, R>::EB;
        if (att) return Shape<O, true, false, R>::EB;
        if (pml) return Shape<O, false, true, R>::EB;
        return Shape<O, false, false, R>::EB;
    };
    switch (order) {
        case 1: return pick(std::integral_constant<int, 1>{});
        case 2: return pick(std::integral_constant<int, 2>{});
        case 3: return pick(std::integral_constant<int, 3>{});
        case 4: return pick(std::integral_constant<int, 4>{});
        default: return pick(std::integral_constant<int, 5>{});
    }
}

// element blocks of one list launch (per shot)
template <typename R>
inline int stage_blocks(int order, int n, bool att, bool pml, int var = 0) {
    const int eb = stage_eb<R>(order, att, pml, var);
    return (n + eb - 1) / eb;
}

}  // namespace nexd
