// The stage kernel of straight-sided meshes: FP32 TVD schemes and FP64.
//
// On a straight-sided tetrahedron the metric, the Jacobian and the face
// scales are constant and the face frames orthonormal, so a stage's right-hand
// side is one product per element,
//   rhs_i = Dr C_r,i + Ds C_s,i + Dt C_t,i + LIFT F_i,   C_o,i = o_x F_i + o_y G_i + o_z H_i,
// with A = [Dr|Ds|Dt|LIFT] (Np x (3 Np + 4 NpF)) on the matrix cores, 9
// columns an element, and with attenuation 6 more for the common rates of the
// memory variables, LIFT F_9+s less the strain rate s.  Volume and lifted face
// values meet in the accumulators: one value per node and column goes back to
// the node threads, where the general kernel (plain_kernels.hpp) writes and
// reads 27 derivatives (or 15) and 16 lifted values.
//
// The reference's metric varies between the nodes of an element by 1.5e-7,
// because its operators differentiate linear functions no better; the host
// moves that pattern, the same in every element, into the operators
// (affine_mesh) and so keeps the reference's derivatives to rounding with one
// metric per element.  Its face scales and frames vary by 2e-7 from single-
// precision geometry; their mean changes seismograms by 3e-8 to 8e-8, so FP32
// takes the mean and the normal alone, FP64 every node's scale and the whole
// frame.  Meshes that are not of this kind (affine_mesh) are left to the general
// kernel.
//
// FP32, what bounds it: matrix and vector instructions share the SIMDs, and with
// the general kernel the vector instructions were most of them (N = 3 elastic,
// 64 shots: vector 44 %, matrix 25 % of the time, 1 TB/s).  So
//   - the upwind flux is formed from the normal only (affine_flux): traction
//     and velocity jumps split into their normal and tangential parts, no
//     division and 3 of 9 frame values;
//   - the contravariant columns outside the PML are formed from q in LDS on
//     the way into the product, with the column's nine coefficients (metric
//     times material) in registers;
//   - neighbour traces load beside the element's own values: their indices
//     need only the element id;
//   - the product runs on the BF16 matrix instruction, operator and columns
//     each as the sum of three bfloat16 (24 bits of the columns exactly, 27 of
//     the operator) and the six products above 2^-24: 96 cycles for 32 values
//     where the FP32 instruction takes 256, and with fewer roundings: that one
//     rounds after every product (rms error 2.5 eps R at 64 products, R the
//     root of their squares' sum), this one 0.8 with the five small products in
//     a sum of their own.  The seismograms' error against 64 bits, over random
//     sizes, orders 2 to 5, with and without attenuation and PML, is 0.2 to 1.1
//     of the general kernel's (one FP32 chain over the whole product would give
//     1.3 to 1.8).
// Measured against the general kernel, per stage: N = 3 elastic, 64 shots on
// 3,072 tets 360 -> 269 us; elastic single shots N = 2, 3, 4, 5 33 -> 26, 44 ->
// 29, 68 -> 37, 195 -> 95 us; N = 4 with attenuation and PML, 8 shots, stages
// 1 and 2 1,466 -> 1,294 and 2,174 -> 1,953 us (3.2 and 3.5 TB/s of traffic; a
// large copy reaches 4.7).  Vector instructions are now 42 to 53 % of the time,
// matrix instructions 15 to 29 %.  Order 1 stays with the general kernel (a
// step of 4 values: no faster here).
//
// FP64: the same product on the FP64 matrix instruction, 64 cycles for 16 x 16 x
// 4.  The general kernel spent a PML block's time (N = 4 with attenuation, stage
// 2, 74k cycles) on loads and the PML update 31 %, face term 15 %, LIFT 7 %,
// volume term and its metric 31 %, memory variables 13 %.  Here the face term runs
// beside the PML update on the waves without nodes, and 15 columns in one product
// replace 27 and the LIFT's 16 columns for 15 (9) values: 126 instead of 171 matrix
// instructions a wave.  Where 16-row tiles and column tiles do not share out
// evenly over four waves, the waves are split over the rows (row_groups: N = 5
// a row tile each).  The flux is upwind_flux without divisions.
// Per stage, before and after: N = 4 with attenuation and PML on 192,000 tets,
// stages 1 and 2 1,975 -> 1,694 and 2,925 -> 2,553 us (2.3 and 2.5 TB/s; loads are
// 38 % of a block's time, the product 25 %), N = 5 RK3 on 6,006 tets 176 -> 104
// us in the PML and 56 -> 39 outside, N = 3 RK4 on 3,072 tets 16.5 -> 11.2 us, on 162
// tets 11.3 -> 6.2 us (the last two also by smaller blocks, affine_shape_f64).
// Three blocks per CU instead of two (168 registers): 1,762 and 2,877 us.
#pragma once
#include <type_traits>

#include "plain_kernels.hpp"

namespace nexd {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x4_t mfma_bf16(bf16x8_t a, bf16x8_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Eight floats as the sum of three bfloat16 each, exactly: 24 significand bits,
// 8 at a time, each part rounded to nearest.  (Truncated parts would all have
// the value's sign, and the products left out, second part of the operator
// times third of the column, would shift the operator the same way at every
// step.)
__device__ __forceinline__ void split3(const float (&v)[8], bf16x8_t (&b)[3]) {
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    u32x4_t p[3];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float x = v[2 * i], y = v[2 * i + 1];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const unsigned h = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2_t{x, y}, bf16x2_t));
            p[k][i] = h;
            x -= __builtin_bit_cast(float, h << 16);
            y -= __builtin_bit_cast(float, h & 0xffff0000u);
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) b[k] = __builtin_bit_cast(bf16x8_t, p[k]);
}

// values per element staged in LDS: the metric (9), the coefficients of the
// columns (7, see column_terms) and the material terms of the flux
constexpr int kAffElem = 23;
enum AffElem { AE_MET = 0, AE_COEF = 9, AE_VP = 16, AE_VS, AE_LAM, AE_MU, AE_LVL, AE_P1, AE_P2 };

// The upwind flux of one face node (upwind_flux) with an orthonormal frame,
// scaled by fs.  With T = sigma n the traction of the jump and v its velocity,
// T_n = T.n, T_t = T - n T_n, v_n, v_t alike:
//   stress    n n^T (z1 - z2) + I z2 + n a^T + a n^T,   a = vs T_t - mu v_t
//   velocity  n z7 - T_t / rho + vs v_t
//   z1 = vp T_n - (lam + 2 mu) v_n,  z2 = lam vp/(lam + 2 mu) T_n - lam v_n,  z7 = -T_n / rho + vp v_n
// (s s^T + t t^T = I - n n^T, so the tangents drop out), and of the anelastic
// part, a1 = T_n/(vp rho) - v_n, c = T_t/(2 vs rho) - v_t/2: n n^T a1 + n c^T + c n^T.
template <bool ATT>
__device__ __forceinline__ void affine_flux(float n0, float n1, float n2, float fs, const float *el, float coef_ef3,
                                            bool free, const float dq[9], float out[ATT ? 15 : 9]) {
    const float vp = el[AE_VP], vs = el[AE_VS], lam = el[AE_LAM], mu = el[AE_MU], lvl = el[AE_LVL];
    const float ft = free ? -2.f * fs : fs, fv = free ? 0.f : fs;
    const float T0 = ft * (dq[0] * n0 + dq[3] * n1 + dq[5] * n2);
    const float T1 = ft * (dq[3] * n0 + dq[1] * n1 + dq[4] * n2);
    const float T2 = ft * (dq[5] * n0 + dq[4] * n1 + dq[2] * n2);
    const float v0 = fv * dq[6], v1 = fv * dq[7], v2 = fv * dq[8];
    const float Tn = T0 * n0 + T1 * n1 + T2 * n2, vn = v0 * n0 + v1 * n1 + v2 * n2;
    const float t0 = T0 - n0 * Tn, t1 = T1 - n1 * Tn, t2 = T2 - n2 * Tn;
    const float u0 = v0 - n0 * vn, u1 = v1 - n1 * vn, u2 = v2 - n2 * vn;
    const float z1 = vp * Tn - (lam + 2.f * mu) * vn, z2 = lvl * Tn - lam * vn, dz = z1 - z2;
    const float a0 = vs * t0 - mu * u0, a1 = vs * t1 - mu * u1, a2 = vs * t2 - mu * u2;
    const float m0 = n0 * dz, m1 = n1 * dz, m2 = n2 * dz;
    out[0] = n0 * (m0 + 2.f * a0) + z2;
    out[1] = n1 * (m1 + 2.f * a1) + z2;
    out[2] = n2 * (m2 + 2.f * a2) + z2;
    out[3] = n0 * (m1 + a1) + n1 * a0;
    out[4] = n1 * (m2 + a2) + n2 * a1;
    out[5] = n0 * (m2 + a2) + n2 * a0;
    const float z7 = coef_ef3 * Tn + vp * vn;   // coef_ef3 = -1/rho
    out[6] = n0 * z7 + (coef_ef3 * t0 + vs * u0);
    out[7] = n1 * z7 + (coef_ef3 * t1 + vs * u1);
    out[8] = n2 * z7 + (coef_ef3 * t2 + vs * u2);
    if constexpr (ATT) {
        const float p1 = el[AE_P1], p2 = el[AE_P2];   // 1/(vp rho), 1/(2 vs rho)
        const float b = p1 * Tn - vn;
        const float c0 = p2 * t0 - 0.5f * u0, c1 = p2 * t1 - 0.5f * u1, c2 = p2 * t2 - 0.5f * u2;
        const float k0 = n0 * b, k1 = n1 * b, k2 = n2 * b;
        out[9] = n0 * (k0 + 2.f * c0);
        out[10] = n1 * (k1 + 2.f * c1);
        out[11] = n2 * (k2 + 2.f * c2);
        out[12] = n0 * (k1 + c1) + n1 * c0;
        out[13] = n1 * (k2 + c2) + n2 * c1;
        out[14] = n0 * (k2 + c2) + n2 * c0;
    }
}

// Column cc of an element: C_o = sum_k o_k * coef_k * q[row_k], k = x, y, z.
// Rows and coefficient numbers (0..3: ef0..ef3 of elastic_flux_node, 4: 0,
// 5: -1, 6: -1/2) as four bits a column: the fluxes F, G, H of the 9 fields,
// then the strain rates with the sign and factor they have in the memory-
// variable rates.
constexpr unsigned long long pack_nibbles(const int (&v)[15]) {
    unsigned long long r = 0;
    for (int i = 0; i < 15; ++i) r |= (unsigned long long)v[i] << (4 * i);
    return r;
}
//                                            0  1  2  3  4  5  6  7  8  ex ey ez exy eyz exz
constexpr int kRowX[15] = {6, 6, 6, 7, 0, 8, 0, 3, 5, 6, 0, 0, 7, 0, 8};
constexpr int kCofX[15] = {0, 1, 1, 2, 4, 2, 3, 3, 3, 5, 4, 4, 6, 4, 6};
constexpr int kRowY[15] = {7, 7, 7, 6, 8, 0, 3, 1, 4, 0, 7, 0, 6, 8, 0};
constexpr int kCofY[15] = {1, 0, 1, 2, 2, 4, 3, 3, 3, 4, 5, 4, 6, 6, 4};
constexpr int kRowZ[15] = {8, 8, 8, 0, 7, 6, 5, 4, 2, 0, 0, 8, 0, 7, 6};
constexpr int kCofZ[15] = {1, 1, 0, 4, 2, 2, 3, 3, 3, 4, 4, 5, 4, 6, 6};
constexpr unsigned long long kRows[3] = {pack_nibbles(kRowX), pack_nibbles(kRowY), pack_nibbles(kRowZ)};
constexpr unsigned long long kCofs[3] = {pack_nibbles(kCofX), pack_nibbles(kCofY), pack_nibbles(kCofZ)};

// Block shape.  256 threads; node threads (element-in-block, node) hold the
// fields, all four waves share the product.
template <int ORDER, bool ATT, bool PML, typename R, int VAR>
struct AffShape {
    static constexpr bool F64 = sizeof(R) == 8;
    static constexpr int NP = Dims<ORDER>::NP, NPF = Dims<ORDER>::NPF, NFP = Dims<ORDER>::NFP;
    static constexpr int NTHR = 256, NW = 4;
    static constexpr int NCOL = ATT ? 15 : 9;       // columns of an element: rhs, memory-variable rates
    static constexpr int NV = NCOL;                 // odd: the node threads' row reads fall in different banks
    static constexpr int SFN = NFP | 1;             // face values: row of face nodes, odd
    static constexpr int ROWS = PML ? 9 + 27 : 9;   // q, and in the PML the contravariant fluxes [3][9]
    // blocks per CU the shape is sized for; FP32: VAR 1 is the autotuner's
    // alternative, FP64: VAR 1 and 2 have a half and a quarter of the elements
    static constexpr int BPC = F64 || VAR ? 2 : 4;
    static constexpr int off_face(int eb) { return ROWS * eb * NP; }
    static constexpr int off_elem(int eb) {
        const int nt = eb * NP, f = off_face(eb) + eb * NCOL * SFN, v = nt * NV, e = 24 * nt + 4 * eb;
        return f > v ? (f > e ? f : e) : (v > e ? v : e);
    }
    static constexpr int lds_reals(int eb) { return off_elem(eb) + kAffElem * eb; }
    // FP64: row tiles split over RG groups of waves, column tiles over the
    // NW / RG waves of a group, for the fewest products of the busiest wave
    static constexpr int RTV = (NP + 15) / 16;                      // row (node) tiles
    static constexpr int products(int eb, int rg) {
        const int ctl = (eb * NCOL + 15) / 16;
        return ((RTV + rg - 1) / rg) * ((ctl + NW / rg - 1) / (NW / rg));
    }
    static constexpr int row_groups(int eb) {
        int best = 1;
        if (RTV >= 2 && products(eb, 2) < products(eb, best)) best = 2;
        if (RTV >= 3 && products(eb, 4) < products(eb, best)) best = 4;
        return best;
    }
    static constexpr int pick_f64() {
        int eb = NTHR / NP;
        if (PML && eb * NP > 192 && 192 / NP >= 2) eb = 192 / NP;
        // a thread's face nodes in registers: two, in the PML five of the face waves
        while (eb > 1 && (lds_reals(eb) * 8 + 8 * eb + 64 > 160 * 1024 / BPC ||
                          eb * NFP > (PML ? 5 * 64 * (NW - (eb * NP + 63) / 64) : 2 * NTHR)))
            --eb;
        const int part = (eb + (1 << VAR) - 1) >> VAR;
        return PML && part < 2 ? 2 : part;   // the last element's fluxes of two stages fit two elements' rows
    }
    static constexpr int pick_eb() {
        if (F64) return pick_f64();
        int eb = NTHR / NP;
        // Fewer elements where that fills the waves' column tiles better:
        // N = 4 with attenuation 4 elements in 4 tiles, one a wave (7 in 7
        // leave one wave half idle and the others spilling; 3,000-tet box, 4
        // shots 0.21 -> 0.18 ms a step), N = 3 with attenuation 8 in 8 (12 in 12
        // spill; 105 -> 91 us a step of 4 shots on 5,184 tets), N = 2 in the PML 10 in 10 (12 in 12;
        // both stages 403 -> 393 us), N = 2 elastic 21 in 12 (25 in 15; 54 ->
        // 51 us).  Elsewhere the largest block was the fastest (N = 3 elastic
        // 7, 10, 11, 12 elements: 318, 293, 287, 269 us a stage).
        const int cap = ORDER == 4 && ATT && !PML   ? 4
                        : ORDER == 3 && ATT && !PML ? 8
                        : ORDER == 2 && ATT && PML  ? 10
                        : ORDER == 2 && !ATT && !PML ? 21
                                                     : eb;
        if (cap < eb) eb = cap;
        // with the PML one wave at least is left to the face term
        if (PML && eb * NP > 192 && 192 / NP >= 2) eb = 192 / NP;
        while (eb > 1 && lds_reals(eb) * 4 + 8 * eb + 64 > 160 * 1024 / BPC) --eb;
        return eb;
    }
    static constexpr int EB = pick_eb();
    static constexpr int NT = EB * NP;
    static constexpr int NWN = (NT + 63) / 64;       // waves with node threads
    static constexpr bool FW = PML && NWN < NW;      // the others do the face term meanwhile
    static constexpr int NFT = FW ? 64 * (NW - NWN) : NTHR;   // threads of the face term
    static constexpr int NFN = EB * NFP;
    static constexpr int FIT = (NFN + NFT - 1) / NFT;
    static constexpr int LDS = lds_reals(EB);
    static constexpr int OFF_F = off_face(EB), OFF_E = off_elem(EB);
    static constexpr int NCT = EB * NCOL, CTL = (NCT + 15) / 16;   // columns, column tiles
    // values of a lane: 3 per node 4 ks + l/16, then one per face node; in steps of 8
    static constexpr int KS = (NP + 3) / 4, KSV = 3 * KS, KSL = NFP / 4, KT = KSV + KSL, NS = (KT + 7) / 8;
    static constexpr int CPW = (CTL + NW - 1) / NW;    // column tiles of a wave
    static constexpr int TG = RTV > 2 ? 1 : 2;   // column tiles in one pass (accumulator registers)
    static constexpr int RG = F64 ? row_groups(EB) : 1, RW = (RTV + RG - 1) / RG;   // row tiles of a wave
    static constexpr int CG = NW / RG, CW = (CTL + CG - 1) / CG;                    // FP64: its column tiles
};


__device__ __forceinline__ void block_barrier() {
    // __syncthreads for a block whose waves reach it in different branches
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// RC: the recomputing RK2 kernels (stage_kernel in plain_kernels.hpp says
// what they leave out; here without attenuation or PML they only fix the
// stage), 0: any stage of any TVD scheme.
template <int ORDER, bool ATT, bool PML, typename R, bool LS, int VAR, int RC>
__global__ void __launch_bounds__(256, (AffShape<ORDER, ATT, PML, R, VAR>::BPC))
affine_kernel(StageArgs<R> a) {
    using S = AffShape<ORDER, ATT, PML, R, VAR>;
    constexpr bool F64 = S::F64, WEIGHTED = !F64;
    constexpr int NP = S::NP, NPF = S::NPF, NFP = S::NFP, EB = S::EB, NT = S::NT, SFN = S::SFN, NCOL = S::NCOL, NV = S::NV;
    constexpr int NTHR = S::NTHR, NW = S::NW, FIT = S::FIT, NFT = S::NFT, NFN = S::NFN;
    // planes through buffer descriptors with PML or attenuation; without, the
    // few loads of a thread come out 2 % faster as global ones
    constexpr bool BUF = PML || ATT;
    __shared__ __align__(16) R lds[S::LDS];
    R *sQ = lds;                        // [9][NT]
    R *sC = lds + 9 * NT;               // [3][9][NT] contravariant fluxes (PML)
    R *sF = lds + S::OFF_F;             // [EB][NCOL][SFN] face values
    R *sE = lds + S::OFF_E;             // [EB][kAffElem]
    R *sV = lds;                        // [NT][NV] the product, over everything before sE
    static_assert(24 * NT + 4 * EB <= S::OFF_E, "energy values must fit the LDS");

    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const size_t ng = (size_t)a.nglob;
    const int it_step = *a.d_it;
    // one contiguous range of blocks per XCD, shots fastest (stage_kernel)
    const unsigned nb = gridDim.x, xcd = blockIdx.x % kXcds, rank = blockIdx.x / kXcds;
    const unsigned per = nb / kXcds, extra = nb % kXcds;
    const unsigned lb = xcd * per + (xcd < extra ? xcd : extra) + rank;
    const int shot = (int)(lb % (unsigned)a.nshot), eblk = (int)(lb / (unsigned)a.nshot);
    const R *qin = a.qin + (size_t)shot * 9 * ng;
    const R *qbase = a.qbase + (size_t)shot * 9 * ng;
    R *qout = a.qout + (size_t)shot * 9 * ng;
    const R *matc = a.matc + (size_t)shot * a.mat_stride;
    const unsigned pnb = (unsigned)(ng * sizeof(R));
    const unsigned pnb_base = RC == 1 || (RC == 0 && a.irk == 1) ? 0u : pnb;

    const bool node_thr = t < NT;
    const int eb = node_thr ? t / NP : 0, j = node_thr ? t - (t / NP) * NP : 0;
    const int idx = eblk * EB + eb;
    const bool valid = node_thr && idx < a.nlist;
    const int e = valid ? a.elist[idx] : 0;
    const unsigned g32 = (unsigned)e * NP + j;
    const size_t g = (size_t)e * NP + j;
    const R dt = a.dt_elem ? a.dt_elem[e] : a.dt;

    // Element constants into LDS.  Elements past the end of the list take
    // element 0's; their values are finite and never stored.
    auto stage_elements = [&](int th, int nth) {
        for (int i = th; i < EB; i += nth) {
            const int b = eblk * EB + i, ee = b < a.nlist ? a.elist[b] : 0;
            const R *m = a.emet + (size_t)ee * 12, *mc = matc + (size_t)ee * 8;
            R met[9];
#pragma unroll
            for (int k = 0; k < 9; ++k) met[k] = m[k];
            const R vp = mc[0], vs = mc[1], lam = mc[3], mu = mc[4], lvl = mc[5], irho = mc[6];
            R *el = sE + i * kAffElem;
#pragma unroll
            for (int k = 0; k < 9; ++k) el[AE_MET + k] = met[k];
            el[AE_COEF + 0] = -(lam + R(2) * mu); el[AE_COEF + 1] = -lam; el[AE_COEF + 2] = -mu; el[AE_COEF + 3] = -irho;
            el[AE_COEF + 4] = R(0); el[AE_COEF + 5] = -R(1); el[AE_COEF + 6] = -R(0.5);
            el[AE_VP] = vp; el[AE_VS] = vs; el[AE_LAM] = lam; el[AE_MU] = mu; el[AE_LVL] = lvl;
            if constexpr (ATT) { el[AE_P1] = irho / vp; el[AE_P2] = R(0.5) * irho / vs; }
        }
    };

    // The face nodes of thread th of the face term: what does not depend on
    // this block's own values, the neighbour traces among it
    R fq[FIT][9];
    f32x4_t fg[F64 ? 1 : FIT];
    R ffr[F64 ? FIT : 1][9], ffs[F64 ? FIT : 1];
    int fnb[FIT], fown[FIT];
    auto face_load = [&](int th) {
        int fe[FIT];
#pragma unroll
        for (int i = 0; i < FIT; ++i) {
            const int q = th + NFT * i, fb = (q < NFN ? q : 0) / NFP, b = eblk * EB + fb;
            fe[i] = b < a.nlist ? a.elist[b] : 0;
        }
#pragma unroll
        for (int i = 0; i < FIT; ++i) {
            const int q = th + NFT * i, qq = q < NFN ? q : 0, fb = qq / NFP, k = qq - fb * NFP;
            fnb[i] = a.nbrt[(size_t)fe[i] * NFP + k];
            if constexpr (F64) {
                ffs[i] = a.fscale[(size_t)fe[i] * NFP + k];
#pragma unroll
                for (int c = 0; c < 9; ++c) ffr[i][c] = a.frame[((size_t)fe[i] * 4 + k / NPF) * 9 + c];
            } else {
                fg[i] = *reinterpret_cast<const f32x4_t *>(a.fgeo + ((size_t)fe[i] * 4 + k / NPF) * 4);
            }
            fown[i] = fb * NP + a.fmask[k];
        }
#pragma unroll
        for (int i = 0; i < FIT; ++i) {
            // a boundary face's index is past every plane: its loads return 0
            const unsigned gn = fnb[i] >= 0 ? (unsigned)fnb[i] : 0xffffffffu / (unsigned)sizeof(R);
#pragma unroll
            for (int f = 0; f < 9; ++f) fq[i][f] = pload<true>(qin + f * ng, pnb, gn);
        }
    };
    auto face_flux = [&](int th) {
#pragma unroll
        for (int i = 0; i < FIT; ++i) {
            const int q = th + NFT * i;
            if (q < NFN) {
                const int fb = q / NFP, k = q - fb * NFP;
                const bool fvalid = eblk * EB + fb < a.nlist;
                R dq[9], fl[NCOL];
#pragma unroll
                for (int f = 0; f < 9; ++f) {
                    dq[f] = fq[i][f] - sQ[f * NT + fown[i]];
                }
                const R *el = sE + fb * kAffElem;
                // the jump of a boundary face is its own trace, here with the
                // other sign; absorbing faces (-2) change the sign once more
                if constexpr (F64) {
                    const R fs = fvalid ? (fnb[i] == -1 ? R(-0.5) : R(0.5)) * ffs[i] : R(0);
                    upwind_flux<R>(ffr[i], el[AE_VP], el[AE_VS], el[AE_LAM], el[AE_MU], el[AE_LVL], -el[AE_COEF + 3],
                                   el[AE_P1], el[AE_P2], fnb[i] == -1, fs, dq, fl, fl + (ATT ? 9 : 0), ATT);
                } else {
                    const R fs = fvalid ? (fnb[i] == -1 ? -fg[i][3] : fg[i][3]) : R(0);
                    affine_flux<ATT>(fg[i][0], fg[i][1], fg[i][2], fs, el, el[AE_COEF + 3], fnb[i] == -1, dq, fl);
                }
                R *dst = sF + fb * NCOL * SFN + k;
#pragma unroll
                for (int f = 0; f < NCOL; ++f) dst[f * SFN] = fl[f];
            }
        }
    };

    R qs[9];
    int src_first = -1, rec_slot_e = -1;
    auto node_load = [&]() {
        src_first = a.src_head[(size_t)shot * (a.nglob / NP) + e];
        rec_slot_e = a.rec_slot[e];
#pragma unroll
        for (int f = 0; f < 9; ++f) qs[f] = pload<BUF>(qin + f * ng, pnb, g32);
    };
    auto node_store = [&]() {
#pragma unroll
        for (int f = 0; f < 9; ++f) sQ[f * NT + t] = qs[f];
    };

    if constexpr (!PML) {
        if (node_thr) node_load();
        stage_elements(t, NTHR);
        face_load(t);
        if (node_thr) node_store();
        __syncthreads();
        face_flux(t);
    } else {
        // node waves: loads, PML update; face waves meanwhile the face term
        // (without any left, FW false, every wave does it afterwards)
        if (S::FW && w >= S::NWN) {
            const int th = t - 64 * S::NWN;
            stage_elements(th, NFT);
            face_load(th);
            block_barrier();   // q, element constants and the staged fluxes are in LDS
            face_flux(th);
            block_barrier();   // the flux rows may be written
        } else {
            constexpr int NNT = S::FW ? 64 * S::NWN : NTHR;   // threads here
            // the last element's fluxes wait in the flux rows until the update
            // is done: [27][NP], and with RC 2 those of stage 1 behind them
            constexpr bool LASTF = RC != 1;
            constexpr int NLASTF = RC == 2 ? 54 * NP : 27 * NP, NLS = LASTF ? (NLASTF + NNT - 1) / NNT : 1;
            static_assert(!LASTF || NLASTF <= 27 * NT, "last-element fluxes must fit the flux rows");
            R *sLast = sC, *sLast1 = sC + 27 * NP;
            R lst[NLS];
            if constexpr (LASTF) {
                if (a.pml_compat) {
                    const R *lf = a.last_flux + (size_t)shot * 27 * NP;
                    const R *lf1 = RC == 2 ? a.last_flux1 + (size_t)shot * 27 * NP : lf;
#pragma unroll
                    for (int r = 0; r < NLS; ++r) {
                        const int i = t + r * NNT;
                        if constexpr (RC == 2) lst[r] = *(i < 27 * NP ? lf + i : lf1 + (i < 54 * NP ? i - 27 * NP : 0));
                        else lst[r] = lf[i < 27 * NP ? i : 0];
                    }
                }
            }
            const R *pin = a.pin + (size_t)shot * 27 * ng;
            const R *pbase = a.pbase + (size_t)shot * 27 * ng;
            R *pout = a.pout + (size_t)shot * 27 * ng;
            R pc[9], cur[27], bse[RC == 0 ? 27 : 1], mv[9], lam = 0, mu = 0, irho = 0;
            if (node_thr) {
                node_load();
                const R *pmlc = a.pmlc + (size_t)shot * a.pmlc_stride_ng * ng;
#pragma unroll
                for (int k = 0; k < 9; ++k) pc[k] = pload<BUF>(pmlc + k * ng, pnb, g32);
#pragma unroll
                for (int c = 0; c < 27; ++c) cur[c] = pload<BUF>(pin + c * ng, pnb, g32);
                if constexpr (RC == 0) {
#pragma unroll
                    for (int c = 0; c < 27; ++c) bse[c] = pload<BUF>(pbase + c * ng, pnb_base, g32);
                }
                typedef R r4 __attribute__((ext_vector_type(4)));
                const r4 *m4 = reinterpret_cast<const r4 *>(a.emet + (size_t)e * 12);
                const r4 ma = m4[0], mb = m4[1], mc = m4[2];
#pragma unroll
                for (int k = 0; k < 4; ++k) { mv[k] = ma[k]; mv[4 + k] = mb[k]; }
                mv[8] = mc[0];
                lam = matc[(size_t)e * 8 + 3]; mu = matc[(size_t)e * 8 + 4]; irho = matc[(size_t)e * 8 + 6];
            }
            if constexpr (!S::FW) stage_elements(t, NTHR);
            if constexpr (LASTF) {
                if (a.pml_compat) {
#pragma unroll
                    for (int r = 0; r < NLS; ++r)
                        if (t + r * NNT < NLASTF) sC[t + r * NNT] = lst[r];
                }
            }
            if (node_thr) node_store();
            block_barrier();
            R cf[27];
            if (node_thr) {
                // modified fluxes and the ADE update of f',g',h', as in
                // stage_kernel (src/timeloopMod.f90:399-405, src/rungekuttaMod.f90:52-63)
                R Fm[9], Gm[9], Hm[9];
                elastic_flux_node(qs, -(lam + R(2) * mu), -lam, -mu, -irho, Fm, Gm, Hm);
                const RkStage<R> rs = rk_stage<R, RC>(a.scheme, a.irk, a.w13, a.w23, a.lsa, a.lsb);
                const bool on = !a.pml_on || a.pml_on[shot] != 0;
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    R pv[9];
                    const R al = on ? pc[d] : R(0), dk = on ? pc[3 + d] : R(0);
                    const R rk = on ? R(1) / pc[6 + d] : R(1);
                    const R *FF = d == 0 ? Fm : (d == 1 ? Gm : Hm);
                    const int skip = d == 0 ? 4 : (d == 1 ? 5 : 3);   // identically zero
#pragma unroll
                    for (int i = 0; i < 9; ++i) {
                        const int c = d * 9 + i;
                        R c0 = on ? cur[c] : R(0);
                        if constexpr (RC == 2) {
                            const R dadt1 = -al * c0 - dk * (c0 + sLast1[c * NP + j]);
                            R none = 0;
                            c0 = rk_update<R, false, false, 1>(rs, c0, none, dadt1, dt);
                        }
                        const R mod = (c0 + FF[i]) * rk;
#pragma unroll
                        for (int o = 0; o < 3; ++o) {
                            const R m = mv[3 * o + d];
                            if (d == 0) cf[o * 9 + i] = i != skip ? m * mod : R(0);
                            else if (i != skip) cf[o * 9 + i] = cf[o * 9 + i] + m * mod;
                        }
                        if constexpr (RC == 1) continue;
                        const R lastv = sLast[c * NP + j];
                        const R u = RC == 2 || a.pml_compat ? lastv : mod;
                        const R dadt = -al * c0 - dk * (c0 + u);
                        if constexpr (RC == 2) pv[i] = rk_update<R, false, false, 2>(rs, c0, cur[c], dadt, dt);
                        else if constexpr (RC == 0) pv[i] = rk_update<R, LS>(rs, c0, bse[c], dadt, dt);
                    }
                    if (RC != 1 && valid) {
#pragma unroll
                        for (int i = 0; i < 9; ++i) pstore<BUF>(pout + (d * 9 + i) * ng, pnb, g32, pv[i]);
                    }
                    if constexpr (LS) {
                        if (valid) {
                            R *pres = a.pres + (size_t)shot * 27 * ng;
#pragma unroll
                            for (int i = 0; i < 9; ++i) pstore<BUF>(pres + (d * 9 + i) * ng, pnb, g32, bse[d * 9 + i]);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            block_barrier();
            if (node_thr) {
#pragma unroll
                for (int c = 0; c < 27; ++c) sC[c * NT + t] = cf[c];
            }
        }
        if constexpr (!S::FW) {
            face_load(t);
            face_flux(t);
        }
    }

    // ---- the product -----------------------------------------------------
    constexpr int RTV = S::RTV, CTL = S::CTL;
    if constexpr (F64) {
        // Wave w takes row tiles RW (w % RG).. and column tiles w / RG, w / RG +
        // CG, ..: at value s of its column's list a lane supplies one B value,
        // and the operator's fragments of the wave's row tiles load PREF values
        // ahead.
        constexpr int RW = S::RW, RG = S::RG, CW = S::CW, CG = S::CG, KT = S::KT, PREF = 12 / RW;
        typedef double f64x4_t __attribute__((ext_vector_type(4)));
        const int r0 = (w % RG) * RW, c0 = w / RG;
        const double *ak = reinterpret_cast<const double *>(a.AK) + lane;
        double af[PREF][RW];
        auto load_a = [&](int s) {
#pragma unroll
            for (int r = 0; r < RW; ++r) af[s % PREF][r] = ak[(s * RTV + (r0 + r < RTV ? r0 + r : RTV - 1)) * 64];
        };
#pragma unroll
        for (int s = 0; s < PREF; ++s) load_a(s);
        __syncthreads();   // q, flux rows and face values are in LDS
        f64x4_t acc[CW][RW];
        R K[CW][9], C[CW][3];
        int row[CW][3], lrow[CW];
#pragma unroll
        for (int c = 0; c < CW; ++c) {
            const int col = (c0 + c * CG) * 16 + (lane & 15);
            const bool cok = col < S::NCT;
            const int ce = cok ? col / NCOL : 0, cc = cok ? col - (col / NCOL) * NCOL : 0;
            lrow[c] = S::OFF_F + (ce * NCOL + cc) * SFN + (lane >> 4);
            const R *el = sE + ce * kAffElem;
            const bool flux = PML && cc < 9;   // stored contravariant fluxes
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const R cof = el[AE_COEF + (int)((kCofs[k] >> (4 * cc)) & 15)];
                row[c][k] = (flux ? (9 + 9 * k + cc) : (int)((kRows[k] >> (4 * cc)) & 15)) * NT + ce * NP;
#pragma unroll
                for (int o = 0; o < 3; ++o) {
                    const R m = el[AE_MET + 3 * o + k] * cof;
                    K[c][3 * o + k] = flux ? (o == k ? R(1) : R(0)) : m;
                }
            }
#pragma unroll
            for (int r = 0; r < RW; ++r) acc[c][r] = f64x4_t{0, 0, 0, 0};
        }
#pragma unroll
        for (int s = 0; s < KT; ++s) {
#pragma unroll
            for (int c = 0; c < CW; ++c) {
                R v;
                if (s < S::KSV) {
                    if (s % 3 == 0) {
                        const int m = 4 * (s / 3) + (lane >> 4);
                        const int mm = 4 * (s / 3) + 3 < NP || m < NP ? m : 0;   // the operator is zero beyond Np
                        const R x = lds[row[c][0] + mm], y = lds[row[c][1] + mm], z = lds[row[c][2] + mm];
#pragma unroll
                        for (int o = 0; o < 3; ++o)
                            C[c][o] = K[c][3 * o] * x + K[c][3 * o + 1] * y + K[c][3 * o + 2] * z;
                    }
                    v = C[c][s % 3];
                } else {
                    v = lds[lrow[c] + 4 * (s - S::KSV)];
                }
#pragma unroll
                for (int r = 0; r < RW; ++r) acc[c][r] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[s % PREF][r], v, acc[c][r], 0, 0, 0);
            }
            if (s + PREF < KT) load_a(s + PREF);
            if (s % 3 == 2) __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();   // everything before the element constants is dead
        // accumulator element v: node row 4v + l/16 of the row tile, column l%16
#pragma unroll
        for (int c = 0; c < CW; ++c) {
            const int col = (c0 + c * CG) * 16 + (lane & 15);
            if (col < S::NCT) {
                const int ce = col / NCOL, cc = col - ce * NCOL;
#pragma unroll
                for (int r = 0; r < RW; ++r)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int node = (r0 + r) * 16 + 4 * v + (lane >> 4);
                        if (node < NP) sV[(ce * NP + node) * NV + cc] = acc[c][r][v];
                    }
            }
        }
    } else {
    // Each wave takes column tiles w, w+4, .. against all row tiles, TG of
    // them at a time.  Unit u = (step u / RTV, row tile u % RTV): its three
    // A parts load PREF units ahead.
    constexpr int CPW = S::CPW, NU = S::NS * RTV, PREF = 2;
    const u32x4_t *ak = reinterpret_cast<const u32x4_t *>(a.AK) + lane;
    bf16x8_t af[PREF + 1][3];
    auto load_a = [&](int u) {
#pragma unroll
        for (int p = 0; p < 3; ++p) af[u % (PREF + 1)][p] = __builtin_bit_cast(bf16x8_t, ak[(u * 3 + p) * 64]);
    };
#pragma unroll
    for (int u = 0; u < PREF; ++u) load_a(u);
    __syncthreads();   // q, flux rows and face values are in LDS

    f32x4_t acc[CPW][RTV];
    // TC column tiles from the wave's tile C0 on
    auto product = [&](auto c0_, auto tc_) {
        constexpr int C0 = decltype(c0_)::value, TC = decltype(tc_)::value;
        if constexpr (C0 > 0) {
#pragma unroll
            for (int u = 0; u < PREF; ++u) load_a(u);
        }
        float K[TC][9], C[TC][3];
        f32x4_t lo[TC][RTV];
        int row[TC][3], lrow[TC];
#pragma unroll
        for (int c = 0; c < TC; ++c) {
            const int col = (w + (C0 + c) * NW) * 16 + (lane & 15);
            const bool cok = col < S::NCT;
            const int ce = cok ? col / NCOL : 0, cc = cok ? col - (col / NCOL) * NCOL : 0;
            lrow[c] = S::OFF_F + (ce * NCOL + cc) * SFN + (lane >> 4);
            const float *el = sE + ce * kAffElem;
            const bool flux = PML && cc < 9;   // stored contravariant fluxes
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const float cof = el[AE_COEF + (int)((kCofs[k] >> (4 * cc)) & 15)];
                row[c][k] = (flux ? (9 + 9 * k + cc) : (int)((kRows[k] >> (4 * cc)) & 15)) * NT + ce * NP;
#pragma unroll
                for (int o = 0; o < 3; ++o) {
                    const float m = el[AE_MET + 3 * o + k] * cof;
                    K[c][3 * o + k] = flux ? (o == k ? 1.f : 0.f) : m;
                }
            }
#pragma unroll
            for (int r = 0; r < RTV; ++r) acc[C0 + c][r] = lo[c][r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int st = 0; st < S::NS; ++st) {
            bf16x8_t b[TC][3];
#pragma unroll
            for (int c = 0; c < TC; ++c) {
                // the lane's eight values of the step: C_o at nodes 4 ks + l/16
                // (s = 3 ks + o), then face values 4 ks + l/16
                float v[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int s = 8 * st + i;
                    if (s < S::KSV) {
                        if (s % 3 == 0) {
                            const int m = 4 * (s / 3) + (lane >> 4);
                            const int mm = 4 * (s / 3) + 3 < NP || m < NP ? m : 0;   // the operator is zero beyond Np
                            const float x = lds[row[c][0] + mm], y = lds[row[c][1] + mm], z = lds[row[c][2] + mm];
#pragma unroll
                            for (int o = 0; o < 3; ++o)
                                C[c][o] = K[c][3 * o] * x + K[c][3 * o + 1] * y + K[c][3 * o + 2] * z;
                        }
                        v[i] = C[c][s % 3];
                    } else {
                        v[i] = s < S::KT ? lds[lrow[c] + 4 * (s - S::KSV)] : 0.f;
                    }
                }
                split3(v, b[c]);
            }
#pragma unroll
            for (int r = 0; r < RTV; ++r) {
                const int u = st * RTV + r;
                if (u + PREF < NU) load_a(u + PREF);
                const bf16x8_t(&x)[3] = af[u % (PREF + 1)];
#pragma unroll
                for (int c = 0; c < TC; ++c) {
                    lo[c][r] = mfma_bf16(x[0], b[c][2], lo[c][r]);
                    lo[c][r] = mfma_bf16(x[2], b[c][0], lo[c][r]);
                    lo[c][r] = mfma_bf16(x[1], b[c][1], lo[c][r]);
                    lo[c][r] = mfma_bf16(x[0], b[c][1], lo[c][r]);
                    lo[c][r] = mfma_bf16(x[1], b[c][0], lo[c][r]);
                    acc[C0 + c][r] = mfma_bf16(x[0], b[c][0], acc[C0 + c][r]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int c = 0; c < TC; ++c)
#pragma unroll
            for (int r = 0; r < RTV; ++r) acc[C0 + c][r] = acc[C0 + c][r] + lo[c][r];
    };
    // the wave's last tile may not exist
    auto tiles = [&](auto self, auto c0_) {
        constexpr int C0 = decltype(c0_)::value, N = CPW - C0 < S::TG ? CPW - C0 : S::TG;
        if constexpr (N > 0) {
            if constexpr (CTL % NW == 0 || C0 + N < CPW) {
                product(c0_, std::integral_constant<int, N>{});
                self(self, std::integral_constant<int, C0 + N>{});
            } else if (w + (CPW - 1) * NW < CTL) {
                product(c0_, std::integral_constant<int, N>{});
            } else if constexpr (N > 1) {
                product(c0_, std::integral_constant<int, N - 1>{});
            }
        }
    };
    tiles(tiles, std::integral_constant<int, 0>{});
    __syncthreads();   // everything before the element constants is dead
    // accumulator element v: node row 4*(l/16)+v of the row tile, column l%16
#pragma unroll
    for (int c = 0; c < CPW; ++c) {
        const int col = (w + c * NW) * 16 + (lane & 15);
        if (col < S::NCT) {
            const int ce = col / NCOL, cc = col - ce * NCOL;
#pragma unroll
            for (int r = 0; r < RTV; ++r)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int node = r * 16 + 4 * (lane >> 4) + v;
                    if (node < NP) sV[(ce * NP + node) * NV + cc] = acc[c][r][v];
                }
        }
    }
    }

    // ---- node threads: memory variables, sources, Runge-Kutta update -------
    R th[ATT ? 18 : 1], thb[ATT && RC == 0 ? 18 : 1], gi[ATT && RC == 2 ? 6 : 1], avc[ATT ? 9 : 1];
    R qb[9], alo[9], blo[9];
    const bool comp = a.qlo_out != nullptr;
    const unsigned nel = (unsigned)(ng / NP);
    if (node_thr) {
        if constexpr (ATT) {
            const R *thin = a.thin + (size_t)shot * 18 * ng;
            const R *av = a.anel + (size_t)shot * a.anel_stride;
#pragma unroll
            for (int c = 0; c < 18; ++c) th[c] = pload<BUF>(thin + c * ng, pnb, g32);
            if constexpr (RC == 2) {
#pragma unroll
                for (int c = 0; c < 6; ++c) gi[c] = pload<BUF>(a.rate_in + ((size_t)shot * 6 + c) * ng, pnb, g32);
            }
            if constexpr (RC == 0) {
#pragma unroll
                for (int c = 0; c < 18; ++c) thb[c] = pload<BUF>(a.thbase + ((size_t)shot * 18 + c) * ng, pnb_base, g32);
            }
#pragma unroll
            for (int c = 0; c < 9; ++c) avc[c] = pload<BUF>(av, nel * (unsigned)(NMB * 3 * sizeof(R)), (unsigned)e * (NMB * 3) + c);
        }
        if constexpr (RC != 1) {
#pragma unroll
            for (int f = 0; f < 9; ++f) qb[f] = pload<BUF>(qbase + f * ng, pnb_base, g32);
        }
        if (comp) {
#pragma unroll
            for (int f = 0; f < 9; ++f) alo[f] = pload<BUF>(a.qlo_in + ((size_t)shot * 9 + f) * ng, pnb, g32);
            if constexpr (RC != 1) {
#pragma unroll
                for (int f = 0; f < 9; ++f) blo[f] = pload<BUF>(a.qlo_base + ((size_t)shot * 9 + f) * ng, pnb_base, g32);
            }
        }
    }
    __syncthreads();
    R qnew[9], rhs[9];
    if (node_thr) {
        const R *v = sV + t * NV;
#pragma unroll
        for (int i = 0; i < 9; ++i) rhs[i] = v[i];
        const RkStage<R> rs = rk_stage<R, RC>(a.scheme, a.irk, a.w13, a.w23, a.lsa, a.lsb);
        if constexpr (ATT) {
            R gn[6];
#pragma unroll
            for (int c = 0; c < 6; ++c) gn[c] = v[9 + c];
            // one mechanism at a time (src/timeloopMod.f90:426-461): every
            // memory variable advances by w (g - theta)
#pragma unroll
            for (int i = 0; i < NMB; ++i) {
                const R wl = a.wl[i], a1 = avc[i * 3 + 0], a2 = avc[i * 3 + 1], a3 = avc[i * 3 + 2];
                R tm[6];
#pragma unroll
                for (int c = 0; c < 6; ++c) {
                    tm[c] = th[i * 6 + c];
                    if constexpr (RC == 2) {
                        R none = 0;
                        tm[c] = rk_update<R, false, false, 1>(rs, tm[c], none, wl * (gi[c] - tm[c]), dt);
                    }
                }
                rhs[0] = rhs[0] + a3 * tm[0] + a1 * (tm[1] + tm[2]);
                rhs[1] = rhs[1] + a3 * tm[1] + a1 * (tm[2] + tm[0]);
                rhs[2] = rhs[2] + a3 * tm[2] + a1 * (tm[0] + tm[1]);
                rhs[3] = rhs[3] + a2 * tm[3];
                rhs[4] = rhs[4] + a2 * tm[4];
                rhs[5] = rhs[5] + a2 * tm[5];
                if constexpr (RC != 1) {
#pragma unroll
                    for (int c = 0; c < 6; ++c) {
                        const int k = i * 6 + c;
                        const R r = wl * (gn[c] - tm[c]);
                        if constexpr (RC == 2) th[k] = rk_update<R, false, WEIGHTED, 2>(rs, tm[c], th[k], r, dt);
                        else th[k] = rk_update<R, LS, WEIGHTED>(rs, tm[c], thb[k], r, dt);
                    }
                }
            }
            if (valid) {
                if constexpr (RC == 1) {
#pragma unroll
                    for (int c = 0; c < 6; ++c) pstore<BUF>(a.rate_out + ((size_t)shot * 6 + c) * ng, pnb, g32, gn[c]);
                } else {
#pragma unroll
                    for (int k = 0; k < 18; ++k) pstore<BUF>(a.thout + ((size_t)shot * 18 + k) * ng, pnb, g32, th[k]);
                }
                if constexpr (LS) {
#pragma unroll
                    for (int k = 0; k < 18; ++k) pstore<BUF>(a.thres + ((size_t)shot * 18 + k) * ng, pnb, g32, thb[k]);
                }
            }
        }
        if (valid) add_sources<NP>(a, shot, j, src_first, it_step, rhs);
        if (!LS && comp) {
            const int scheme = RC ? 2 : a.scheme, irk = RC ? RC : a.irk;
#pragma unroll
            for (int f = 0; f < 9; ++f) {
                R lo;
                const R b = RC == 1 ? qs[f] : qb[f], bl = RC == 1 ? alo[f] : blo[f];
                rk_combine_comp<R>(scheme, irk, qs[f], alo[f], b, bl, rhs[f], dt, a.w13, a.w23, qnew[f], lo);
                if (valid) {
                    pstore<BUF>(qout + f * ng, pnb, g32, qnew[f]);
                    pstore<BUF>(a.qlo_out + ((size_t)shot * 9 + f) * ng, pnb, g32, lo);
                }
            }
        } else {
#pragma unroll
            for (int f = 0; f < 9; ++f) {
                if constexpr (RC == 1) qb[f] = R(0);
                qnew[f] = rk_update<R, LS, WEIGHTED, RC>(rs, qs[f], qb[f], rhs[f], dt);
            }
            if (valid) {
#pragma unroll
                for (int f = 0; f < 9; ++f) pstore<BUF>(qout + f * ng, pnb, g32, qnew[f]);
                if constexpr (LS) {
#pragma unroll
                    for (int f = 0; f < 9; ++f) pstore<BUF>(a.qres + ((size_t)shot * 9 + f) * ng, pnb, g32, qb[f]);
                }
            }
        }
    }

    // ---- post-step (src/timeloopMod.f90:482-516) ---------------------------
    if (RC == 1) return;
    if (RC == 2 || a.last_stage) {
        if (valid) {
            if (a.u_full) {
#pragma unroll
                for (int c = 0; c < 3; ++c) a.u_full[c * ng + g] = a.u_full[c * ng + g] + dt * qnew[6 + c];
            }
            if (rec_slot_e >= 0) update_receiver<NP>(a, shot, j, rec_slot_e, dt, qnew, rhs);
        }
        if (a.blk_energy) {
            const R rho = node_thr ? matc[(size_t)e * 8 + 2] : R(1);
            block_energy<ORDER, EB, NTHR>(a, lds, shot, eblk, node_thr, valid, t, eb, j, e, rho, qnew);
        }
    }
}

}  // namespace nexd
