// Host-side conversion of the reference's arrays (Fortran column-major,
// 1-based) into the device layout of the stage kernels, with the checks the
// C-ABI promises.  Shared by the single-shot and the batched contexts.
#pragma once
#include <cstring>
#include <string>
#include <vector>

namespace nexd {

struct OpsHost {
    std::vector<double> D;    // [3][NP][NP]
    std::vector<double> LT;   // [NFP][NP]
    std::vector<double> M;    // [NP][NP]
    std::vector<int> fm;      // [4][NPF] 0-based
};

inline std::string convert_operators(int np, int npf, const double *dr, const double *ds, const double *dt,
                                     const double *lift, const double *mass, const int *fmask, OpsHost &o) {
    if (!dr || !ds || !dt || !lift || !mass || !fmask) return "null operator";
    const int nfp = 4 * npf;
    o.D.assign((size_t)3 * np * np, 0.0);
    o.LT.assign((size_t)nfp * np, 0.0);
    o.M.assign((size_t)np * np, 0.0);
    o.fm.assign((size_t)4 * npf, 0);
    const double *src[3] = {dr, ds, dt};
    for (int d = 0; d < 3; ++d)
        for (int i = 0; i < np; ++i)
            for (int m = 0; m < np; ++m) o.D[((size_t)d * np + i) * np + m] = src[d][(size_t)m * np + i];
    for (int k = 0; k < nfp; ++k)
        for (int j = 0; j < np; ++j) o.LT[(size_t)k * np + j] = lift[(size_t)k * np + j];
    for (int i = 0; i < np; ++i)
        for (int k = 0; k < np; ++k) o.M[(size_t)i * np + k] = mass[(size_t)k * np + i];
    for (int f = 0; f < 4; ++f)
        for (int i = 0; i < npf; ++i) {
            const int v = fmask[f * npf + i] - 1;
            if (v < 0 || v >= np) return "fmask entry out of range";
            o.fm[f * npf + i] = v;
        }
    return "";
}

// Dr, Ds, Dt in the A-operand order of the 16x16x4 MFMA (row tile rt,
// k-step ks, lane l -> [rt][ks][l]); lane l of k-step ks holds tile row
// l%16 at column 4ks + l/16 (zero beyond Np).  Accumulator element v of a
// lane in lane group g = l/16 is tile row 4v + g (FP64 instruction) or
// 4g + v (FP32).  The rows are packed so that each lane group owns nodes
// g, g+4, g+8, ... with their three operator rows in order: element v of
// row tile rt is row q = 4rt + v of the group, node g + 4*(q/3), operator
// q%3.  A lane thus receives the three derivatives of each of its nodes,
// across consecutive tiles, with no padding row (3*ceil(Np/4) rows per
// group in ceil(3*ceil(Np/4)/4) tiles).
inline std::vector<double> mfma_operator_fragments(const std::vector<double> &D, int np, bool f64) {
    const int npg = (np + 3) / 4, nt = (3 * npg + 3) / 4, nk = (np + 3) / 4;
    std::vector<double> out((size_t)nt * nk * 64, 0.0);
    for (int rt = 0; rt < nt; ++rt)
        for (int ks = 0; ks < nk; ++ks)
            for (int l = 0; l < 64; ++l) {
                const int i = l % 16, m = 4 * ks + l / 16;
                const int g = f64 ? i % 4 : i / 4, v = f64 ? i / 4 : i % 4;
                const int q = 4 * rt + v, node = g + 4 * (q / 3), op = q % 3;
                if (node < np && m < np) out[((size_t)rt * nk + ks) * 64 + l] = D[((size_t)op * np + node) * np + m];
            }
    return out;
}

// [Dr | Ds | Dt] (Np x 3Np) in the A-operand order of the 16x16x4 MFMA, for
// the volume term of PML elements, which differentiates contravariant fluxes
// (each column needs sum_o D_o C_o): row tile rt holds nodes 16rt..16rt+15;
// k-step ks covers operator o = ks / KS at nodes 4(ks % KS)..+3 (KS =
// ceil(Np/4)); lane l holds node 16rt + l%16 at column 4(ks % KS) + l/16 of
// operator o (zero beyond Np).  Layout [rt][ks][l].
inline std::vector<double> mfma_operator_fragments_k(const std::vector<double> &D, int np) {
    const int nt = (np + 15) / 16, kso = (np + 3) / 4, nk = 3 * kso;
    std::vector<double> out((size_t)nt * nk * 64, 0.0);
    for (int rt = 0; rt < nt; ++rt)
        for (int ks = 0; ks < nk; ++ks)
            for (int l = 0; l < 64; ++l) {
                const int op = ks / kso, m = 4 * (ks % kso) + l / 16, node = 16 * rt + l % 16;
                if (node < np && m < np) out[((size_t)rt * nk + ks) * 64 + l] = D[((size_t)op * np + node) * np + m];
            }
    return out;
}

// LIFT in the A-operand order of the 16x16x4 MFMA: row tile mt holds nodes
// 16mt..16mt+15, k-step ks face nodes 4ks..4ks+3; lane l holds node
// 16mt + l%16 at face node 4ks + l/16 (zero beyond Np).  LT is [NFP][NP]
// with LT[k][j] = LIFT(j,k).
inline std::vector<double> mfma_lift_fragments(const std::vector<double> &LT, int np, int nfp) {
    const int nt = (np + 15) / 16, nk = nfp / 4;
    std::vector<double> out((size_t)nt * nk * 64, 0.0);
    for (int mt = 0; mt < nt; ++mt)
        for (int ks = 0; ks < nk; ++ks)
            for (int l = 0; l < 64; ++l) {
                const int i = 16 * mt + l % 16, k = 4 * ks + l / 16;
                if (i < np) out[((size_t)mt * nk + ks) * 64 + l] = LT[(size_t)k * np + i];
            }
    return out;
}

// the nearest bfloat16 (finite values), its bits
inline unsigned short bf16_bits(double x) {
    const float f = (float)x;
    unsigned u;
    std::memcpy(&u, &f, 4);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}
inline double bf16_value(unsigned short b) {
    const unsigned u = (unsigned)b << 16;
    float f;
    std::memcpy(&f, &u, 4);
    return f;
}

// [Dr | Ds | Dt | LIFT] for the affine kernels, in the A-operand order of the
// 16x16x32 BF16 MFMA, every entry as the sum of three bfloat16 (27 bits):
// [step][row tile][part][lane][8].  Row tile rt holds nodes 16rt..16rt+15
// (lane l: node 16rt + l%16).  The k index is dealt so that a lane of the B
// operand supplies values of its own: entry i of step st is value s = 8 st + i
// of lane group l/16, for s = 3 ks + o (ks < ceil(Np/4)) operator o at node
// 4ks + l/16, then LIFT at face nodes 4ks + l/16; zero beyond Np and past the
// last value.  LIFT enters as the general FP32 kernel has it, rounded to single
// precision: its rounding and those of face scales, normals, material and step
// act like another wave speed (4.7e-6, 4.3e-6, 2.6e-6, 0.9e-6 and 1.6e-6 of the
// seismograms after 101 steps at N = 2), and partly offset each other.
inline std::vector<unsigned short> mfma_affine_fragments(const std::vector<double> &D, const std::vector<double> &LT,
                                                         int np, int nfp) {
    const int nt = (np + 15) / 16, ksv = 3 * ((np + 3) / 4), kt = ksv + nfp / 4, ns = (kt + 7) / 8;
    std::vector<unsigned short> out((size_t)ns * nt * 3 * 512, 0);
    for (int s = 0; s < kt; ++s)
        for (int rt = 0; rt < nt; ++rt)
            for (int l = 0; l < 64; ++l) {
                const int node = 16 * rt + l % 16, k = 4 * (s < ksv ? s / 3 : s - ksv) + l / 16;
                if (node >= np || (s < ksv && k >= np)) continue;
                double x = s < ksv ? D[((size_t)(s % 3) * np + node) * np + k] : (double)(float)LT[(size_t)k * np + node];
                for (int p = 0; p < 3; ++p) {
                    const unsigned short b = bf16_bits(x);
                    out[((((size_t)(s / 8) * nt + rt) * 3 + p) * 64 + l) * 8 + s % 8] = b;
                    x -= bf16_value(b);
                }
            }
    return out;
}

// The same in FP64, for the 16x16x4 MFMA: [value s][row tile][lane], s and the
// lanes as above.
inline std::vector<double> mfma_affine_fragments_f64(const std::vector<double> &D, const std::vector<double> &LT, int np,
                                                     int nfp) {
    const int nt = (np + 15) / 16, ksv = 3 * ((np + 3) / 4), kt = ksv + nfp / 4;
    std::vector<double> out((size_t)kt * nt * 64, 0.0);
    for (int s = 0; s < kt; ++s)
        for (int rt = 0; rt < nt; ++rt)
            for (int l = 0; l < 64; ++l) {
                const int node = 16 * rt + l % 16, k = 4 * (s < ksv ? s / 3 : s - ksv) + l / 16;
                if (node >= np || (s < ksv && k >= np)) continue;
                out[((size_t)s * nt + rt) * 64 + l] = s < ksv ? D[((size_t)(s % 3) * np + node) * np + k] : LT[(size_t)k * np + node];
            }
    return out;
}

// The mass matrix in the A-operand order of the 16x16x4 MFMA (the energy's
// products M y): row tile mt holds nodes 16mt..16mt+15, k-step ks nodes
// 4ks..4ks+3; lane l holds M(16mt + l%16, 4ks + l/16), zero beyond Np.  M is
// [NP][NP] row-major.
inline std::vector<double> mfma_mass_fragments(const std::vector<double> &M, int np) {
    const int nt = (np + 15) / 16, nk = (np + 3) / 4;
    std::vector<double> out((size_t)nt * nk * 64, 0.0);
    for (int mt = 0; mt < nt; ++mt)
        for (int ks = 0; ks < nk; ++ks)
            for (int l = 0; l < 64; ++l) {
                const int i = 16 * mt + l % 16, k = 4 * ks + l / 16;
                if (i < np && k < np) out[((size_t)mt * nk + ks) * 64 + l] = M[(size_t)i * np + k];
            }
    return out;
}

struct MeshHost {
    std::vector<double> metric;  // [9][nglob]
    std::vector<double> jac;     // [nglob]
    std::vector<double> fscale;  // [nelem][NFP]
    std::vector<double> frame;   // [nelem][4][9]
    std::vector<int> nbr;        // [nelem][4][NPF]
    std::vector<int> ftype;      // [nelem][4]
};

// err is "" on success; unsupported features are reported with a leading '!'
inline std::string convert_mesh(int nelem, int np, int npf, const std::vector<int> &fm, const int *ibool,
                                const double *const metric_in[9], const double *jacobian, const double *fscale,
                                const int *neighbor, const int *face, const int *ibt, const int *ibn,
                                const double *nnormal, const double *stangential, const double *ttangential,
                                MeshHost &m) {
    for (int k = 0; k < 9; ++k)
        if (!metric_in[k]) return "null mesh array";
    if (!ibool || !jacobian || !fscale || !neighbor || !face || !ibt || !ibn || !nnormal || !stangential ||
        !ttangential)
        return "null mesh array";
    const size_t ng = (size_t)nelem * np;
    const int nfp = 4 * npf;
    for (size_t i = 0; i < ng; ++i)
        if (ibool[i] != (int)i + 1) return "!ibool must be (ie-1)*Np+j";
    m.metric.resize(9 * ng);
    for (int k = 0; k < 9; ++k) std::memcpy(m.metric.data() + k * ng, metric_in[k], sizeof(double) * ng);
    m.jac.assign(jacobian, jacobian + ng);
    m.fscale.assign(fscale, fscale + (size_t)nelem * nfp);
    m.frame.resize((size_t)nelem * 36);
    m.nbr.resize((size_t)nelem * 4 * npf);
    m.ftype.resize((size_t)nelem * 4);
    for (int e = 0; e < nelem; ++e) {
        for (int f = 0; f < 4; ++f) {
            for (int k = 0; k < 3; ++k) {
                m.frame[(e * 4 + f) * 9 + k] = nnormal[(e * 4 + f) * 3 + k];
                m.frame[(e * 4 + f) * 9 + 3 + k] = stangential[(e * 4 + f) * 3 + k];
                m.frame[(e * 4 + f) * 9 + 6 + k] = ttangential[(e * 4 + f) * 3 + k];
            }
            const int n = neighbor[e * 4 + f], fc = face[e * 4 + f];
            for (int i = 0; i < npf; ++i) {
                const size_t idx = ((size_t)e * 4 + f) * npf + i;
                if ((size_t)ibt[idx] != (size_t)e * np + fm[f * npf + i] + 1)
                    return "!ibt must be ibool(fmask(:,is),ie)";
            }
            if (n > 0) {
                if (n > nelem) return "neighbor out of range";
                if (fc < 1 || fc > 4) return "face of an interior face must be 1..4";
                m.ftype[e * 4 + f] = fc - 1;
                for (int i = 0; i < npf; ++i) {
                    const size_t idx = ((size_t)e * 4 + f) * npf + i;
                    const int v = ibn[idx] - 1;
                    if (v < 0 || (size_t)v >= ng) return "ibn out of range";
                    m.nbr[idx] = v;
                }
            } else if (n == 0) {
                if (fc != -1 && fc != -2) return "boundary face must be free (-1) or absorbing (-2)";
                m.ftype[e * 4 + f] = fc;
                for (int i = 0; i < npf; ++i) m.nbr[((size_t)e * 4 + f) * npf + i] = -1;
            } else {
                return "!partition interfaces (neighbor == -1) are not supported";
            }
        }
    }
    return "";
}

// inverse of a 3 x 3 matrix (row-major); false if it is singular
inline bool invert3(const double *a, double *r) {
    const double c0 = a[4] * a[8] - a[5] * a[7], c1 = a[5] * a[6] - a[3] * a[8], c2 = a[3] * a[7] - a[4] * a[6];
    const double d = a[0] * c0 + a[1] * c1 + a[2] * c2, i = 1.0 / d;
    r[0] = c0 * i; r[1] = (a[2] * a[7] - a[1] * a[8]) * i; r[2] = (a[1] * a[5] - a[2] * a[4]) * i;
    r[3] = c1 * i; r[4] = (a[0] * a[8] - a[2] * a[6]) * i; r[5] = (a[2] * a[3] - a[0] * a[5]) * i;
    r[6] = c2 * i; r[7] = (a[1] * a[6] - a[0] * a[7]) * i; r[8] = (a[0] * a[4] - a[1] * a[3]) * i;
    return d != 0;
}

// The geometry of a straight-sided mesh, one set per element, for the affine
// kernels.
//
// The Jacobian dx/d(r,s,t) of such an element is constant, but the reference
// forms it with its Dr, Ds, Dt, whose rows differentiate a linear function to
// about 1.5e-7 only (single-precision literals): J(i) = G (I + E(i)) at node i,
// with E the same for every element, as the node coordinates are linear in r,
// s, t.  Its derivatives are then
//   sum_o M(i)_ok D_o f = sum_p Ginv_pk sum_o [(I + E(i))^-1]_op D_o f,   M = J^-1:
// the constant metric Ginv with operators whose rows are combined once.  G is
// the mean of J over the element's nodes, E comes from the first element.
struct AffineHost {
    std::vector<double> emet;    // [nelem][12] Ginv
    std::vector<double> fgeo;    // [nelem][4][4] normal, half the mean face scale
    std::vector<int> nbrt;       // [nelem][NFP] neighbour node, -1 free, -2 absorbing
    std::vector<double> comb;    // [np][3][3] (I + E)^-1 of each node, rows o
};

// Whether the mesh is of that kind: every element's metric is the first
// element's pattern times a constant, for the FP32 kernels to 1e-6 (relative),
// for the FP64 ones to 1e-11.  The meshes of the host set-up are to 3e-14 to
// 1e-12, growing with the mesh: that is the rounding of the node coordinates.
// (Against the same vertices in extended precision the set-up's metric at the
// nodes and this one differ equally: rms 4.7e-14 and 4.8e-14 on 2,352 tets at N
// = 3, 1.9e-13 and 2.0e-13 on 8,712 at N = 4.)  The FP32 kernels also take one
// face scale and the normal alone: face scales equal to their mean and frames
// orthonormal to 1e-6 (the set-up's are to 2e-7).  Fills `o` if so.
inline bool affine_mesh(const MeshHost &m, int nelem, int np, int npf, bool f64, AffineHost &o) {
    constexpr double tol = 1e-6;
    const size_t ng = (size_t)nelem * np;
    const int nfp = 4 * npf;
    o.emet.assign((size_t)nelem * 12, 0.0);
    o.fgeo.resize((size_t)nelem * 16);
    o.nbrt.resize((size_t)nelem * nfp);
    o.comb.assign((size_t)np * 9, 0.0);
    std::vector<double> E((size_t)np * 9), C((size_t)np * 9);   // I + E and its inverse, [9][np]
    {
        std::vector<double> J((size_t)np * 9);
        double G[9] = {0}, Gi[9], M[9], t[9];
        for (int j = 0; j < np; ++j) {
            for (int k = 0; k < 9; ++k) M[k] = m.metric[k * ng + j];
            if (!invert3(M, &J[(size_t)j * 9])) return false;
            for (int k = 0; k < 9; ++k) G[k] += J[(size_t)j * 9 + k] / np;
        }
        if (!invert3(G, Gi)) return false;
        for (int j = 0; j < np; ++j) {
            for (int r = 0; r < 3; ++r)
                for (int q = 0; q < 3; ++q) {
                    t[3 * r + q] = 0;
                    for (int k = 0; k < 3; ++k) t[3 * r + q] += Gi[3 * r + k] * J[(size_t)j * 9 + 3 * k + q];
                    E[(size_t)(3 * r + q) * np + j] = t[3 * r + q];
                }
            if (!invert3(t, &o.comb[(size_t)j * 9])) return false;
            for (int k = 0; k < 9; ++k) C[(size_t)k * np + j] = o.comb[(size_t)j * 9 + k];
        }
    }
    for (int e = 0; e < nelem; ++e) {
        // Ginv: the mean of (I + E) M over the nodes, then M against (I + E)^-1 Ginv
        const double *M = m.metric.data() + (size_t)e * np;
        double Gi[9] = {0}, big = 0;
        for (int r = 0; r < 3; ++r)
            for (int k = 0; k < 3; ++k) {
                double s0 = 0, s1 = 0, s2 = 0;
                for (int j = 0; j < np; ++j) {
                    s0 += E[(size_t)(3 * r) * np + j] * M[k * ng + j];
                    s1 += E[(size_t)(3 * r + 1) * np + j] * M[(3 + k) * ng + j];
                    s2 += E[(size_t)(3 * r + 2) * np + j] * M[(6 + k) * ng + j];
                }
                Gi[3 * r + k] = (s0 + s1 + s2) / np;
            }
        for (int k = 0; k < 9; ++k) {
            const double b = Gi[k] < 0 ? -Gi[k] : Gi[k];
            if (!(b <= big)) big = b;   // NaN stays and fails below
        }
        const double lim = (f64 ? 1e-11 : tol) * big;
        int bad = !(big > 0);
        for (int r = 0; r < 3; ++r)
            for (int k = 0; k < 3; ++k) {
                const double *t = M + (size_t)(3 * r + k) * ng, *c = &C[(size_t)3 * r * np];
                for (int j = 0; j < np; ++j) {
                    const double d = c[j] * Gi[k] + c[np + j] * Gi[3 + k] + c[2 * np + j] * Gi[6 + k] - t[j];
                    bad |= !(d <= lim) | !(-d <= lim);
                }
            }
        if (bad) return false;
        for (int k = 0; k < 9; ++k) o.emet[(size_t)e * 12 + k] = Gi[k];
        for (int f = 0; f < 4; ++f) {
            const double *fs = m.fscale.data() + (size_t)e * nfp + f * npf, *fr = m.frame.data() + ((size_t)e * 4 + f) * 9;
            double s = 0;
            for (int i = 0; i < npf; ++i) s += fs[i];
            s /= npf;
            for (int i = 0; i < npf; ++i) {
                const double d = fs[i] - s;
                if (!f64) bad |= !(d <= tol * s) | !(-d <= tol * s);
            }
            for (int x = 0; x < 3; ++x)
                for (int y = x; y < 3; ++y) {
                    const double d = fr[3 * x] * fr[3 * y] + fr[3 * x + 1] * fr[3 * y + 1] + fr[3 * x + 2] * fr[3 * y + 2] -
                                     (x == y ? 1.0 : 0.0);
                    if (!f64) bad |= !(d <= tol) | !(-d <= tol);
                }
            double *g = o.fgeo.data() + ((size_t)e * 4 + f) * 4;
            for (int k = 0; k < 3; ++k) g[k] = fr[k];
            g[3] = 0.5 * s;
            const int ft = m.ftype[(size_t)e * 4 + f];
            const size_t at = (size_t)e * nfp + f * npf;
            for (int i = 0; i < npf; ++i) o.nbrt[at + i] = ft >= 0 ? m.nbr[at + i] : ft;
        }
        if (bad) return false;
    }
    return true;
}

// the combined operators: row i of operator p is sum_o comb(i)_op D_o(i,:)
inline std::vector<double> affine_operators(const std::vector<double> &D, int np, const std::vector<double> &comb) {
    std::vector<double> out((size_t)3 * np * np, 0.0);
    for (int p = 0; p < 3; ++p)
        for (int i = 0; i < np; ++i)
            for (int q = 0; q < 3; ++q)
                for (int j = 0; j < np; ++j)
                    out[((size_t)p * np + i) * np + j] += comb[(size_t)i * 9 + 3 * q + p] * D[((size_t)q * np + i) * np + j];
    return out;
}

inline void pml_coefficients(size_t ng, const double *ddx, const double *ddy, const double *ddz,
                             const double *alphax, const double *alphay, const double *alphaz, const double *kx,
                             const double *ky, const double *kz, std::vector<double> &pc) {
    pc.resize(9 * ng);
    for (size_t g = 0; g < ng; ++g) {
        pc[0 * ng + g] = alphax[g]; pc[1 * ng + g] = alphay[g]; pc[2 * ng + g] = alphaz[g];
        pc[3 * ng + g] = ddx[g] / kx[g]; pc[4 * ng + g] = ddy[g] / ky[g]; pc[5 * ng + g] = ddz[g] / kz[g];
        pc[6 * ng + g] = kx[g]; pc[7 * ng + g] = ky[g]; pc[8 * ng + g] = kz[g];
    }
}

}  // namespace nexd
