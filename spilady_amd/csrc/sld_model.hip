// Kernels of the parametric potential model: forward (energy, forces,
// effective fields of frozen configurations) and the parameter adjoint.
//
// The configurations are the replicas of a context; the neighbour lists are
// the context's (rcut_max, rebuilt whenever positions change). Energies are
// E = sum_i (pe_i + me_i + me0_i), the quantity whose negative gradients are
// the forces and effective fields of calculate_force_energy_CPU.cpp:33-301
// and calculate_spin_CPU.cpp:111-199. Forces and fields are written compact:
// replica r's atoms start at coff[r].
//
// Adjoint: given upstream gradients gE (per replica), gF, gH (per atom),
// grad_theta = sum gE dE/dtheta + gF . dF/dtheta + gH . dH/dtheta. With the
// pair force written as F_i = sum_j (-dudr_ij / r_ij) r_ij, the force term is
// sum over ordered pairs of c_ij d(dudr_ij)/dtheta with
// c_ij = -(gF_i . r_ij) / r_ij; the F'(rho) part of dudr is gathered per atom
// through Q_i = sum_j (c_ij + c_ji) f'(r_ij) (first pass). Pair geometry is
// recomputed in each pass, not stored.
#include <hip/hip_runtime.h>

#include "sld_kernels.h"
#include "sld_model.h"
#include "sld_model_device.h"

namespace sld {

// column k of the r value table at lookup n: the row holds the interpolation pair
__device__ __forceinline__ double lerp_pair(const double* row, int k, double ratio) {
    const double2 t = reinterpret_cast<const double2*>(row)[k];
    return t.x * ratio + t.y * (1.0 - ratio);
}

// density and F'(rho) of every atom (calculate_rho_CPU.cpp:33-92,
// calculate_force_energy_CPU.cpp:98-107; the Fe Landau coefficients do not
// depend on rho) and, for the adjoint (kQ), Q_i = sum_j (c_ij + c_ji) f'(r_ij).
//
// Four lanes an atom, lane j taking list entries j, j + 4, ...; the next
// position is on its way while a pair is added. f and f' are tables of their
// own, 8 MB of which the range below kFEnd stays in the L2s: from the 128-byte
// rows of all columns, a lane an atom, the two sums took 218 and 234 us at
// 262,144 atoms, and the adjoint made both, now 61 and, together, 81.
template <bool kQ>
__global__ __launch_bounds__(256) void k_model_rho(ModelTab M, Phys P, Dev D, double* rho_out, double* fp_out,
                                                   const int* coff, const double* gF, double* Q) {
    const int lb = xcd_block((4 * D.N + blockDim.x - 1) / blockDim.x);
    if (lb < 0) return;
    const int i = (lb * blockDim.x + threadIdx.x) >> 2, j = threadIdx.x & 3;
    if (i >= D.N) return;
    const int rr = D.arep[i];
    if (rr < 0) return;
    const Rep& R = D.rep[rr];
    const double safe_sq = R.box.safe_sq;
    const double end_sq = fmin(P.rcut_pot_sq, kFEnd * kFEnd);
    const double3 ri = d3(D.r[i]);
    const size_t c0 = kQ ? (size_t)coff[rr] - R.atom0 : 0;  // of atom a: 3 (c0 + a)
    double3 gi = make_double3(0.0, 0.0, 0.0);
    if (kQ) gi = make_double3(gF[3 * (c0 + i)], gF[3 * (c0 + i) + 1], gF[3 * (c0 + i) + 2]);
    double rho = 0.0, q = 0.0;
    const int nn = D.nbn[i];
    const int* nb = D.nb + (size_t)i * kMaxNb;
    auto entry = [&](int k) { return k < nn ? nb[k] : i; };
    int a = entry(j), next = entry(j + 4);
    double4 ra = D.r[a];
    for (int k = j; k < nn; k += 4) {
        const int at = a;
        double3 rij = sub3(ri, d3(ra));
        a = next;
        ra = D.r[a];
        next = entry(k + 8);
        double rsq = sq3(rij);
        if (__builtin_expect(rsq >= safe_sq, 0)) {
            rij = min_image(R.box, rij);
            rsq = sq3(rij);
        }
        if (rsq < end_sq) {
            const double r = sqrt(rsq);
            int n;
            double ratio;
            interp_index(r, M.in_over_rmax, n, ratio);
            rho += lerp_at(M.f, n, ratio);
            if (kQ) {
                const double* g = gF + 3 * (c0 + at);
                q += -dot3(sub3(gi, make_double3(g[0], g[1], g[2])), rij) / r * lerp_at(M.df, n, ratio);
            }
        }
    }
    rho = quad_sum(rho);
    if (kQ) q = quad_sum(q);
    if (j == 0) {
        int n;
        double ratio;
        interp_index(rho, M.in_over_rhomax, n, ratio);
        rho_out[i] = rho;
        fp_out[i] = lerp_tab(M.h, kMHStride, MH_DF, n, ratio);
        if (kQ) Q[i] = q;
    }
}
template __global__ void k_model_rho<false>(ModelTab, Phys, Dev, double*, double*, const int*, const double*, double*);
template __global__ void k_model_rho<true>(ModelTab, Phys, Dev, double*, double*, const int*, const double*, double*);

// Energies, forces and fields: four lanes an atom, blocks of kFwdAtoms atoms,
// which are the rows of the energy's partial sums. 262,144 atoms take 135 us, a
// line of the 128 MB table for each of 5.8 M pairs (5.5 TB/s); a lane an atom,
// whose pairs waited for one another, took 265.
__global__ __launch_bounds__(4 * kFwdAtoms) void k_model_forward(ModelTab M, Phys P, Dev D, const double* rho,
                                                       const double* fp, const int* coff, double* F,
                                                       double* H, double* partials) {
    const int nblocks = (D.N + kFwdAtoms - 1) / kFwdAtoms;
    const int lb = xcd_block(nblocks);
    if (lb < 0) return;  // whole padding block
    const int i = lb * kFwdAtoms + (threadIdx.x >> 2), lane4 = threadIdx.x & 3;
    double acc = 0.0;
    const int rr = i < D.N ? D.arep[i] : -1;
    if (rr >= 0) {
        const Rep& R = D.rep[rr];
        const double safe_sq = R.box.safe_sq;
        const double3 ri = d3(D.r[i]);
        const double3 si = d3(D.s[i]);
        const double si_sq = sq3(si);
        const double fpi = fp[i];
        double3 f = make_double3(0.0, 0.0, 0.0), h = make_double3(0.0, 0.0, 0.0);
        double e = 0.0, S = 0.0;
        const int nn = D.nbn[i];
        const int* nb = D.nb + (size_t)i * kMaxNb;
        for (int k = lane4; k < nn; k += 4) {
            const int j = nb[k];
            double3 rij = sub3(ri, d3(D.r[j]));
            double rsq = sq3(rij);
            if (__builtin_expect(rsq >= safe_sq, 0)) {
                rij = min_image(R.box, rij);
                rsq = sq3(rij);
            }
            const double r = sqrt(rsq);
            int n;
            double ratio;
            interp_index(r, M.in_over_rmax, n, ratio);
            const double* row = M.r + (size_t)n * kMRStride;
            double dudr = 0.0;
            if (r < P.rcut_pot) {
                dudr = (fpi + fp[j]) * lerp_pair(row, MR_DF, ratio) + lerp_pair(row, MR_DV, ratio);
                e += 0.5 * lerp_pair(row, MR_V, ratio);
            }
            if (r < P.rcut_mag) {
                const double4 sj4 = D.s[j];
                const double3 sj = d3(sj4);
                const double X = dot3(si, sj) - sqrt(si_sq * sq3(sj));
                const double J = lerp_pair(row, MR_J, ratio);
                dudr += -lerp_pair(row, MR_DJ, ratio) * X;
                e += -0.5 * J * X;
                h = add3(h, mul3(J, sj));
                S += J * sj4.w;
            }
            f = add3(f, mul3(-dudr / r, rij));
        }
        e = quad_sum(e);
        S = quad_sum(S);
        f = make_double3(quad_sum(f.x), quad_sum(f.y), quad_sum(f.z));
        h = make_double3(quad_sum(h.x), quad_sum(h.y), quad_sum(h.z));
        int n;
        double ratio;
        interp_index(rho[i], M.in_over_rhomax, n, ratio);
        const double s2 = si_sq, s4 = s2 * s2;
        e += lerp_tab(M.h, kMHStride, MH_F, n, ratio);
        e += M.L[0] * s2 + M.L[1] * s4 + M.L[2] * s4 * s2 + M.L[3] * s4 * s4;
        const double kl = -(2.0 * M.L[0] + 4.0 * M.L[1] * s2 + 6.0 * M.L[2] * s4 + 8.0 * M.L[3] * s4 * s2);
        const double s0 = sqrt(s2);
        const double hc = s0 > 0.0 ? -S / s0 : 0.0;
        h = add3(h, mul3(kl + hc, si));
        const size_t c = (size_t)coff[rr] + (i - R.atom0);
        if (lane4 < 3) {
            F[3 * c + lane4] = lane4 == 0 ? f.x : lane4 == 1 ? f.y : f.z;
            H[3 * c + lane4] = lane4 == 0 ? h.x : lane4 == 1 ? h.y : h.z;
        }
        if (lane4 == 0) acc = e;
    }
    __shared__ double sh[4 * kFwdAtoms / 64];
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double v = 0.0;
        for (int w = 0; w < 4 * kFwdAtoms / 64; ++w) v += sh[w];
        partials[lb] = v;
    }
}


// The basis functions of the 16 pair parameters, one a lane: with d = R - r for
// r < R, a density or pair spline is d^3, dJ/dA is d^3 / rc^3 and dJ/drc is
// 3 A d^2 r / rc^4, all of them d^2 (alpha d + beta r).
struct Basis {
    double R, alpha, beta;
    int bridge;  // place among the knots of the quintic bridge, or -1
};

__device__ __forceinline__ Basis pair_basis(const ModelTab& M, int l) {
    Basis B;
    const double irc = 1.0 / M.Jrc;
    B.R = l < 6 ? kDFR[l] : l < 14 ? kDVR[l - 6] : M.Jrc;
    B.alpha = l < 14 ? 1.0 : l == 14 ? irc * irc * irc : 0.0;
    B.beta = l == 15 ? 3.0 * M.JA * (irc * irc) * (irc * irc) : 0.0;
    B.bridge = l >= 6 && l < 14 ? l - 6 : -1;
    return B;
}

// value and derivative at r near the knot, where the stencil sees it,
// interpolated in the entries of the table
__device__ __forceinline__ double2 basis_knot(const Basis& B, double step, double in_over_rmax, double r) {
    auto at = [&](double x) {
        const double d = fmax(B.R - x, 0.0);
        return d * d * fma(B.alpha, d, B.beta * x);
    };
    int n;
    double ratio;
    interp_index(r, in_over_rmax, n, ratio);
    double2 out = make_double2(0.0, 0.0);
#pragma unroll 1
    for (int e = n - 1; e <= n; ++e) {
        const double x = step * (double)(e + 1), dx = 1e-3 * x;
        double q = __builtin_amdgcn_rcp(x);
        q = fma(fma(-x, q, 1.0), q, q);
        q = fma(fma(-x, q, 1.0), q, q);
        const double s = 45.0 * (at(x + dx) - at(x - dx)) - 9.0 * (at(fma(2.0, dx, x)) - at(fma(-2.0, dx, x))) +
                         (at(fma(3.0, dx, x)) - at(fma(-3.0, dx, x)));
        const double w = e == n ? 1.0 - ratio : ratio;
        out.x = fma(w, at(x), out.x);
        out.y = fma(w, s * (q * (1000.0 / 60.0)), out.y);
    }
    return out;
}

// value and derivative of a pair spline that reaches the quintic bridge below 2,
// where the ZBL core ends at 1.8, interpolated in its entries
__device__ __forceinline__ double2 basis_bridge(const double* bridge, int row0, int k, double R, double step,
                                             double in_over_rmax, double r) {
    int n;
    double ratio;
    interp_index(r, in_over_rmax, n, ratio);
    double2 out = make_double2(0.0, 0.0);
    // one point after another: the points side by side would cost the whole
    // kernel registers for this rare pair
#pragma unroll 1
    for (int e = n - 1; e <= n; ++e) {
        const double x = step * (double)(e + 1);
        const double w = e == n ? 1.0 - ratio : ratio;
        auto at = [&](int s) {
            const double xs = stencil_x(x, s), d = fmax(R - xs, 0.0);
            return xs <= 1.8   ? 0.0
                   : xs <= 2.0 ? bridge[(size_t)(e - row0) * kModelBridgeRow + 9 * s + 1 + k]
                               : d * d * d;
        };
        double sum = 0.0;
#pragma unroll 1
        for (int s = 1; s < 7; s += 2) sum += (s == 1 ? 45e0 : s == 3 ? -9e0 : 1e0) * (at(s) - at(s + 1));
        out.x += w * at(0);
        out.y += w * (sum / (60e0 * (x / 1000e0)));
    }
    return out;
}

// Value and derivative at r as a table of step h interpolates them. Away from
// the knots the 6-point derivative of these cubics is their derivative, and the
// table gives g + q g'' with q = (r - x0)(x1 - r) / 2 between the entries x0 and
// x1. Near a knot or in the bridge (rest turns true, 0 returned) that is off by
// 1e-11, and the entries themselves are evaluated: basis_rest.
__device__ __forceinline__ double2 basis_smooth(const Basis& B, double r, double q, bool& rest) {
    double2 out = make_double2(0.0, 0.0);
    rest = false;
    if (r * 0.9969 < B.R) {  // else every point of the stencil is past the knot
        rest = r * 1.0031 >= B.R || (B.bridge >= 0 && r * 0.9969 <= 2.0);
        if (!rest) {
            const double d = B.R - r, g = 3.0 * B.alpha;
            out.x = fma(q, fma(2.0 * g, d, B.beta * fma(-4.0, d, 2.0 * r)), d * d * fma(B.alpha, d, B.beta * r));
            out.y = fma(q, fma(6.0, B.beta, -2.0 * g), d * fma(-g, d, B.beta * fma(-2.0, r, d)));
        }
    }
    return out;
}

__device__ __forceinline__ double2 basis_rest(const ModelTab& M, const Basis& B, double r) {
    if (B.bridge >= 0 && r * 0.9969 <= 2.0)
        return basis_bridge(M.bridge, M.row0, B.bridge, B.R, M.step, M.in_over_rmax, r);
    return basis_knot(B, M.step, M.in_over_rmax, r);
}

// adjoint, second pass: the kNParam components of grad_theta, in partial sums
// of a block's atoms [lb * per_block, (lb + 1) * per_block).
//
// Sixteen lanes an atom. First they take a pair each: geometry, lookup and the
// weights of the three kinds of parameters (density and pair spline, exchange)
// go to LDS. Then lane l goes over the pairs for its own pair parameter, whose
// basis function it evaluates: a table of them has 512 bytes a lookup, 3 GB a
// call at 262,144 atoms and as much as the memory gives (712 us, and 70 us and
// 256 MB to build the table at every parameter change), and the arithmetic takes
// 252 us; of 4,096 atoms 16 (119). The pairs near a lane's knot, one in 120, wait
// for the end of the round: some lane of a wave has one in two of five pairs, but
// a lane has one or two of its 16, and their two stencils in the pairs' order
// would cost 355 us. 127 registers for four waves a SIMD, with the points in the
// bridge one after another (side by side 12 spilled, 275 us).
constexpr int kAdjWaves = 4;

__global__ __launch_bounds__(64 * kAdjWaves, 4) void k_model_adjoint(ModelTab M, Phys P, Dev D, int per_block,
                                                                  const double* rho, const double* fp,
                                                                  const double* Q, const int* coff, const double* gE,
                                                                  const double* gF, const double* gH,
                                                                  double* partials) {
    __shared__ double sR[kAdjWaves][64];     // r
    __shared__ double sW[kAdjWaves][6][64];  // weights of the derivative, then of the value
    __shared__ double sQ[kAdjWaves][64];     // q of the interpolation
    __shared__ double sP[kAdjWaves][2][16];
    const int nblocks = (D.N + per_block - 1) / per_block;
    const int lb = xcd_block(nblocks);
    if (lb < 0) return;  // whole padding block
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l = lane & 15;
    const Basis B = pair_basis(M, l);
    const int kind = l < 6 ? 0 : l < 14 ? 1 : 2;
    double acc = 0.0, one = 0.0;  // this lane's pair parameter; lanes 0 to 5: aa, bb and Landau A to D
    const int end = min(lb * per_block + per_block, D.N);
    for (int i0 = lb * per_block + 4 * wave; i0 < end; i0 += 4 * kAdjWaves) {
        const int i = i0 + (lane >> 4);
        const int rr = i < end ? D.arep[i] : -1;
        const Rep& R = D.rep[rr < 0 ? 0 : rr];
        const double safe_sq = R.box.safe_sq;
        const int nn = rr < 0 ? 0 : D.nbn[i];
        const int* nb = D.nb + (size_t)i * kMaxNb;
        double3 ri = make_double3(0.0, 0.0, 0.0), si = ri, gf = ri, gh = ri;
        double fpi = 0.0, ge = 0.0;
        if (rr >= 0) {
            ri = d3(D.r[i]);
            si = d3(D.s[i]);
            fpi = fp[i];
            ge = gE[rr];
            const size_t ci = (size_t)coff[rr] + (i - R.atom0);
            gf = make_double3(gF[3 * ci], gF[3 * ci + 1], gF[3 * ci + 2]);
            gh = make_double3(gH[3 * ci], gH[3 * ci + 1], gH[3 * ci + 2]);
        }
        const double si_sq = sq3(si), si0 = sqrt(si_sq);
        const double gh_si = dot3(gh, si);
        double val = 0.0;  // the value's part: drho/da_k, or the sum itself
        for (int k0 = 0; __ballot(k0 < nn) != 0; k0 += 16) {
            double rp = M.rmax, qp = 0.0, w[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
            if (k0 + l < nn) {
                const int j = nb[k0 + l];
                double3 rij = sub3(ri, d3(D.r[j]));
                double rsq = sq3(rij);
                if (__builtin_expect(rsq >= safe_sq, 0)) {
                    rij = min_image(R.box, rij);
                    rsq = sq3(rij);
                }
                const double r = sqrt(rsq);
                const double cij = -dot3(gf, rij) / r;
                if (r < P.rcut_pot || r < P.rcut_mag) {
                    int n;
                    double ratio;
                    interp_index(r, M.in_over_rmax, n, ratio);
                    rp = r;
                    qp = 0.5 * M.step * M.step * ratio * (1.0 - ratio);
                }
                if (r < P.rcut_pot) {
                    w[0] = cij * (fpi + fp[j]);
                    w[1] = cij;
                    w[3] = 1.0;
                    w[4] = ge * 0.5;
                }
                if (r < P.rcut_mag) {
                    const double4 sj4 = D.s[j];
                    const double3 sj = d3(sj4);
                    const double X = dot3(si, sj) - sqrt(si_sq * sq3(sj));
                    w[2] = -cij * X;
                    w[5] = ge * (-0.5 * X) + (dot3(gh, sj) - (si0 > 0.0 ? sj4.w / si0 * gh_si : 0.0));
                }
            }
            sR[wave][lane] = rp;
            sQ[wave][lane] = qp;
#pragma unroll
            for (int q = 0; q < 6; ++q) sW[wave][q][lane] = w[q];
            wave_fence();
            const int left = min(nn - k0, 16);
            unsigned later = 0;  // bit p: pair p near this lane's knot
            for (int p = 0; p < left; ++p) {
                const int at = (lane & 48) + p;
                bool rest;
                const double2 b = basis_smooth(B, sR[wave][at], sQ[wave][at], rest);
                acc += sW[wave][kind][at] * b.y;
                val += sW[wave][3 + kind][at] * b.x;
                later |= (unsigned)rest << p;
            }
            for (; later; later &= later - 1) {
                const int at = (lane & 48) + __builtin_ctz(later);
                const double2 b = basis_rest(M, B, sR[wave][at]);
                acc += sW[wave][kind][at] * b.y;
                val += sW[wave][3 + kind][at] * b.x;
            }
            wave_fence();
        }
        if (rr >= 0) {
            // one-body terms: F(rho_i) (energy), F'(rho_i) (through Q_i), Landau
            int n;
            double ratio;
            interp_index(rho[i], M.in_over_rhomax, n, ratio);
            const double* h0 = M.h + (size_t)(n - 1) * kMHStride;
            const double* h1 = h0 + kMHStride;
            const double slope_f = (h1[MH_F] - h0[MH_F]) * M.in_over_rhomax;
            const double slope_fp = (h1[MH_DF] - h0[MH_DF]) * M.in_over_rhomax;
            const double qi = Q[i];
            acc += kind == 0 ? (ge * slope_f + qi * slope_fp) * val : val;
            const double s2 = si_sq, s4 = s2 * s2, s6 = s4 * s2;
            if (l < 2) {
                const int kv = l == 0 ? MH_AA : MH_BB, kd = l == 0 ? MH_DAA : MH_DBB;
                one += ge * lerp_tab(M.h, kMHStride, kv, n, ratio) + qi * lerp_tab(M.h, kMHStride, kd, n, ratio);
            }
            if (l == 2) one += ge * s2 - 2.0 * gh_si;
            if (l == 3) one += ge * s4 - 4.0 * s2 * gh_si;
            if (l == 4) one += ge * s6 - 6.0 * s4 * gh_si;
            if (l == 5) one += ge * s4 * s4 - 8.0 * s6 * gh_si;
        }
    }
    acc += __shfl_xor(acc, 16, 64);
    acc += __shfl_xor(acc, 32, 64);
    one += __shfl_xor(one, 16, 64);
    one += __shfl_xor(one, 32, 64);
    if (lane < 16) {
        sP[wave][0][l] = acc;
        sP[wave][1][l] = one;
    }
    __syncthreads();
    const int t = threadIdx.x;
    if (t < kNParam) {
        // theta's order: 14 splines, aa and bb, the two of J, Landau
        const int which = t < 14 || t == P_JA || t == P_JRC ? 0 : 1;
        const int at = t < 14 ? t : t < P_JA ? t - P_AA : t < P_LA ? t - P_JA + 14 : t - P_LA + 2;
        double v = 0.0;
        for (int w = 0; w < kAdjWaves; ++w) v += sP[w][which][at];
        partials[(size_t)t * nblocks + lb] = v;
    }
}

}  // namespace sld
