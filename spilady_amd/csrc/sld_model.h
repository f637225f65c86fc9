// The differentiable potential model: energies, forces and effective fields
// of frozen configurations as functions of the DD05 and Fe exchange/Landau
// parameters, with their parameter adjoint.
#pragma once

#include <memory>
#include <vector>

namespace sld {

// Parameter vector theta:
//   [0..5]   a_k   density spline coefficients      f(r) = sum a_k (R_k - r)^3, r < R_k   (DD05.cpp:20-43)
//   [6..13]  V_k   pair spline coefficients         V(r) = sum V_k (R_k - r)^3, r > 2      (DD05.cpp:64-164)
//   [14..15] aa bb embedding F(rho)                                                        (DD05.cpp:6-18)
//   [16..17] A rc  exchange J(r) = A (1 - r/rc)^3, r < rc                                 (JijFe.cpp:5-14)
//   [18..21] Landau A B C D (constants for Fe)                                             (JijFe.cpp:18-43)
constexpr int kNParam = 22;
enum ParamIndex { P_A0 = 0, P_V0 = 6, P_AA = 14, P_BB = 15, P_JA = 16, P_JRC = 17, P_LA = 18 };

// Columns of the model tables (10^6 entries each, the reference's sampling
// and 6-point derivative stencil):
//   r value table   [N][16]: the interpolation pair (t[n-1], t[n]) of each of f' V V' J J', then padding:
//                            a lookup touches one 128-byte line
//   f, f'           [N]:     for the passes that read nothing else
//   rho table       [N][8]:  F F' dF/daa dF'/daa dF/dbb dF'/dbb - -
constexpr int kMRStride = 16;
constexpr int kMHStride = 8;
enum MRCol { MR_DF = 0, MR_V, MR_DV, MR_J, MR_DJ };
enum MHCol { MH_F = 0, MH_DF, MH_AA, MH_DAA, MH_BB, MH_DBB };

// The quintic bridge of the pair term at the stencil points of the rows that
// reach it, theta-independent: row n, point s (x, x + dx, x - dx, x + 2dx, ...)
// holds the bridge of the ZBL end alone, then that of each knot alone. Rows
// [row0, row0 + nrow) of the r tables; points outside the bridge hold 0.
constexpr int kModelBridgeRow = 7 * 9;
struct ModelBridge {
    int row0 = 0, nrow = 0;
    std::vector<double> q;  // [nrow][7][9]
};
// Built on the host (up to 16 threads, about 50 ms on 8 and 26 MB); the last
// kModelBridges cutoffs stay with the process, older ones with their contexts.
constexpr int kModelBridges = 4;
std::shared_ptr<const ModelBridge> model_bridge(double rcut_max);

// What the device needs to fill the tables at theta.
struct ModelCoef {
    double a[6], V[8], aa, bb, JA, Jrc;
    double as, ln2;        // ZBL screening length, log 2
    double rmax, rhomax;
    int row0;              // first row of the bridge values
};

// The reference's parameter values (DD05.cpp, JijFe.cpp).
void model_default_params(double* theta);
// The coefficients of the tables at theta, sampled on [0, rcut_max] and [0, rhomax].
ModelCoef model_coef(const double* theta, double rcut_max, const ModelBridge& bridge);

}  // namespace sld
