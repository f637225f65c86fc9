// Device construction of the parametric model's tables (sld_model.h).
//
// The host loop that used to fill them (10^6 rows of 46 columns, a 6-point
// stencil behind every second one, 16 threads) took about 250 ms of every
// parameter change, against 2 ms for the whole loss gradient of 262,144
// atoms. The rows are independent, so one thread makes one row and the rows
// leave through LDS as contiguous lines: 192 MB in 85
// us (the r values 66, the rho table 19).
//
// Every value is evaluated in the order of the forms' definition with no
// contraction, so a table entry is the host's to the rounding of exp and log
// (the ZBL core and F(rho)). The quintic bridge (1.8 < r <= 2) cancels terms of
// 1e5 down to 1, so there the powers' last bit would show: its theta-independent
// polynomials come from the host (ModelBridge), one value for each of a row's
// seven stencil points.
#include <hip/hip_runtime.h>

#include "sld_kernels.h"
#include "sld_model.h"
#include "sld_model_device.h"

#pragma clang fp contract(off)

namespace sld {

// d^3 rounded once, as pow(d, 3) is: the splines' terms cancel to a hundredth of
// the largest, and the stencil divides what is left by 1e-3
__device__ __forceinline__ double cube(double d) {
    const double p = d * d;
    return fma(p, d, fma(d, d, -p) * d);
}

__device__ __forceinline__ double cube_knot(double R, double r) { return r < R ? cube(R - r) : 0e0; }

__device__ __forceinline__ double cube_j(double r, double rc) { return r < rc ? cube(1.0 - r / rc) : 0e0; }

// DD05.cpp:45-62
__device__ __forceinline__ double zbl(double r, double as) {
    const double x = r / as;
    const double v = 0.1818e0 * exp(-3.2 * x) + 0.5099e0 * exp(-0.9423 * x) + 0.2802e0 * exp(-0.4029 * x) +
                     0.02817e0 * exp(-0.2016 * x);
    return 26e0 * 26e0 * 14.3992 * v / r;
}

__device__ __forceinline__ double big_f(const ModelCoef& m, double rho) {
    const double s = sqrt(rho);
    if (rho >= 1e0) return -m.aa * s;
    return -m.aa * s - m.bb / m.ln2 * (1e0 - s) * log(2e0 - rho);
}

// Row n of the r value table holds the pairs (t[n-1], t[n]) of its columns;
// a block of 256 threads evaluates entries n0 - 1 .. n0 + 254 and writes rows
// n0 .. n0 + 254.
__global__ __launch_bounds__(256) void k_model_tab_r(ModelCoef m, const double* bridge, double* out, double* out_f,
                                                     double* out_df) {
    __shared__ double sh[5][256];
    const int t = threadIdx.x;
    const int n0 = 1 + blockIdx.x * 255;
    const int n = n0 - 1 + t;
    if (n < kNInput) {
        const double r = m.rmax / (double)kNInput * (double)(n + 1);
        double f[7], v[7], J[7];
        // a row reads its bridge values only at points of the bridge, which
        // lie inside [row0, row0 + nrow) by construction
        const double* q = bridge + (size_t)(n - m.row0) * kModelBridgeRow;
        for (int s = 0; s < 7; ++s) {
            const double x = stencil_x(r, s);
            double a = 0e0;
            for (int i = 0; i < 6; ++i) a += m.a[i] * cube_knot(kDFR[i], x);
            f[s] = a;
            double b;
            if (x <= 1.8) {
                b = zbl(x, m.as);
            } else if (x <= 2.0) {
                b = q[9 * s];
                for (int k = 0; k < 8; ++k) b += m.V[k] * q[9 * s + 1 + k];
            } else {
                b = 0e0;
                for (int k = 0; k < 8; ++k) b += m.V[k] * cube_knot(kDVR[k], x);
            }
            v[s] = b;
            J[s] = m.JA * cube_j(x, m.Jrc);
        }
        const double df = stencil_deriv(f, r);
        if (t < 255 || n == kNInput - 1) {
            out_f[n] = f[0];
            out_df[n] = df;
        }
        sh[MR_DF][t] = df;
        sh[MR_V][t] = v[0];
        sh[MR_DV][t] = stencil_deriv(v, r);
        sh[MR_J][t] = J[0];
        sh[MR_DJ][t] = stencil_deriv(J, r);
    }
    __syncthreads();
    const int rows = min(255, kNInput - n0);
    double* o = out + (size_t)n0 * kMRStride;
    for (int e = t; e < rows * kMRStride; e += 256) {
        const int row = e / kMRStride, c = e % kMRStride;
        o[e] = c < 10 ? sh[c >> 1][row + (c & 1)] : 0e0;
    }
}

// The rho table: 256 rows of 8 columns a block.
__global__ __launch_bounds__(256) void k_model_tab_h(ModelCoef m, double* out) {
    constexpr int kPad = kMHStride + 1;
    __shared__ double sh[256 * kPad];
    const int t = threadIdx.x;
    const int n0 = blockIdx.x * 256, n = n0 + t;
    double* H = sh + t * kPad;
    if (n < kNInput) {
        const double rho = m.rhomax / (double)kNInput * (double)(n + 1);
        double f[7], a[7], b[7];
        for (int s = 0; s < 7; ++s) {
            const double x = stencil_x(rho, s);
            const double sq = sqrt(x);
            f[s] = big_f(m, x);
            a[s] = -sq;
            b[s] = x >= 1e0 ? 0e0 : -(1e0 - sq) * log(2e0 - x) / m.ln2;
        }
        H[MH_F] = f[0];
        H[MH_DF] = stencil_deriv(f, rho);
        H[MH_AA] = a[0];
        H[MH_DAA] = stencil_deriv(a, rho);
        H[MH_BB] = b[0];
        H[MH_DBB] = stencil_deriv(b, rho);
        H[6] = 0e0;
        H[7] = 0e0;
    }
    __syncthreads();
    const int rows = min(256, kNInput - n0);
    double* o = out + (size_t)n0 * kMHStride;
    for (int e = t; e < rows * kMHStride; e += 256) o[e] = sh[(e / kMHStride) * kPad + e % kMHStride];
}

}  // namespace sld
