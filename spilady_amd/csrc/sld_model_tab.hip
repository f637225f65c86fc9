// Device construction of the parametric model's tables (sld_model.h).
//
// The host loop that used to fill them (10^6 rows of 46 columns, a 6-point
// stencil behind every second one, 16 threads) took about 250 ms of every
// parameter change, against 2 ms for the whole loss gradient of 262,144
// atoms. The rows are independent, so one thread makes one row and the rows
// leave through LDS as contiguous lines: 448 MB in 154 us (2.9 TB/s; the
// derivative table 70 us, the r values 65 us, the rho table 19 us). A training
// step of 32 x 8,192 atoms went from 278 to 2.58 ms, of 4 x 1,024 from 277 to
// 0.99 ms.
//
// Every value is evaluated in the order of the forms' definition with no
// contraction, so a table entry is the host's to the rounding of exp and log
// (the ZBL core and F(rho)) and of a cube. The quintic bridge (1.8 < r <= 2)
// cancels terms of 1e5 down to 1, so there the powers' last bit would show:
// its theta-independent polynomials come from the host (ModelBridge), one
// value for each of a row's seven stencil points.
#include <hip/hip_runtime.h>

#include "sld_kernels.h"
#include "sld_model.h"

#pragma clang fp contract(off)

namespace sld {

__constant__ static const double kDFR[6] = {3.0, 2.8666666666666666, 2.7333333333333333, 2.6, 2.4, 2.3};
__constant__ static const double kDVR[8] = {4.1, 3.8, 3.5, 3.2, 2.9, 2.6, 2.4, 2.3};

// stencil slot s of a row at x: x, x + dx, x - dx, x + 2dx, x - 2dx, x + 3dx, x - 3dx
__device__ __forceinline__ double stencil_x(double x, int s) {
    const double dx = x / 1000e0;
    const double d = (double)((s + 1) >> 1) * dx;
    return s == 0 ? x : (s & 1 ? x + d : x - d);
}

__device__ __forceinline__ double stencil_deriv(const double (&v)[7], double x) {
    const double dx = x / 1000e0;
    return (45e0 * (v[1] - v[2]) - 9e0 * (v[3] - v[4]) + (v[5] - v[6])) / (60e0 * dx);
}

__device__ __forceinline__ double cube_knot(double R, double r) {
    const double d = R - r;
    return r < R ? d * d * d : 0e0;
}

__device__ __forceinline__ double cube_j(double r, double rc) {
    const double q = 1.0 - r / rc;
    return r < rc ? q * q * q : 0e0;
}

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
__global__ __launch_bounds__(256) void k_model_tab_r(ModelCoef m, const double* bridge, double* out) {
    __shared__ double sh[6][256];
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
        sh[MR_F][t] = f[0];
        sh[MR_DF][t] = stencil_deriv(f, r);
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
        o[e] = c < 12 ? sh[c >> 1][row + (c & 1)] : 0e0;
    }
}

// The derivative table: 64 rows of 32 columns a block of 64 threads.
__global__ __launch_bounds__(64) void k_model_tab_rd(ModelCoef m, const double* bridge, double* out) {
    constexpr int kPad = kMRDStride + 1;  // rows start on different LDS banks
    __shared__ double sh[64 * kPad];
    const int t = threadIdx.x;
    const int n0 = blockIdx.x * 64, n = n0 + t;
    if (n < kNInput) {
        const double r = m.rmax / (double)kNInput * (double)(n + 1);
        const double* q = bridge + (size_t)(n - m.row0) * kModelBridgeRow;
        double* D = sh + t * kPad;
        for (int k = 0; k < 6; ++k) {
            double v[7];
            for (int s = 0; s < 7; ++s) v[s] = cube_knot(kDFR[k], stencil_x(r, s));
            D[2 * k] = v[0];
            D[2 * k + 1] = stencil_deriv(v, r);
        }
        for (int k = 0; k < 8; ++k) {
            double v[7];
            for (int s = 0; s < 7; ++s) {
                const double x = stencil_x(r, s);
                v[s] = x <= 1.8 ? 0e0 : x <= 2.0 ? q[9 * s + 1 + k] : cube_knot(kDVR[k], x);
            }
            D[12 + 2 * k] = v[0];
            D[13 + 2 * k] = stencil_deriv(v, r);
        }
        double a[7], b[7];
        for (int s = 0; s < 7; ++s) {
            const double x = stencil_x(r, s);
            a[s] = cube_j(x, m.Jrc);
            const double u = 1.0 - x / m.Jrc;
            b[s] = x < m.Jrc ? m.JA * 3.0 * (u * u) * x / (m.Jrc * m.Jrc) : 0e0;
        }
        D[28] = a[0];
        D[29] = stencil_deriv(a, r);
        D[30] = b[0];
        D[31] = stencil_deriv(b, r);
    }
    __syncthreads();
    const int rows = min(64, kNInput - n0);
    double* o = out + (size_t)n0 * kMRDStride;
    for (int e = t; e < rows * kMRDStride; e += 64) o[e] = sh[(e / kMRDStride) * kPad + e % kMRDStride];
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
