// The parametric model's knots and sampling, for its table and adjoint kernels.
#pragma once

namespace sld {

__constant__ static const double kDFR[6] = {3.0, 2.8666666666666666, 2.7333333333333333, 2.6, 2.4, 2.3};
__constant__ static const double kDVR[8] = {4.1, 3.8, 3.5, 3.2, 2.9, 2.6, 2.4, 2.3};

// f and its stencil derivative are 0 at the entries from 3 / 0.997 on
constexpr double kFEnd = 3.0091;

// stencil slot s of a row at x: x, x + dx, x - dx, x + 2dx, x - 2dx, x + 3dx,
// x - 3dx; to the bit the host's, which decides by it what rows the bridge has
__device__ __forceinline__ double stencil_x(double x, int s) {
#pragma clang fp contract(off)
    const double dx = x / 1000e0;
    const double d = (double)((s + 1) >> 1) * dx;
    return s == 0 ? x : (s & 1 ? x + d : x - d);
}

__device__ __forceinline__ double stencil_deriv(const double (&v)[7], double x) {
#pragma clang fp contract(off)
    const double dx = x / 1000e0;
    return (45e0 * (v[1] - v[2]) - 9e0 * (v[3] - v[4]) + (v[5] - v[6])) / (60e0 * dx);
}

}  // namespace sld
