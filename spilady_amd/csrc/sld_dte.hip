// Kernels of the electron subsystem's diffusion (core_dTe_CPU.cpp:47-217).
//
// Compiled with the two-address FMA off (-fmacf64-inst): the polynomials of
// the heat capacity are long chains of a*t + c with c kept in registers, and
// the two-address form overwrites its addend, so each term cost a move.
#include <hip/hip_runtime.h>

#include "sld_kernels.h"

namespace sld {

// core_dTe sub-step (core_dTe_CPU.cpp:51-55,66-140): A(h) adds the lattice's
// and spins' energy, B(h) relaxes towards them, C diffuses. What A and B take
// of a cell is constant over a core_dTe call: k_dte_ab leaves it in M.src for
// the other sub-step kernels, h dE and g = -G / (3b) with G = (Gel + Ges) h /
// k_B (16 bytes a cell instead of the 32 of the four fields they come from).

// One relaxation T -> T + increment is RK4 over T (exp(-G / C(T)) - 1), C = 3
// tanh(bT) (core_dTe_CPU.cpp:91-129). The exponent is u = (g/T) K(x^2) with
// x = bT, K = x coth x, so T (e^u - 1) = g K (1 + u/2 + ...): one reciprocal
// and two polynomials, where the defining form spends a division and an exp
// and cancels (u is 0.001 to 0.1 at 1 fs, larger the colder the electrons).
// ok turns false outside the fitted temperatures or for |u| > 1/4 (NaN
// included).
constexpr Poly<13> kRelaxK = scaled(kXCothX, 1.0, kCeB* kCeB);     // K(x^2) in T^2
constexpr double kPolyT2Max = kPolyXMax * kPolyXMax / (kCeB * kCeB);
// (e^u - 1) / u for |u| <= 1/4: the next term is 2^-24 / 13! = 1e-17
constexpr double kExpm1[12] = {1.0,           1.0 / 2.0,      1.0 / 6.0,       1.0 / 24.0,
                               1.0 / 120.0,   1.0 / 720.0,    1.0 / 5040.0,    1.0 / 40320.0,
                               1.0 / 362880.0, 1.0 / 3628800.0, 1.0 / 39916800.0, 1.0 / 479001600.0};

__device__ __forceinline__ double relax_fast(double g, double T, bool& ok) {
    const double t = T * T;
    double r = __builtin_amdgcn_rcp(T);  // 1/T to about an ulp in two Newton steps
    r = fma(fma(-T, r, 1.0), r, r);
    r = fma(fma(-T, r, 1.0), r, r);
    const double w = g * horner2(kRelaxK.c, t);
    const double u = w * r;
    ok = ok && T >= 1e-30 && t <= kPolyT2Max && fabs(u) <= 0.25;
    return w * horner2(kExpm1, u);
}

__device__ __forceinline__ double relax_any(double g, double T) {
    return T * (exp(g * (3.0 * kCeB) / (3.0 * tanh_bt(kCeB * T))) - 1.0);
}

// The stages are carried as k h (the reference divides each k by h and
// multiplies it back): the same increments up to rounding. A loop, so that the
// code and its 25 coefficients stay small.
template <class F>
__device__ __forceinline__ double rk4(double T0, F relax) {
    double q = 0.0, sum = 0.0;
#pragma unroll 1
    for (int k = 0; k < 4; ++k) {
        q = relax(fma(k == 0 ? 0.0 : k == 3 ? 1.0 : 0.5, q, T0));
        sum = fma(k == 0 || k == 3 ? 1.0 : 2.0, q, sum);
    }
    return fma(sum, 1.0 / 6.0, T0);
}

// n times T(E), B(h), E(T) and, after all but the last of n == 2, A(h) twice:
// n == 2 takes the energy a sub-step's C left to the one the next C starts
// from. Returns the energy, T the temperature of the last relaxation.
// Every lane takes the polynomial route, without branches; a wave with a lane
// outside its range repeats that lane's cell with the library's functions.
__device__ __forceinline__ double dte_relax_steps(double e0, double dE, double g, int n, double& T) {
    bool ok = true;
    double e = e0;
#pragma unroll 1
    for (int k = 0; k < n; ++k) {
        if (k > 0) e = (e + dE) + dE;
        ok = ok && e <= kPolyEMax && e >= 1e-200;
        T = ee_to_te_fit(e);
        T = rk4(T, [&](double x) { return relax_fast(g, x, ok); });
        const double t = T * T;
        ok = ok && t <= kPolyT2Max;
        e = te_to_ee_fit(t);
    }
    if (__builtin_expect(!ok, 0)) {
        e = e0;
#pragma unroll 1
        for (int k = 0; k < n; ++k) {
            if (k > 0) e = (e + dE) + dE;
            T = rk4(ee_to_te(e), [&](double x) { return relax_any(g, x); });
            e = te_to_ee(T);
        }
    }
    return e;
}

// What A and B take of cell c: h dE and g (see above).
__device__ __forceinline__ double2 dte_source(const Mesh& M, int c, double h) {
    double dE = 0.0, G = 0.0;
    if (M.lattlang) {
        dE += M.Gel[c] * M.Tl[c];
        G += M.Gel[c];
    }
    if (M.spinlang) {
        dE += M.Ges[c] * M.TsL[c];
        G += M.Ges[c];
    }
    return make_double2(dE * h, G * (h / kBoltz) * (-1.0 / (3.0 * kCeB)));
}

// the first sub-step's A(h), B(h), then Ee = E(Te) as C starts
__global__ __launch_bounds__(256) void k_dte_ab(double h, Mesh M, double* partials) {
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    double acc[1] = {0.0};
    if (c < M.C) {
        const double2 src = dte_source(M, c, h);
        M.src[c] = src;
        double T;
        const double ee = dte_relax_steps(te_to_ee(M.Te[c]) + src.x, src.x, src.y, 1, T);
        M.Te[c] = T;
        M.Ee[c] = ee;
        acc[0] = ee;
    }
    block_partials<1>(acc, partials);
}

// The C diffusion sweeps (core_dTe_CPU.cpp:155-197), one workgroup per tile of
// the mesh (sld_dte_plan.h): the temperatures of the tile's cells, of their
// closure and of what those read come into LDS, the levels of the schedule
// run there with a workgroup barrier between them, and the tile writes its
// own cells to the other copy of the mesh, which no tile of the launch reads.
// The reference recomputes E(Te) of a cell first; the stored Ee of the cell's
// last update is that value up to one rounding.
//
// A sweep is a chain of up to 20 dependent cell updates whatever the mesh
// size, and the tile with the longest chain ends the launch: at 69^3 and 23^3
// cells most tiles have 8 levels, the last few 18, in either sweep. A launch per
// level cost 3.5 us each; here a level costs one LDS round trip, the update's FP64
// chain and a barrier, 600 cycles or 0.25 us, of which neither the number of waves
// nor the lists' loads are a part any more (33 x 25 x 10 cells, 28 levels of both
// sweeps: 12.6 us a launch, 14.2 with the lists requested one level ahead, whose
// hand-over waited for them, and a branch per lane for temperatures outside the
// fit; 7^3 cells, 40 levels, in a launch of their own 14.2 and 15.7).
// The energy partials are one per tile: its cells in slot order, 64 at a
// time, so the sum does not depend on the block size.
constexpr int kAhead = 4;  // levels

// a thread's first update of level l; bound: in lane l, the first update of level l
__device__ __forceinline__ uint4 dte_request(const DteTile& T, const uint4* upd, int bound, int l) {
    return upd[min(__builtin_amdgcn_readlane(bound, min(l, T.nlev)) + (int)threadIdx.x, T.nent - 1)];
}

// one update (core_dTe_CPU.cpp:161-190)
__device__ __forceinline__ void dte_update(uint4 d, double* sT, double* sE, double px, double py, double pz) {
    // keeps the split of the last word here: ahead of the loop's end it
    // would wait for the requests
    asm volatile("" : "+v"(d.w));
    char* q = reinterpret_cast<char*>(sT);
    auto at = [&](uint32_t o) -> double& { return *reinterpret_cast<double*>(q + o); };
    const uint32_t self = d.x & 0xffffu;
    const double txp = at(d.x >> 16), txm = at(d.y & 0xffffu);
    const double typ = at(d.y >> 16), tym = at(d.z & 0xffffu);
    const double tzp = at(d.z >> 16), tzm = at(d.w & 0xffffu);
    const double tc = at(self);
    double& E = *reinterpret_cast<double*>(reinterpret_cast<char*>(sE) + self);
    double ee = E;
    ee = fma(fma(-2.0, tc, txp + txm), px, ee);
    ee = fma(fma(-2.0, tc, typ + tym), py, ee);
    ee = fma(fma(-2.0, tc, tzp + tzm), pz, ee);
    E = ee;
    double T = ee_to_te_fit(ee);
    if (__builtin_expect(__ballot(!te_fits(ee)) != 0, 0)) T = ee_to_te(ee);  // without a branch per lane
    at(self) = T;
}

// The levels of a tile, a workgroup barrier after each. ring[l]: the thread's
// first update of level l < kAhead; from there on they are requested kAhead
// levels ahead (straight-line code, so that the wait before an update leaves
// the later requests in flight).
__device__ __forceinline__ void dte_levels(const DteTile& T, const uint4* upd, int bound, uint4 (&ring)[kAhead],
                                           double* sT, double* sE, double px, double py, double pz) {
    const int t = threadIdx.x, B = blockDim.x, lane = t & 63;
    const int after = __shfl_down(bound, 1, 64);
    if (__ballot(lane < T.nlev && after - bound > B) == 0) {  // a thread has at most one update a level
        // past the last level nothing is left to update
        int lo = 0, hi = __builtin_amdgcn_readlane(bound, 1);
        for (int l0 = 0; l0 < T.nlev; l0 += kAhead) {
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const uint4 d = ring[u];
                const bool on = lo + t < hi;
                lo = hi;
                hi = __builtin_amdgcn_readlane(bound, min(l0 + u + 2, T.nlev));
                ring[u] = dte_request(T, upd, bound, l0 + u + kAhead);
                if (on) dte_update(d, sT, sE, px, py, pz);
                __syncthreads();
            }
        }
    } else {
        for (int l = 0; l < T.nlev; ++l) {
            const int hi = __builtin_amdgcn_readlane(bound, l + 1);
            for (int k = __builtin_amdgcn_readlane(bound, l) + t; k < hi; k += B)
                dte_update(upd[k], sT, sE, px, py, pz);
            __syncthreads();
        }
    }
}

template <int U>
__global__ __launch_bounds__(512) void k_dte_sweep(DteTiles S, DteSweepArgs A) {
    extern __shared__ double sT[];
    __shared__ double sp[kDteMaxSlot / 64 + 1];
    const int t = threadIdx.x, B = blockDim.x, lane = t & 63;
    if ((int)blockIdx.x == ((S.ntile + 7) & ~7)) {  // the block past the tiles adds the starting energies
        if (t < 64) {
            double a = 0.0;
            for (int k0 = t; k0 < A.na; k0 += 8 * 64) {
                double v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = k0 + u * 64 < A.na ? A.pa[k0 + u * 64] : 0.0;
#pragma unroll
                for (int u = 0; u < 8; ++u) a += v[u];
            }
            a = wave_sum(a);
            if (t == 0) A.start[0] = a;
        }
        return;
    }
    const int tl = (int)(blockIdx.x & 7) * ((S.ntile + 7) >> 3) + (int)(blockIdx.x >> 3);  // see xcd_block
    if (tl >= S.ntile) return;
    const DteTile T = S.tile[tl];
    const uint4* upd = S.upd + T.upd0;
    const int32_t* slot = S.slot + T.slot0;
    const int bound = S.lev[T.lev0 + lane];  // lane l: first update of level l
    double* sE = sT + S.max_slot;
    // a thread's first U slots t, t + B, ... are in flight together, and their
    // cells stay in registers until the results go out: 8 where a thread has
    // that many (69^3 cells: 11.1 us a launch instead of 12.2), 4 where the
    // other four would be loads for nothing (40^3: 8.2 and 9.3)
    int32_t c[U];
#pragma unroll
    for (int u = 0; u < U; ++u) c[u] = slot[min(t + u * B, T.nslot - 1)];
    uint4 ring[kAhead];
#pragma unroll
    for (int l = 0; l < kAhead; ++l) ring[l] = dte_request(T, upd, bound, l);
    {
        double a[U], e[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int cell = T.origin + (c[u] >> 1);
            a[u] = A.Tin[cell];
            e[u] = t + u * B < T.nupd ? A.Ein[cell] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (t + u * B < T.nslot) sT[t + u * B] = a[u];
            if (t + u * B < T.nupd) sE[t + u * B] = e[u];
        }
    }
    for (int s = t + U * B; s < T.nslot; s += B) {
        const int cell = T.origin + (slot[s] >> 1);
        sT[s] = A.Tin[cell];
        if (s < T.nupd) sE[s] = A.Ein[cell];
    }
    __syncthreads();
    dte_levels(T, upd, bound, ring, sT, sE, A.px, A.py, A.pz);
    const int nch = (T.nupd + 63) >> 6;
    auto put = [&](int s, int32_t c) {
        const bool own = s < T.nupd && (c & 1) != 0;
        const double ee = own ? sE[s] : 0.0;
        if (own) {
            A.Eout[T.origin + (c >> 1)] = ee;
            if (A.Tout) A.Tout[T.origin + (c >> 1)] = sT[s];
        }
        if (A.ends) {
            const double v = wave_sum(ee);
            if (lane == 0) sp[s >> 6] = v;
        }
    };
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (((t + u * B) >> 6) < nch) put(t + u * B, c[u]);
    for (int s = t + U * B; (s >> 6) < nch; s += B) put(s, slot[min(s, T.nslot - 1)]);
    if (A.ends) {
        __syncthreads();
        if (t < 64) {
            double a = 0.0;
            for (int k = t; k < nch; k += 64) a += sp[k];
            a = wave_sum(a);
            if (t == 0) A.ends[tl] = a;
        }
    }
}

template __global__ void k_dte_sweep<4>(DteTiles, DteSweepArgs);
template __global__ void k_dte_sweep<8>(DteTiles, DteSweepArgs);

// the final energy of a sub-step from its n partials, by every block of 256
// threads for itself in the same fixed order
__device__ __forceinline__ double dte_end_total(const double* p, int n) {
    __shared__ double sh[4];
    const int t = threadIdx.x;
    double a = 0.0;
    for (int k = t; k < n; k += 256) a += p[k];
    a = wave_sum(a);
    if ((t & 63) == 0) sh[t >> 6] = a;
    __syncthreads();
    return (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// The sub-step's cell work between two diffusions. With 64 cells a wave and
// 1,284 blocks at 328,509 cells every wave is resident at once, and the time is
// the launch, one round trip to memory and a wave's own instruction stream:
// the two polynomials of a relaxation instead of a division and an exp, and
// wave sums without LDS, took it from 17.0 to 12.1 us there, from 6.9 to 4.6
// at 12,167 cells.
// end of one sub-step and start of the next: renormalise (core_dTe_CPU.cpp:199-216),
// B(h), A(h), then the next sub-step's A(h), B(h) and E(Te) as its C starts.
// The Te and Ee that the first A(h) leaves are overwritten by the second
// before anything reads them, so only the final values are stored.
__global__ __launch_bounds__(256) void k_dte_finish_ab(Mesh M, const double* E, const double* start,
                                                       const double* ends, int nend, double* partials) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    const int cc = c < M.C ? c : M.C - 1;
    const double2 src = M.src[cc];
    const double e0 = E[cc];
    const double f = start[0] / dte_end_total(ends, nend);
    double acc[1] = {0.0};
    if (c < M.C) {
        double T;
        const double ee = dte_relax_steps(e0 * f, src.x, src.y, 2, T);
        M.Te[c] = T;
        M.Ee[c] = ee;
        acc[0] = ee;
    }
    block_partials<1>(acc, partials);
}

// renormalise to the starting total (core_dTe_CPU.cpp:199-216), then B(h), A(h)
__global__ __launch_bounds__(256) void k_dte_finish(Mesh M, const double* E, const double* start, const double* ends,
                                                    int nend) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    const double f = start[0] / dte_end_total(ends, nend);
    if (c >= M.C) return;
    const double2 src = M.src[c];
    double T;
    const double ee = dte_relax_steps(E[c] * f, src.x, src.y, 1, T) + src.x;
    M.Ee[c] = ee;
    M.Te[c] = ee_to_te(ee);
}

// A whole core_dTe call of a small mesh, one tile, in one workgroup: the
// temperatures, energies and sources stay in LDS for all sub-steps. A sub-step
// takes its levels (0.25 us each, 40 at 7^3 and 8 at even sides), one relaxation a thread and two sums, and no
// launch: a call of 7^3 cells 680 us where two launches a sub-step took 970, of
// 8^3 297 (621), of 10^3 442 (615). From there on the relaxations, two and more a
// thread, are worth more compute units: 11^3 936 and 942, 12^3 744 and 636, so
// the line is at kDteSmall cells. (The relaxation as a function of its own, to
// spare scalar registers, made the levels slower: 885 us at 7^3.) Always 512
// threads: 128, which sweep_block = 64 once gave, made a call of 10^3 cells 1,088
// us where a launch a level had taken 1,045; 256 are as good below 300 cells only.
__global__ __launch_bounds__(kDteSmallBlock) void k_dte_small(DteTiles S, Mesh M, double h, double px, double py,
                                                              double pz, int nloop) {
    extern __shared__ double sT[];
    __shared__ double sp[kDteSmall / 64];
    const int t = threadIdx.x, B = blockDim.x, lane = t & 63;
    const DteTile T = S.tile[0];
    const uint4* upd = S.upd + T.upd0;
    const int32_t* slot = S.slot + T.slot0;
    const int bound = S.lev[T.lev0 + lane];
    double* sE = sT + kDteSmall;
    double2* src = reinterpret_cast<double2*>(sE + kDteSmall);
    uint4 first[kAhead];
#pragma unroll
    for (int l = 0; l < kAhead; ++l) first[l] = dte_request(T, upd, bound, l);
    // sum of the energies, in chunks of 64 cells
    const int nch = (M.C + 63) >> 6;
    auto total = [&]() {
        for (int q = t >> 6; q < nch; q += B >> 6) {
            const int s = q * 64 + lane;
            const double v = wave_sum(s < M.C ? sE[s] : 0.0);
            if (lane == 0) sp[q] = v;
        }
        __syncthreads();
        return wave_sum(lane < nch ? sp[lane] : 0.0);
    };
    for (int s = t; s < M.C; s += B) {
        const int c = T.origin + (slot[s] >> 1);
        const double2 a = dte_source(M, c, h);
        double Tn;
        sE[s] = dte_relax_steps(te_to_ee(M.Te[c]) + a.x, a.x, a.y, 1, Tn);
        sT[s] = Tn;
        src[s] = a;
    }
    __syncthreads();
    for (int it = 0; it < nloop; ++it) {
        const double start = total();
        uint4 ring[kAhead];
#pragma unroll
        for (int l = 0; l < kAhead; ++l) ring[l] = first[l];
        dte_levels(T, upd, bound, ring, sT, sE, px, py, pz);
        const double f = start / total();
        // renormalise, B(h), A(h), and the next sub-step's A(h), B(h)
        const bool last = it + 1 == nloop;
        for (int s = t; s < M.C; s += B) {
            const double2 a = src[s];
            double Tn;
            double ee = dte_relax_steps(sE[s] * f, a.x, a.y, last ? 1 : 2, Tn);
            if (last) {
                ee += a.x;
                Tn = ee_to_te(ee);
            }
            sE[s] = ee;
            sT[s] = Tn;
        }
        __syncthreads();
    }
    for (int s = t; s < M.C; s += B) {
        const int c = T.origin + (slot[s] >> 1);
        M.Ee[c] = sE[s];
        M.Te[c] = sT[s];
    }
}

}  // namespace sld
