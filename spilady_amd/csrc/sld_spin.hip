// The spin sweep kernel (calculate_spin_CPU.cpp:33-199, core_ds_CPU.cpp:35-127).
//
// Compiled with the two-address FMA off (-fmacf64-inst), like sld_dte.hip: the
// series coefficients then stay in scalar registers.
#include <hip/hip_runtime.h>

#include "sld_kernels.h"

namespace sld {

// The Landau field plus the Heisenberg correction -(sum J|s_j|/|s|) s is m s
// with m = -(2A + 4B s^2 + 6C s^4 + 8D s^6) - sum J|s_j| / |s|
// (calculate_spin_CPU.cpp:131-140); lan holds the four coefficients
// -2A, -4B, -6C, -8D. A spin of length zero has no direction to be corrected
// along: the bound on s^2 keeps m finite there.
__device__ __forceinline__ double landau_scale(double3 s, const double4& lan, double sjs) {
    const double s2 = sq3(s);
    const double k = fma(fma(fma(lan.w, s2, lan.z), s2, lan.y), s2, lan.x);
    return fma(-sjs, rsqrt_normal(fmax(s2, 1e-300)), k);
}

// Rotation of s about Heff by |Heff| dt / hbar (core_ds_CPU.cpp:90-127), made
// once for both half-rotations of a step. With w = -Heff dt / hbar (its length
// is the angle) and x = w.w,
//   s' = s + S w x s + C w x (w x s),  S = sin|w| / |w|,  C = (1 - cos|w|) / x,
// the Rodrigues form without the axis: S and C are series in x, so an angle up
// to 1 rad (a step of 1 fs turns a spin by 0.2 to 0.4) needs no square root,
// division or sincos, and 1 - cos does not cancel. A larger angle is halved n
// times, then doubled back: with h half the angle, S = S(h) cos h, C = S(h)^2 / 2
// and cos h = 1 - h^2 C(h).
struct Rot {
    double3 w;
    double S, C;
};

__device__ __forceinline__ Rot make_rot(double3 H, double dt) {
    // sum (-x)^n / (2n+1)! and / (2n+2)!: the next terms are 1/19! and 1/20!
    constexpr double kS[9] = {1.0,
                              -1.0 / 6.0,
                              1.0 / 120.0,
                              -1.0 / 5040.0,
                              1.0 / 362880.0,
                              -1.0 / 39916800.0,
                              1.0 / 6227020800.0,
                              -1.0 / 1307674368000.0,
                              1.0 / 355687428096000.0};
    constexpr double kC[9] = {1.0 / 2.0,
                              -1.0 / 24.0,
                              1.0 / 720.0,
                              -1.0 / 40320.0,
                              1.0 / 3628800.0,
                              -1.0 / 479001600.0,
                              1.0 / 87178291200.0,
                              -1.0 / 20922789888000.0,
                              1.0 / 6402373705728000.0};
    Rot r;
    r.w = mul3(-dt / kHbar, H);
    double x = sq3(r.w);
    int n = 0;
    while (__builtin_expect(x > 1.0 && n < 600, 0)) {
        x *= 0.25;
        ++n;
    }
    r.S = horner2(kS, x);
    r.C = horner2(kC, x);
    while (__builtin_expect(n > 0, 0)) {
        const double c = fma(-x, r.C, 1.0);
        r.C = 0.5 * r.S * r.S;
        r.S *= c;
        x *= 4.0;
        --n;
    }
    return r;
}

__device__ __forceinline__ double3 apply_rot(const Rot& r, double3 s) {
    const double3 t = cross3(r.w, s);
    const double3 u = cross3(r.w, t);
    return make_double3(fma(r.C, u.x, fma(r.S, t.x, s.x)), fma(r.C, u.y, fma(r.S, t.y, s.y)),
                        fma(r.C, u.z, fma(r.S, t.z, s.z)));
}

// value of the lane whose index differs in bit 0 (XOR = 1) or bit 1 (XOR = 2)
template <int XOR>
__device__ __forceinline__ double quad_swap(double v) {
    constexpr int kPerm = XOR == 1 ? 0xb1 : 0x4e;  // quad_perm [1,0,3,2], [2,3,0,1]
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, kPerm, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), kPerm, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double quad_sum(double v) {
    v += quad_swap<1>(v);
    return v + quad_swap<2>(v);
}

// One dependency level of a core_ds sweep: each listed cell walks its list
// head to tail (forward) or tail to head (backward)
// (calculate_spin_CPU.cpp:33-235, core_ds_CPU.cpp:35-83).
//
// Cells of a level do not interact, so all a walk can miss of its neighbours
// are the new spins of its own cell's earlier atoms. A wave takes up to 16
// cells in two phases:
// 1. four lanes per atom: the field H = Hext + sum J s_j and S = sum J|s_j|
//    over the spins as they are, lane j adding list entries 4j..4j+3 and
//    4j+16..4j+19; J of each pair of atoms of one cell goes into a triangle in
//    LDS;
// 2. the lanes of a cell walk it: an atom is updated from LDS alone, and what
//    its spin changed by is added to the fields of the cell's later atoms.
// The sum H + sum J (s_new - s_old) is the field of the sequential walk up to
// the rounding of the corrections. Every lane of a cell computes the same
// update and the additions to one field come in walking order, so the result
// does not depend on the lanes, nor on the cells per wave.
//
// A walk that loads as it goes waits for memory once an atom and fetches a
// neighbour's line again for every atom that reads it; here a launch waits
// about four times in all. What is left is the update itself, 240 instructions
// a visit (about 0.7 us for a wave on its own) and, at 2 M atoms, the traffic:
// 41.7 us a level on average (108 MB) where the walk took 46 (164 MB); levels
// of 27 cells of 9 atoms 18.5 us instead of 30, of 960 cells 15.0 instead of 18.
// LDS is kept to 14 KB for 11 waves a compute unit: with 22 KB (16 cells a
// wave) 2 M atoms took 50 us.

constexpr int kSpinAtoms = 80;    // atoms of a wave's pass in LDS (8 cells of 10)
constexpr int kSpinPairs = 496;   // and pairs of atoms of one cell (one of 32, 8 of 11)
static_assert(kSpinAtoms >= kCellCap && kSpinPairs >= kCellCap * (kCellCap - 1) / 2, "any one cell fits a pass");
static_assert(kMaxMag == 32, "four lanes hold an atom's list in two chunks of four each");

// lanes: lanes that walk a cell, a power of two with ncw * lanes <= 64
template <bool kLang>
__global__ __launch_bounds__(64) void k_spin_phase(const int* cells, int ncell, int ncw, int lanes, int backward,
                                                   int store_fields, double dt, Phys P, Dev D) {
    __shared__ double sH[4][kSpinAtoms];              // field x, y, z and sum J|s_j|
    __shared__ double sS[4][kSpinAtoms];              // spin x, y, z and its length
    __shared__ double sZ[kLang ? 3 : 1][kSpinAtoms];  // Langevin normals
    __shared__ double sL[kLang ? 4 : 1][kSpinAtoms];  // Landau coefficients
    __shared__ int sA[kSpinAtoms];                    // atom
    __shared__ double sJ[kSpinPairs];
    const int lane = threadIdx.x;
    const int lb = xcd_block((ncell + ncw - 1) / ncw);
    if (lb < 0) return;
    // lane k < ncw: the k-th cell of the wave
    int c = -1, n = 0;
    if (lane < ncw && lb * ncw + lane < ncell) {
        c = cells[lb * ncw + lane];
        n = D.cn[c];
    }
    // atoms and pairs of the cells up to this lane's
    int atoms = n, pairs = n * (n - 1) / 2;
#pragma unroll
    for (int d = 1; d < 16; d <<= 1) {
        const int ta = __shfl_up(atoms, d, 64), tp = __shfl_up(pairs, d, 64);
        if (lane >= d) {
            atoms += ta;
            pairs += tp;
        }
    }
    const int atom0 = atoms - n, pair0 = pairs - n * (n - 1) / 2;
    const double dth = dt / 2.0, gS = P.gamma_S;
    const double ch = gS * dth, cq = gS * (dt / 4.0);
    double cz = 0.0;
    if (kLang && c >= 0) {
        const double Tk = P.eltemp ? D.Te[c] : D.rep[D.crep[c]].temperature;
        cz = dt * sqrt(2.0 * Tk * gS / dt);
    }
    // passes over as many cells as fit in LDS
    for (int k0 = 0; k0 < ncw;) {
        const int a0 = __builtin_amdgcn_readlane(atom0, k0), p0 = __builtin_amdgcn_readlane(pair0, k0);
        const unsigned long long fit =
            __ballot(lane >= k0 && lane < ncw && atoms - a0 <= kSpinAtoms && pairs - p0 <= kSpinPairs);
        const int k1 = k0 + __builtin_ctzll(~(fit >> k0));  // cells [k0, k1)
        const int natom = __builtin_amdgcn_readlane(atoms, k1 - 1) - a0;
        const int npair = __builtin_amdgcn_readlane(pairs, k1 - 1) - p0;
        for (int i = lane; i < npair; i += 64) sJ[i] = 0.0;
        wave_fence();
        const int j = lane & 3;
        for (int f0 = 0; f0 < natom; f0 += 16) {
            const int f = f0 + (lane >> 2);
            int k = k0;
            for (int q = k0 + 1; q < k1; ++q) k += f >= __builtin_amdgcn_readlane(atom0, q) - a0 ? 1 : 0;
            const int ck = __shfl(c, k, 64), nk = __shfl(n, k, 64);
            const int q = f - (__shfl(atom0, k, 64) - a0);
            double* tri = sJ + (__shfl(pair0, k, 64) - p0) + q * (q - 1) / 2;  // pairs of the atom and its predecessors
            if (f < natom) {
                const int a = D.cl[ck * kCellCap + (backward ? nk - 1 - q : q)];
                const int nm = D.nbmn[a];
                // lane j's part of what the update needs besides the field
                double4 own = make_double4(0.0, 0.0, 0.0, 0.0), he = own;
                if (j == 0) own = D.s[a];
                if (kLang && j == 1) own = D.zn[a];
                if (kLang && j == 2) own = D.lan[a];
                if (P.extfield && j == 0) he = D.hext[a];
                double hx = he.x, hy = he.y, hz = he.z, ss = 0.0;
                for (int b0 = 4 * j; b0 < nm; b0 += 16) {
                    const int4 i0 = *reinterpret_cast<const int4*>(D.nbm + (size_t)a * kMaxMag + b0);
                    const double2* js = reinterpret_cast<const double2*>(D.nbJ + (size_t)a * kMaxMag + b0);
                    const double2 j0 = js[0], j1 = js[1];
                    int id[4] = {i0.x, i0.y, i0.z, i0.w};
                    const double J[4] = {j0.x, j0.y, j1.x, j1.y};
                    double4 sj[4];
                    int sl[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (b0 + e >= nm) id[e] = a;
                        sj[e] = D.s[id[e]];
                        sl[e] = D.cslot[id[e]];
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const double Je = b0 + e < nm ? J[e] : 0.0;
                        hx = fma(Je, sj[e].x, hx);
                        hy = fma(Je, sj[e].y, hy);
                        hz = fma(Je, sj[e].z, hz);
                        ss = fma(Je, sj[e].w, ss);
                        const int pos = sl[e] - ck * kCellCap;  // in the list of this cell if 0 <= pos < nk
                        const int qe = backward ? nk - 1 - pos : pos;
                        if ((unsigned)pos < (unsigned)nk && qe < q && b0 + e < nm) tri[qe] = Je;
                    }
                }
                hx = quad_sum(hx);
                hy = quad_sum(hy);
                hz = quad_sum(hz);
                ss = quad_sum(ss);
                if (j == 0) {
                    sS[0][f] = own.x; sS[1][f] = own.y; sS[2][f] = own.z; sS[3][f] = own.w;
                    sA[f] = a;
                }
                if (kLang && j == 1) {
                    sZ[0][f] = own.x; sZ[kLang ? 1 : 0][f] = own.y; sZ[kLang ? 2 : 0][f] = own.z;
                }
                if (kLang && j == 2) {
                    sL[0][f] = -2.0 * own.x; sL[kLang ? 1 : 0][f] = -4.0 * own.y;
                    sL[kLang ? 2 : 0][f] = -6.0 * own.z; sL[kLang ? 3 : 0][f] = -8.0 * own.w;
                }
                if (j == 3) {
                    sH[0][f] = hx; sH[1][f] = hy; sH[2][f] = hz; sH[3][f] = ss;
                }
            }
        }
        wave_fence();
        const int k = k0 + lane / lanes, sub = lane & (lanes - 1);
        const int kk = min(k, k1 - 1);
        const int nk = __shfl(n, kk, 64);
        const int base = __shfl(atom0, kk, 64) - a0;
        const double* tri0 = sJ + (__shfl(pair0, kk, 64) - p0);
        const double ck = __shfl(cz, kk, 64);
        const int nw = k < k1 ? nk : 0;
        for (int q = 0; q < nw; ++q) {
            const int f = base + q;
            const double3 H = make_double3(sH[0][f], sH[1][f], sH[2][f]);
            const double S = sH[3][f];
            const double4 old = make_double4(sS[0][f], sS[1][f], sS[2][f], sS[3][f]);
            const int a = sA[f];
            double3 s = d3(old);
            double3 L = make_double3(0.0, 0.0, 0.0);
            if (!kLang) {
                s = apply_rot(make_rot(H, dt), s);
            } else {
                const double4 lc = make_double4(sL[0][f], sL[kLang ? 1 : 0][f], sL[kLang ? 2 : 0][f],
                                                sL[kLang ? 3 : 0][f]);
                // s + c (H + m v): a stage of the RK2 of the damping, m v the Landau field at v
                auto stage = [&](double3 at, double c, double m, double3 v) {
                    return make_double3(fma(c, fma(m, v.x, H.x), at.x), fma(c, fma(m, v.y, H.y), at.y),
                                        fma(c, fma(m, v.z, H.z), at.z));
                };
                const Rot R = make_rot(H, dth);
                s = apply_rot(R, s);
                double3 st = stage(s, cq, landau_scale(s, lc, S), s);
                s = stage(s, ch, landau_scale(st, lc, S), st);
                s = make_double3(fma(ck, sZ[0][f], s.x), fma(ck, sZ[kLang ? 1 : 0][f], s.y),
                                 fma(ck, sZ[kLang ? 2 : 0][f], s.z));
                st = stage(s, cq, landau_scale(s, lc, S), s);
                const double m = landau_scale(st, lc, S);
                s = stage(s, ch, m, st);
                L = mul3(m, st);
                s = apply_rot(R, s);
            }
            const double w = spin_len(s);
            const double3 ds = sub3(s, d3(old));
            const double dw = w - old.w;
            for (int p = q + 1 + sub; p < nk; p += lanes) {
                const double J = tri0[p * (p - 1) / 2 + q];
                const int g = base + p;
                sH[0][g] = fma(J, ds.x, sH[0][g]);
                sH[1][g] = fma(J, ds.y, sH[1][g]);
                sH[2][g] = fma(J, ds.z, sH[2][g]);
                sH[3][g] = fma(J, dw, sH[3][g]);
            }
            if (sub == 0) {
                D.s[a] = make_double4(s.x, s.y, s.z, w);
                // the fields of the forward sweep are overwritten by the
                // backward sweep before anything reads them
                if (store_fields) {
                    if (kLang) D.sjs[a] = S;
                    D.hh[a] = make_double4(H.x, H.y, H.z, 0.0);
                    D.hl[a] = make_double4(L.x, L.y, L.z, 0.0);
                }
            }
            wave_fence();
        }
        k0 = k1;
    }
}
template __global__ void k_spin_phase<false>(const int*, int, int, int, int, int, double, Phys, Dev);
template __global__ void k_spin_phase<true>(const int*, int, int, int, int, int, double, Phys, Dev);

}  // namespace sld
