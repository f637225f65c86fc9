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
// division or sincos, and 1 - cos does not cancel. A larger angle is brought to
// [-pi/4, pi/4] by quarter turns, pi/2 in two doubles: exactly, for any angle of
// less than 2^50; beyond that an angle's own last bit is more than a turn, and
// the loop only keeps the result a rotation.
struct Rot {
    double3 w, v;  // v = C w
    double S;
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
    const double x = sq3(r.w);
    double y = x, a = 0.0, angle = 0.0;
    int q = 0;  // quarter turns
    const bool large = __builtin_expect(!(x <= 1.0), 0);
    if (large) {
        constexpr double kHi = 1.5707963267948966, kLo = 6.123233995736766e-17;  // pi/2
        angle = a = sqrt_any(x);
        for (int n = 0; n < 24 && !(fabs(a) <= 0.8); ++n) {
            const double k = rint(a * (1.0 / kHi));
            a = fma(-k, kLo, fma(-k, kHi, a));
            q += (int)fma(-4.0, floor(0.25 * k), k);
        }
        y = a * a;
    }
    r.S = horner2(kS, y);
    double C = horner2(kC, y);
    if (large) {
        const double sn = a * r.S, vs = y * C, cs = 1.0 - vs;  // sin, 1 - cos, cos
        q &= 3;
        r.S = (q == 0 ? sn : q == 1 ? cs : q == 2 ? -sn : -cs) / angle;
        C = (q == 0 ? vs : q == 1 ? 1.0 + sn : q == 2 ? 1.0 + cs : 1.0 - sn) / x;
    }
    r.v = mul3(C, r.w);
    return r;
}

// s + (S t + (C w) x t), t = w x s: the turn first, its roundings being those of
// the smaller sum (0.9e-16 at 0.3 rad; added to s term by term 1.1e-16, and 1 % less time)
__device__ __forceinline__ double3 apply_rot(const Rot& r, double3 s) {
    const double3 t = cross3(r.w, s);
    return make_double3(s.x + fma(r.v.y, t.z, fma(-r.v.z, t.y, r.S * t.x)),
                        s.y + fma(r.v.z, t.x, fma(-r.v.x, t.z, r.S * t.y)),
                        s.z + fma(r.v.x, t.y, fma(-r.v.y, t.x, r.S * t.z)));
}

// value of the lane N places before in the row of 16, or 0
template <int N>
__device__ __forceinline__ int row_shr(int v) {
    return __builtin_amdgcn_update_dpp(0, v, 0x110 + N, 0xf, 0xf, true);
}

// v | the values of the other three lanes of the quad
__device__ __forceinline__ unsigned quad_or(unsigned v) {
    v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0xb1, 0xf, 0xf, true);
    return v | (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x4e, 0xf, 0xf, true);
}

// One dependency level of a core_ds sweep: each listed cell walks its list
// head to tail (forward) or tail to head (backward)
// (calculate_spin_CPU.cpp:33-235, core_ds_CPU.cpp:35-83).
//
// Cells of a level do not interact, so all a walk can miss of its neighbours
// are the new spins of its own cell's earlier atoms. And of those it needs only
// the ones within the exchange range: an atom whose earlier neighbours in the
// cell are done can be updated, whatever else is still to come. A wave takes
// the cells that fit its 64 lanes, a lane per atom:
// 1. four lanes gather an atom's field H = Hext + sum J s_j and S = sum J|s_j|
//    over the spins as they are, lane j adding list entries 4j..4j+3 and
//    4j+16..4j+19; J of each pair of atoms of one cell goes into a triangle in
//    LDS, and the atom's earlier neighbours into a bit mask;
// 2. in each round the atoms that wait for none are updated, and then every
//    atom adds J times their change to its own field, in walking order.
// The sum H + sum J (s_new - s_old) is the field of the sequential walk up to
// the rounding of the corrections. A cell's rounds depend on its own atoms
// only, so the result does not depend on how many cells share a wave.
//
// A walk that loads as it goes waits for memory once an atom and fetches a
// neighbour's line again for every atom that reads it; here a launch waits
// about four times in all. The update is a chain of 250 instructions, about 0.7
// us for a wave on its own, so rounds count: cells of 9.3 atoms on average and
// 16 at most need 6.1 and 9 of them, cells of 6.5 and 10 need 4.9 and 6.
// At 27 cells a launch that leaves 3 us of launch, 2 of first loads, 1 of
// gathering and 4 of rounds: 10.0 us where the walk atom by atom took 16.5. Of
// 2 M atoms a level moves 104 MB in 31.5 us (39.5); registers are kept to 128 for
// four waves a SIMD, the atoms' own values loaded after the gathering (before
// it: 150 registers, 1 us more at 64 x 16,000 atoms, 0.2 less at 2,000).

constexpr int kSpinPairs = 496;  // pairs of atoms of one cell in a pass (one of 32, 8 of 11)
static_assert(kCellCap <= 32 && kSpinPairs >= kCellCap * (kCellCap - 1) / 2, "any one cell fits a pass");
static_assert(kMaxMag == 32, "four lanes hold an atom's list in two chunks of four each");

template <bool kLang>
__global__ __launch_bounds__(64) void k_spin_phase(const int* cells, int ncell, int ncw, int backward,
                                                   int store_fields, double dt, Phys P, Dev D) {
    __shared__ double sV[4][64];  // phase 1: field x, y, z and sum J|s_j|; phase 2: change of the spin and its length
    __shared__ unsigned sM[64];   // bit q: the atom's neighbour at place q of its cell's walk comes earlier
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
    // atoms and pairs of the cells before this lane's, in the low and the high half
    const int own_sum = n | (n * (n - 1) / 2) << 16;
    int sum = own_sum;
    sum += row_shr<1>(sum);
    sum += row_shr<2>(sum);
    sum += row_shr<4>(sum);
    sum += row_shr<8>(sum);
    const int atoms = sum & 0xffff, pairs = sum >> 16;
    const int sum0 = sum - own_sum;
    const double dth = dt / 2.0, gS = P.gamma_S;
    const double ch = gS * dth, cq = gS * (dt / 4.0), noise = 2.0 * gS / dt;
    // passes over as many cells as fit the lanes and the triangles
    for (int k0 = 0; k0 < ncw;) {
        const int s0 = __builtin_amdgcn_readlane(sum0, k0), a0 = s0 & 0xffff, p0 = s0 >> 16;
        const unsigned long long fit =
            __ballot(lane >= k0 && lane < ncw && atoms - a0 <= 64 && pairs - p0 <= kSpinPairs);
        const int k1 = k0 + __builtin_ctzll(~(fit >> k0));  // cells [k0, k1)
        const int natom = __builtin_amdgcn_readlane(atoms, k1 - 1) - a0;
        // this lane's atom: cell ck of nk atoms, the first of them in lane base, place q in its walk
        int ck = __builtin_amdgcn_readlane(c, k0), nk = __builtin_amdgcn_readlane(n, k0), base = 0, tri = 0;
        for (int u = k0 + 1; u < k1; ++u) {
            const int su = __builtin_amdgcn_readlane(sum0, u) - s0;
            const int cu = __builtin_amdgcn_readlane(c, u), nu = __builtin_amdgcn_readlane(n, u);
            if (lane >= (su & 0xffff)) {
                ck = cu;
                nk = nu;
                base = su & 0xffff;
                tri = su >> 16;
            }
        }
        const int q = lane - base;
        tri += q * (q - 1) / 2;  // pairs of the atom and its predecessors
        const bool mine = lane < natom;
        int a = 0, rep = 0;
        double Tk = 0.0;
        double4 own = make_double4(0.0, 0.0, 0.0, 0.0), lc = own, zn = own;
        double3 H = d3(own);
        if (mine) {
            a = D.cl[ck * kCellCap + (backward ? nk - 1 - q : q)];
            if (kLang && !P.eltemp) rep = D.crep[ck];
        }
        const int j = lane & 3;
        const int place = (tri << 16) | (q << 8) | nk;
        for (int f0 = 0; f0 < natom; f0 += 16) {
            const int f = f0 + (lane >> 2);
            const int af = __shfl(a, f, 64), cf = __shfl(ck, f, 64), pf = __shfl(place, f, 64);
            const int qf = (pf >> 8) & 255, nf = pf & 255;
            double* trif = sJ + (pf >> 16);
            if (f < natom) {
                double hx = 0.0, hy = 0.0, hz = 0.0, ss = 0.0;
                unsigned earlier = 0;
                // the first chunk's ids and J do not wait for the list's length
                const int* ids = D.nbm + (size_t)af * kMaxMag + 4 * j;
                const double2* js = reinterpret_cast<const double2*>(D.nbJ + (size_t)af * kMaxMag + 4 * j);
                int4 i0 = *reinterpret_cast<const int4*>(ids);
                double2 j0 = js[0], j1 = js[1];
                const int nm = D.nbmn[af];
                for (int b0 = 4 * j; b0 < nm; b0 += 16) {
                    if (b0 >= 16) {
                        i0 = *reinterpret_cast<const int4*>(ids + 16);
                        j0 = js[8];
                        j1 = js[9];
                    }
                    int id[4] = {i0.x, i0.y, i0.z, i0.w};
                    const double J[4] = {j0.x, j0.y, j1.x, j1.y};
                    double4 sj[4];
                    int sl[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (b0 + e >= nm) id[e] = af;
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
                        const int pos = sl[e] - cf * kCellCap;  // in the list of this cell if 0 <= pos < nf
                        const int qe = backward ? nf - 1 - pos : pos;
                        if ((unsigned)pos < (unsigned)nf && qe < qf && b0 + e < nm) {
                            trif[qe] = Je;
                            earlier |= 1u << qe;
                        }
                    }
                }
                hx = quad_sum(hx);
                hy = quad_sum(hy);
                hz = quad_sum(hz);
                ss = quad_sum(ss);
                earlier = quad_or(earlier);
                sV[j][f] = j == 0 ? hx : j == 1 ? hy : j == 2 ? hz : ss;
                if (j == 0) sM[f] = earlier;
            }
        }
        if (mine) {
            own = D.s[a];
            if (kLang) {
                lc = D.lan[a];
                zn = D.zn[a];
                Tk = P.eltemp ? D.Te[ck] : D.rep[rep].temperature;
            }
            if (P.extfield) H = d3(D.hext[a]);
        }
        wave_fence();
        double S = 0.0;
        unsigned long long earlier = 0;  // lanes whose atoms this one waits for
        if (mine) {
            H = make_double3(H.x + sV[0][lane], H.y + sV[1][lane], H.z + sV[2][lane]);
            S = sV[3][lane];
            earlier = (unsigned long long)sM[lane] << base;
        }
        wave_fence();
        lc = make_double4(-2.0 * lc.x, -4.0 * lc.y, -6.0 * lc.z, -8.0 * lc.w);
        const double czk = dt * sqrt_any(Tk * noise);
        const double* J0 = sJ + tri - base;  // J0[u]: with the atom of lane u
        double3 s = d3(own), L = make_double3(0.0, 0.0, 0.0);
        double w = own.w;
        // a round ends at least the first atom of each walk that is not done
        const unsigned long long all = natom < 64 ? (1ull << natom) - 1 : ~0ull;
        for (unsigned long long done = 0; done != all;) {
            const bool ready = mine && !((done >> lane) & 1) && !(earlier & ~done);
            const unsigned long long now = __ballot(ready);
            if (ready) {
                if (!kLang) {
                    s = apply_rot(make_rot(H, dt), s);
                } else {
                    // s + c (H + m v): a stage of the RK2 of the damping, m v the Landau field at v
                    auto stage = [&](double3 at, double c, double m, double3 v) {
                        return make_double3(fma(c, fma(m, v.x, H.x), at.x), fma(c, fma(m, v.y, H.y), at.y),
                                            fma(c, fma(m, v.z, H.z), at.z));
                    };
                    const Rot R = make_rot(H, dth);
                    s = apply_rot(R, s);
                    double3 st = stage(s, cq, landau_scale(s, lc, S), s);
                    s = stage(s, ch, landau_scale(st, lc, S), st);
                    s = make_double3(fma(czk, zn.x, s.x), fma(czk, zn.y, s.y), fma(czk, zn.z, s.z));
                    st = stage(s, cq, landau_scale(s, lc, S), s);
                    const double m = landau_scale(st, lc, S);
                    s = stage(s, ch, m, st);
                    L = mul3(m, st);
                    s = apply_rot(R, s);
                }
                w = spin_len(s);
                sV[0][lane] = s.x - own.x;
                sV[1][lane] = s.y - own.y;
                sV[2][lane] = s.z - own.z;
                sV[3][lane] = w - own.w;
            }
            wave_fence();
            for (unsigned long long m = earlier & now; m; m &= m - 1) {
                const int u = __builtin_ctzll(m);
                const double J = J0[u];
                H = make_double3(fma(J, sV[0][u], H.x), fma(J, sV[1][u], H.y), fma(J, sV[2][u], H.z));
                S = fma(J, sV[3][u], S);
            }
            wave_fence();
            done |= now;
        }
        if (mine) {
            D.s[a] = make_double4(s.x, s.y, s.z, w);
            // the fields of the forward sweep are overwritten by the
            // backward sweep before anything reads them
            if (store_fields) {
                if (kLang) D.sjs[a] = S;
                D.hh[a] = make_double4(H.x, H.y, H.z, 0.0);
                D.hl[a] = make_double4(L.x, L.y, L.z, 0.0);
            }
        }
        k0 = k1;
    }
}
template __global__ void k_spin_phase<false>(const int*, int, int, int, int, double, Phys, Dev);
template __global__ void k_spin_phase<true>(const int*, int, int, int, int, double, Phys, Dev);

}  // namespace sld
