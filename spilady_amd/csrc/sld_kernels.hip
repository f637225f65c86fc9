// HIP kernels of the spin-lattice engine (gfx950, FP64).
//
// Work decomposition: a wave per link cell for the neighbour build and density,
// four lanes per atom for the force pass, eight lanes per link cell for the
// Langevin momentum with local collective motion and the cell temperatures.
// The spin sweeps are launched one dependency level at a time by the host;
// within a launch no two cells interact. The electron diffusion sweeps run all
// their levels inside tiles of the mesh.
#include <hip/hip_runtime.h>

#include "../../include/spilady_hip.h"
#include "sld_kernels.h"

namespace sld {

// ---------------------------------------------------------------------------
// reductions

// out[k] = sum over blocks of partials[k*nblk + b]; one block of 256 threads for each k.
__global__ __launch_bounds__(256) void k_reduce(const double* partials, int nblk, double* out) {
    __shared__ double sh[256];
    const int t = threadIdx.x, k = blockIdx.x;
    double acc = 0.0;
    for (int b = t; b < nblk; b += 256) acc += partials[(size_t)k * nblk + b];
    sh[t] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (t < s) sh[t] += sh[t + s];
        __syncthreads();
    }
    if (t == 0) out[k] = sh[0];
}

// Per-replica sums: block r of the grid (1,024 threads) reduces partial rows
// [seg[r], seg[r+1]) into out[r * kScal + out_off + k], in an order fixed by
// the row count alone: thread t adds rows t, t + 1024, ... in turn, each wave
// sums its lanes (wave_sum), thread 0 adds the 16 wave sums in order.
__global__ __launch_bounds__(1024) void k_reduce_seg(const double* partials, const int* seg, int nk, double* out,
                                                     int out_off) {
    constexpr int KG = 4;  // components summed together
    __shared__ double sh[KG][16];
    const int t = threadIdx.x;
    const int b0 = seg[blockIdx.x], nb = seg[blockIdx.x + 1] - b0;
    const size_t ntot = (size_t)seg[gridDim.x];  // rows of each component
    for (int k0 = 0; k0 < nk; k0 += KG) {
        const int kk = min(KG, nk - k0);
        // thread t adds rows t + 1024 u in order, eight rows of up to four
        // components in flight
        double acc[KG] = {0.0, 0.0, 0.0, 0.0};
        for (int c0 = t; c0 < nb; c0 += 8 * 1024) {
            double v[8][KG];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int b = c0 + u * 1024;
#pragma unroll
                for (int q = 0; q < KG; ++q)
                    v[u][q] = b < nb && q < kk ? partials[(k0 + q) * ntot + b0 + b] : 0.0;
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int q = 0; q < KG; ++q) acc[q] += v[u][q];
        }
#pragma unroll
        for (int q = 0; q < KG; ++q) {
            acc[q] = wave_sum(acc[q]);
            if ((t & 63) == 0) sh[q][t >> 6] = acc[q];
        }
        __syncthreads();
        if (t < kk) {
            double a = 0.0;
            for (int w = 0; w < 16; ++w) a += sh[t][w];
            out[(size_t)blockIdx.x * kScal + out_off + k0 + t] = a;
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// links (links_CPU.cpp:85-177)

__device__ __forceinline__ bool cells_adjacent(const Box& b, int c0, int c1) {
    int x0 = c0 % b.nx, y0 = (c0 / b.nx) % b.ny, z0 = c0 / (b.nx * b.ny);
    int x1 = c1 % b.nx, y1 = (c1 / b.nx) % b.ny, z1 = c1 / (b.nx * b.ny);
    int dx = (x1 - x0 + b.nx) % b.nx, dy = (y1 - y0 + b.ny) % b.ny, dz = (z1 - z0 + b.nz) % b.nz;
    return (dx <= 1 || dx == b.nx - 1) && (dy <= 1 || dy == b.ny - 1) && (dz <= 1 || dz == b.nz - 1);
}

// new cell of every atom (clamped binning of links_CPU.cpp:96-112)
__global__ __launch_bounds__(256) void k_bin(Dev D) {
    int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= D.N) return;
    const int rr = D.arep[a];
    if (rr < 0) return;
    const Rep& R = D.rep[rr];
    const int old = D.cell[a];
    const int lc = bin_cell(R.box, d3(D.r[a]));
    const int c = R.cell0 + lc;
    D.cell_prev[a] = old;
    D.cell[a] = c;
    if (c != old) {
        if (!cells_adjacent(R.box, old - R.cell0, lc)) atomicOr(D.err, kErrFarMove);
        const int slot = atomicAdd(D.inc_n + c, 1);
        if (slot < kCellCap) D.inc[c * kCellCap + slot] = a;
    }
}

// Rebuild cell c's list. The reference detaches every mover and pushes it at
// the head of its new cell in ascending atom index (links_CPU.cpp:144-173),
// so a cell's new list is [movers in, descending index] + [stayers, old order].
// k_bin has pushed this step's movers into the cell's incoming list in
// arbitrary order; sorting them by index makes the list deterministic.
__global__ __launch_bounds__(128) void k_relink(const int* cl_old, const int* cn_old, Dev D) {
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= D.C) return;
    const int rr = D.crep[c];
    if (rr < 0) return;
    int mv[kCellCap];
    const int ninc = D.inc_n[c];
    bool over = ninc > kCellCap;
    const int nm = over ? kCellCap : ninc;
    for (int k = 0; k < nm; ++k) {
        const int a = D.inc[c * kCellCap + k];
        // insertion keeping descending atom index
        int q = k;
        while (q > 0 && mv[q - 1] < a) { mv[q] = mv[q - 1]; --q; }
        mv[q] = a;
    }
    if (ninc != 0) D.inc_n[c] = 0;
    int* out = D.cl + c * kCellCap;
    int k = 0;
    for (int q = 0; q < nm; ++q) {
        D.cslot[mv[q]] = c * kCellCap + k;
        out[k++] = mv[q];
    }
    int n = cn_old[c];
    for (int q = 0; q < n; ++q) {
        int a = cl_old[c * kCellCap + q];
        if (D.cell[a] == c) {
            if (k < kCellCap) {
                D.cslot[a] = c * kCellCap + k;
                out[k++] = a;
            } else {
                over = true;
            }
        }
    }
    D.cn[c] = k;
    if (over) atomicOr(D.err, kErrCellOverflow);
}

// ---------------------------------------------------------------------------
// neighbour list + density (calculate_rho_CPU.cpp:33-92 for rho, the 27-cell
// scan order of calculate_spin_CPU.cpp:201-235 for the lists)
//
// One wavefront per link cell. The ids of the 27 cells' atoms (slots 0..25,
// then the cell itself, each in list order) are staged in LDS; every lane
// holds up to kCandReg candidate positions in registers. The wave walks the
// cell's atoms and tests all candidates at once; the pairs in range, about one
// test in six, are compacted with a ballot and a lane prefix count into a
// buffer in LDS, so each list keeps the reference's scan order. Then the
// buffered pairs of all the cell's atoms, one per lane, take their square
// root, table rows and list entries: 156 pairs in 3 turns of the wave where
// the tests' lanes would take 18. 2 M atoms take 0.97 ms where lookups inside
// the tests took 1.81 (2,130 to 1,250 instructions a wave, and LDS by the wave
// for 20 waves a compute unit instead of 10); 250,000 atoms 0.24 to 0.135. What
// is left is the tests' arithmetic and 0.7 GB of list entries.

constexpr int kMaxCand = 27 * kCellCap;     // upper bound of candidates
constexpr int kCandReg = 4;                 // passes of 64 candidates held in registers
constexpr int kPairBuf = 256;               // pairs buffered before their table lookups
static_assert(kPairBuf >= kMaxNb, "the pairs of an atom fit the buffer");
static_assert(kNbLds == kPairBuf * 16 + kMaxCand * 4 && kNbLds % 8 == 0, "LDS of a wave");

// lanes below this one that are set in a ballot
__device__ __forceinline__ int lanes_before(unsigned long long m) {
    return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}


static_assert(kCellCap <= 64, "k_nbuild holds a cell's own atoms one per lane");

// lane l's value of v, as a wave-uniform double
__device__ __forceinline__ double readlane_f64(double v, int l) {
    const unsigned long long u = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)u, l);
    const unsigned hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

__global__ __launch_bounds__(256) void k_nbuild(Tables T, Phys P, Dev D, int write_rho) {
    extern __shared__ double s_nb[];  // kNbLds bytes a wave
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    double* rsqs = s_nb + w * (kNbLds / 8);                    // squared distance, then density term
    int2* pairs = reinterpret_cast<int2*>(rsqs + kPairBuf);    // neighbour; own atom | position << 8 | (rcut_mag position + 1) << 16
    int* cand = reinterpret_cast<int*>(pairs + kPairBuf);
    const int wpb = blockDim.x >> 6;
    const int lb = xcd_block((D.C + wpb - 1) / wpb);
    if (lb < 0) return;  // whole padding block, before any barrier
    const int c = lb * wpb + w;
    const int rr = __builtin_amdgcn_readfirstlane(c < D.C ? D.crep[c] : -1);
    const bool valid = rr >= 0;
    Box b{};
    int cell0 = 0;
    if (valid) {
        b = D.rep[rr].box;
        cell0 = D.rep[rr].cell0;
    }
    int cid = 0, cnt = 0;
    if (valid && lane < 27) {
        cid = lane < 26 ? cell0 + neigh_cell(b, c - cell0, lane) : c;
        cnt = D.cn[cid];
    }
    int incl = cnt;
#pragma unroll
    for (int d = 1; d < 32; d <<= 1) {
        int t = __shfl_up(incl, d, 64);
        if (lane >= d) incl += t;
    }
    const int total = __shfl(incl, 26, 64);
    if (valid && lane < 27) {
        // eight list entries at a time, both loads in flight
        const int4* src = reinterpret_cast<const int4*>(D.cl + cid * kCellCap);
        int* o = cand + incl - cnt;
        for (int k = 0; k < cnt; k += 8) {
            const int4 u = src[k >> 2], v = src[(k >> 2) + 1];
            const int e[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if (k + q < cnt) o[k + q] = e[q];
        }
    }
    __syncthreads();
    if (!valid) return;
    const int npass = (total + 63) >> 6;
    // where a lane has no candidate: every comparison of a distance is false
    const double kNaN = __longlong_as_double(0x7ff8000000000000ll);
    const double4 nowhere = make_double4(kNaN, kNaN, kNaN, 0.0);
    int jc[kCandReg];
    double4 rc[kCandReg];
#pragma unroll
    for (int q = 0; q < kCandReg; ++q) {
        int idx = q * 64 + lane;
        jc[q] = (q < npass && idx < total) ? cand[idx] : -1;
        rc[q] = jc[q] >= 0 ? D.r[jc[q]] : nowhere;
    }
    const int nc = D.cn[c];
    const int* own = D.cl + c * kCellCap;
    bool over = false;
    // the cell's own atoms (nc <= kCellCap <= 64): id and position one per
    // lane, loaded once, then read at the loop's uniform index, so no atom
    // waits for its own id and position before its distances
    const int oi = lane < nc ? own[lane] : 0;
    const double4 orv = lane < nc ? D.r[oi] : make_double4(0.0, 0.0, 0.0, 0.0);
    int nbuf = 0, first = 0;            // pairs in the buffer, their first own atom
    int my_off = 0, my_nn = 0, my_nm = 0;  // lane k: buffer offset and counts of own atom k
    for (int k = 0; k < nc; ++k) {
        const int i = __builtin_amdgcn_readlane(oi, k);
        const double3 ri = make_double3(readlane_f64(orv.x, k), readlane_f64(orv.y, k), readlane_f64(orv.z, k));
        int nn = 0, nm = 0;
        auto test = [&](int j, const double4& rj) {
            const double3 d = sub3(ri, d3(rj));
            double rsq = sq3(d);
            if (__builtin_expect(__ballot(rsq >= b.safe_sq) != 0, 0)) (void)min_image_sq(b, d, rsq);
            bool inmax = rsq < P.rcut_max_sq && j != i;
            bool inmag = rsq < P.rcut_mag_sq && inmax;
            const unsigned long long m1 = __ballot(inmax), m2 = __ballot(inmag);
            const int pos = nn + lanes_before(m1), pos2 = nm + lanes_before(m2);
            nn += __popcll(m1);
            nm += __popcll(m2);
            if (__builtin_expect(nn > kMaxNb || nm > kMaxMag, 0)) {
                inmax = inmax && pos < kMaxNb;
                inmag = inmag && pos2 < kMaxMag;
            }
            if (inmax) {
                pairs[nbuf + pos] = make_int2(j, k | (pos << 8) | (inmag ? (pos2 + 1) << 16 : 0));
                rsqs[nbuf + pos] = rsq;
            }
        };
#pragma unroll
        for (int q = 0; q < kCandReg; ++q) {
            if (q >= npass) break;
            test(jc[q], rc[q]);
        }
        // candidates past the registers (more than 64 x kCandReg)
        for (int q = kCandReg; q < npass; ++q) {
            const int idx = q * 64 + lane;
            const int j = idx < total ? cand[idx] : -1;
            test(j, j >= 0 ? D.r[j] : nowhere);
        }
        over |= nn > kMaxNb || nm > kMaxMag;
        nn = nn < kMaxNb ? nn : kMaxNb;
        nm = nm < kMaxMag ? nm : kMaxMag;
        if (lane == k) {
            my_off = nbuf;
            my_nn = nn;
            my_nm = nm;
        }
        nbuf += nn;
        if (nbuf <= kPairBuf - kMaxNb && k + 1 < nc) continue;
        // the buffered pairs, of own atoms first .. k
        wave_fence();
        for (int p0 = 0; p0 < nbuf; p0 += 64) {
            const int p = p0 + lane;
            const bool act = p < nbuf;
            const int2 e = pairs[act ? p : 0];
            const size_t a = (size_t)__shfl(oi, e.y & 255, 64);
            if (!act) continue;
            const double r = sqrt(rsqs[p]);
            int n0;
            double ratio;
            interp_index(r, T.in_over_rmax, n0, ratio);
            const double sf = lerp_at(T.sftab, n0, ratio);
            const int mag = e.y >> 16;
            D.nb[a * kMaxNb + ((e.y >> 8) & 255)] = e.x;
            if (mag) {
                D.nbm[a * kMaxMag + mag - 1] = e.x;
                D.nbJ[a * kMaxMag + mag - 1] = lerp_at(T.jtab, n0, ratio);
            }
            rsqs[p] = r < P.rcut_pot ? sf : 0.0;
        }
        wave_fence();
        // densities: eight lanes an atom
        for (int g = first; g <= k; g += 8) {
            const int q = g + (lane >> 3), l = lane & 7;
            const int qq = q <= k ? q : k;
            const int off = __shfl(my_off, qq, 64), n1 = __shfl(my_nn, qq, 64), n2 = __shfl(my_nm, qq, 64);
            const int a = __shfl(oi, qq, 64);
            double rho = 0.0;
            for (int p = l; p < n1; p += 8) rho += rsqs[off + p];
            rho += __shfl_xor(rho, 1, 8);
            rho += __shfl_xor(rho, 2, 8);
            rho += __shfl_xor(rho, 4, 8);
            if (q <= k && l == 0) {
                D.nbn[a] = n1;
                D.nbmn[a] = n2;
                if (write_rho) D.rho[a] = rho;
            }
        }
        wave_fence();
        nbuf = 0;
        first = k + 1;
    }
    if (over && lane == 0) atomicOr(D.err, kErrNbOverflow);
}

// ---------------------------------------------------------------------------
// force and energy (calculate_force_energy_CPU.cpp:33-301), full neighbour
// list: each atom sums its own pair terms; no atomics.

// dF/drho plus the Landau derivative terms of one atom
// (calculate_force_energy_CPU.cpp:98-107)
__global__ __launch_bounds__(256) void k_fp(Tables T, Dev D) {
    const int lb = xcd_block((D.N + blockDim.x - 1) / blockDim.x);
    if (lb < 0) return;
    int i = lb * blockDim.x + threadIdx.x;
    if (i >= D.N || D.arep[i] < 0) return;
    int n0;
    double ratio;
    interp_index(D.rho[i], T.in_over_rhomax, n0, ratio);
    double s2 = sq3(d3(D.s[i]));
    double dF = lerp_tab(T.rhotab, kRhoStride, H_DF, n0, ratio);
    double dA = lerp_tab(T.rhotab, kRhoStride, H_DA, n0, ratio);
    double dB = lerp_tab(T.rhotab, kRhoStride, H_DB, n0, ratio);
    double dC = lerp_tab(T.rhotab, kRhoStride, H_DC, n0, ratio);
    double dD = lerp_tab(T.rhotab, kRhoStride, H_DD, n0, ratio);
    double s4 = s2 * s2;
    D.r[i].w = dF + (dA * s2 + dB * s4 + dC * s4 * s2 + dD * s4 * s4);
}

// Four lanes an atom: lane j takes list entries j, j + 4, ..., and the sums of
// the four are added at the end. The lanes of a quad fetch each other's data
// together: two lanes load the halves of a pair's r with F'(rho) in r.w, two
// those of its s, and each a column of its table row, so that a load
// instruction touches 32 or 16 lines and not 64; the quad then swaps the pieces
// by register moves (the columns after the interpolation).
//
// What bounds it is the instruction stream, 2,044 a wave of 16 atoms, with three
// waves a SIMD (160 registers) to hide the rows' latency; 1.5 GB come from beyond
// the L2s. 2 M atoms 870 us, where a lane an atom, which loaded all of a pair by
// itself, ten lines, and had eight pairs in flight to hide it, took 1,283 and
// 3.8 GB; 64 x 16,000 atoms 640 (878), 250,000 atoms 108 (155), 2,000 13 (37).
// Tried at 2 M atoms against 893 us on the same clock: rows of 64 bytes with J in
// a table of its own 967, entries of 32 bytes that are not stored twice 1,000,
// loads straight to LDS instead of register moves 970, no loads ahead 1,021, 128
// registers with spills 1,840. |s_i| |s_j| is the root of the squares' product, as
// the one-body terms' squares: the rounded lengths' product (862 us) carries a
// common rounding of them into every pair's energy.
__global__ __launch_bounds__(256) void k_force(Tables T, Phys P, Dev D) {
    const int lb = xcd_block((4 * D.N + blockDim.x - 1) / blockDim.x);
    if (lb < 0) return;
    const int i = (lb * blockDim.x + threadIdx.x) >> 2, j = threadIdx.x & 3;
    if (i >= D.N) return;
    const int rr = D.arep[i];
    if (rr < 0) return;
    const Rep& R = D.rep[rr];
    const Box b = R.box;
    const double4 ri4 = D.r[i];
    const double3 ri = d3(ri4);
    const double3 si = d3(D.s[i]);
    const double si_sq = sq3(si);
    const double fpi = ri4.w;
    double3 f = make_double3(0.0, 0.0, 0.0);
    double pe = 0.0, me = 0.0, me0 = 0.0;
    double st0 = 0.0, st1 = 0.0, st2 = 0.0, st3 = 0.0, st4 = 0.0, st5 = 0.0;
    double m1 = 0.0, m2 = 0.0;  // localvol: sums of 1/r and 1/r^2 within rcut_vol
    const int nn = D.nbn[i];
    const int* nb = D.nb + (size_t)i * kMaxNb;
    // this lane's half of every pair's r or s, and its column of every row
    const double2* rec = reinterpret_cast<const double2*>(j < 2 ? D.r : D.s) + (j & 1);
    const double2* col = reinterpret_cast<const double2*>(T.prow) + j;
    static_assert(P_DSF == 0 && P_DPR == 2 && P_PR == 4 && P_DJ == 6, "the first columns, in the lanes' order");
    constexpr int kRow = kPRowStride / 2;
    double2 v[4];
    auto gather = [&](int id) {
        v[0] = rec[2 * (size_t)quad_from<0>(id)];
        v[1] = rec[2 * (size_t)quad_from<1>(id)];
        v[2] = rec[2 * (size_t)quad_from<2>(id)];
        v[3] = rec[2 * (size_t)quad_from<3>(id)];
    };
    // past the list: a valid atom, never added
    auto entry = [&](int k) { return k < nn ? nb[k] : i; };
    gather(entry(j));
    int next = entry(j + 4);
    for (int k0 = 0; k0 < nn; k0 += 4) {
        double x[4] = {v[0].x, v[1].x, v[2].x, v[3].x}, y[4] = {v[0].y, v[1].y, v[2].y, v[3].y};
        quad_transpose(x, j);
        quad_transpose(y, j);
        const double3 sj = make_double3(x[2], y[2], x[3]);
        const double fpj = y[1];
        double rsq, inv, ratio;
        int n0;
        const double3 rij = min_image_sq(b, sub3(ri, make_double3(x[0], y[0], x[1])), rsq);
        const double r = sqrt_rsqrt(rsq, inv);
        interp_index(r, T.in_over_rmax, n0, ratio);
        double2 q[4];
        q[0] = col[(size_t)quad_from<0>(n0) * kRow];
        q[1] = col[(size_t)quad_from<1>(n0) * kRow];
        q[2] = col[(size_t)quad_from<2>(n0) * kRow];
        q[3] = col[(size_t)quad_from<3>(n0) * kRow];
        const bool in = k0 + j < nn, mag = in && r < P.rcut_mag;
        double2 qJ = make_double2(0.0, 0.0);
        if (mag) qJ = *reinterpret_cast<const double2*>(T.prow + (size_t)n0 * kPRowStride + P_J);
        // the next pairs' loads go out before this one's rows are waited for
        gather(next);
        next = entry(k0 + 8 + j);
        double c[4];
        auto lerp = [&](double2 t, double rt) { return t.x * rt + t.y * (1.0 - rt); };
        c[0] = lerp(q[0], quad_from<0>(ratio));
        c[1] = lerp(q[1], quad_from<1>(ratio));
        c[2] = lerp(q[2], quad_from<2>(ratio));
        c[3] = lerp(q[3], quad_from<3>(ratio));
        quad_transpose(c, j);
        if (!in) continue;
        double dudr = 0.0;
        if (r < P.rcut_pot) {
            dudr = (fpi + fpj) * c[0] + c[1];
            pe += 0.5 * c[2];
        }
        if (mag) {
            const double sdot = dot3(si, sj), stimes = sqrt_any(si_sq * sq3(sj));
            const double Jh = lerp(qJ, ratio) / 2.0;
            dudr += -c[3] * (sdot - stimes);
            me0 += Jh * stimes;
            me += -Jh * sdot;
        }
        const double force = -dudr * inv;
        const double3 fij = mul3(force, rij);
        f = add3(f, fij);
        st0 += fij.x * rij.x; st1 += fij.y * rij.y; st2 += fij.z * rij.z;
        st3 += fij.x * rij.y; st4 += fij.y * rij.z; st5 += fij.z * rij.x;
        if (P.localvol && r < P.rcut_vol) {  // calculate_force_energy_CPU.cpp:80-90
            m1 += inv;
            m2 += inv * inv;
        }
    }
    f = make_double3(quad_sum(f.x), quad_sum(f.y), quad_sum(f.z));
    pe = quad_sum(pe);
    me = quad_sum(me);
    me0 = quad_sum(me0);
    st0 = quad_sum(st0); st1 = quad_sum(st1); st2 = quad_sum(st2);
    st3 = quad_sum(st3); st4 = quad_sum(st4); st5 = quad_sum(st5);
    if (P.localvol) {
        m1 = quad_sum(m1);
        m2 = quad_sum(m2);
    }
    // one-body terms (calculate_force_energy_CPU.cpp:196-215)
    int n0;
    double ratio;
    interp_index(D.rho[i], T.in_over_rhomax, n0, ratio);
    double F = lerp_tab(T.rhotab, kRhoStride, H_F, n0, ratio);
    const double4 lan = D.lan[i];
    const double A = lan.x, B = lan.y, C = lan.z, Dd = lan.w;
    double s4 = si_sq * si_sq;
    pe += F;
    if (P.extfield) me -= dot3(si, d3(D.hext[i]));  // calculate_force_energy_CPU.cpp:199-201
    me += A * si_sq + B * s4 + C * s4 * si_sq + Dd * s4 * s4;
    const double m = P.atmass;
    const double4 p = D.p[i];
    const size_t N = D.N;
    if (j == 0) {
        D.f[i] = make_double4(f.x, f.y, f.z, 0.0);
        D.pe[i] = pe;
        D.me[i] = me;
        D.me0[i] = me0;
    }
    // the reference books -force*r^2 once per pair on the half-shell owner;
    // here each atom keeps half of each of its pairs (same total virial)
    if (j == 1) D.vir[i] = -0.5 * (st0 + st1 + st2);
    // per-atom stress with the kinetic part (calculate_force_energy_CPU.cpp:283-293);
    // with localvol the local volume (:270-276) is normalised over the
    // replica first, so the numerators are stored and k_lvol_apply divides
    const double num[6] = {p.x * p.x / m + st0 / 2.0,   p.y * p.y / m + st1 / 2.0,   p.z * p.z / m + st2 / 2.0,
                           (p.x * p.y) / m + st3 / 2.0, (p.y * p.z) / m + st4 / 2.0, (p.z * p.x) / m + st5 / 2.0};
    double lv = 1.0;
    if (P.localvol) {
        const double local_radius = 0.5 * m1 / m2;
        if (j == 0) D.lvol[i] = 4.0 * kPi / 3.0 * pow(local_radius, 3.0);
    } else {
        lv = R.box_volume / R.natom;
    }
#pragma unroll
    for (int k = 0; k < 6; ++k)
        if (j == (k & 3)) D.stress[k * N + i] = num[k] / lv;
}

// localvol: each replica's sum of the local volumes, one partial per 256
// atom slots (calculate_force_energy_CPU.cpp:270-275)
__global__ __launch_bounds__(256) void k_lvol_sum(Dev D, double* partials) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    double acc[1] = {0.0};
    if (a < D.N && D.arep[a] >= 0) acc[0] = D.lvol[a];
    block_partials<1>(acc, partials);
}

// localvol: the volumes scaled to fill the box, then each atom's stress over
// its volume (calculate_force_energy_CPU.cpp:279-293)
__global__ __launch_bounds__(256) void k_lvol_apply(Dev D, const double* scal) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= D.N) return;
    const int rr = D.arep[a];
    if (rr < 0) return;
    const double volume_factor = D.rep[rr].box_volume / scal[(size_t)rr * kScal + kScalLvol];
    const double lv = D.lvol[a] * volume_factor;
    D.lvol[a] = lv;
    const size_t N = D.N;
#pragma unroll
    for (int k = 0; k < 6; ++k) D.stress[k * N + a] = D.stress[k * N + a] / lv;
}

// ---------------------------------------------------------------------------
// spins (calculate_spin_CPU.cpp:33-199, core_ds_CPU.cpp:35-127)

// Exchange field H = Hext + sum J s_j (Hext with extfield, else 0:
// calculate_spin_CPU.cpp:35-39) and S = sum J |s_j| over the rcut_mag list,
// gathered eight neighbours at a time with all loads of a batch in flight.
__device__ __forceinline__ void exchange_field(int a, const Dev& D, const Phys& P, double3& H, double& S) {
    const int nm = D.nbmn[a];
    const int* ids = D.nbm + (size_t)a * kMaxMag;
    const double* js = D.nbJ + (size_t)a * kMaxMag;
    double hx = 0.0, hy = 0.0, hz = 0.0, ss = 0.0;
    if (P.extfield) {
        const double4 he = D.hext[a];
        hx = he.x; hy = he.y; hz = he.z;
    }
#pragma unroll 1
    for (int b0 = 0; b0 < nm; b0 += 8) {
        const int4 i0 = *reinterpret_cast<const int4*>(ids + b0);
        const int4 i1 = *reinterpret_cast<const int4*>(ids + b0 + 4);
        const int id[8] = {i0.x, i0.y, i0.z, i0.w, i1.x, i1.y, i1.z, i1.w};
        double J[8];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            double2 v = *reinterpret_cast<const double2*>(js + b0 + 2 * q);
            J[2 * q] = v.x; J[2 * q + 1] = v.y;
        }
        double4 sj[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) sj[q] = D.s[b0 + q < nm ? id[q] : a];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            double Jq = b0 + q < nm ? J[q] : 0.0;
            hx += Jq * sj[q].x; hy += Jq * sj[q].y; hz += Jq * sj[q].z;
            ss += Jq * sj[q].w;
        }
    }
    H = make_double3(hx, hy, hz);
    S = ss;
}

// The Langevin normals of one spin pass for every atom (the counter-based
// stream of normal3, keyed by replica seed and stream id, counted by the
// atom's index in its replica and the pass). The pass number is the device
// counter plus an offset fixed by the pass's place in the step, so that the
// launches of a step are the same in every step.
__global__ __launch_bounds__(256) void k_spin_noise(Dev D, int pass_off) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= D.N) return;
    const int rr = D.arep[i];
    if (rr < 0) return;
    const Rep& R = D.rep[rr];
    const uint64_t pass = D.pass_base[0] + (uint64_t)pass_off;
    const double3 z = normal3(R.seed, R.replica, i - R.atom0, pass);
    D.zn[i] = make_double4(z.x, z.y, z.z, 0.0);
}

// advances the device noise-pass counter by the passes a step consumed
__global__ void k_pass_advance(Dev D, int n) {
    if (blockIdx.x == 0 && threadIdx.x == 0) D.pass_base[0] += (uint64_t)n;
}

// Landau coefficients A..D of an atom: interpolation weights of its density,
// then the two table rows (calculate_spin_CPU.cpp:118-121)
struct LanRows {
    double4 lo, hi;
    double ratio;
};

__device__ __forceinline__ LanRows landau_rows(const Tables& T, double rho) {
    int n0;
    double ratio;
    interp_index(rho, T.in_over_rhomax, n0, ratio);
    // rows of 80 bytes: columns A..D are 16-byte aligned, in one line or two
    static_assert(kRhoStride % 2 == 0 && H_A % 2 == 0, "double2 loads");
    const double2* lo = reinterpret_cast<const double2*>(T.rhotab + (size_t)(n0 - 1) * kRhoStride + H_A);
    const double2* hi = reinterpret_cast<const double2*>(T.rhotab + (size_t)n0 * kRhoStride + H_A);
    const double2 l0 = lo[0], l1 = lo[1], h0 = hi[0], h1 = hi[1];
    LanRows L;
    L.lo = make_double4(l0.x, l0.y, l1.x, l1.y);
    L.hi = make_double4(h0.x, h0.y, h1.x, h1.y);
    L.ratio = ratio;
    return L;
}

// The Landau coefficients A..D of every atom at its current density
// (calculate_spin_CPU.cpp:118-121), interpolated as the reference does. The
// density changes once a step (calculate_rho); the four spin sweeps, the
// force pass and the temperature and energy observables in between read the
// coefficients from here, 32 contiguous bytes per atom, instead of two table
// rows of 80 bytes each.
__global__ __launch_bounds__(256) void k_landau(Tables T, Dev D) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= D.N || D.arep[i] < 0) return;
    const LanRows L = landau_rows(T, D.rho[i]);
    const double w = L.ratio, v = 1.0 - L.ratio;
    D.lan[i] = make_double4(L.lo.x * w + L.hi.x * v, L.lo.y * w + L.hi.y * v, L.lo.z * w + L.hi.z * v,
                            L.lo.w * w + L.hi.w * v);
}

// ---------------------------------------------------------------------------
// momenta (core_dp_CPU.cpp:51-312). Every part of the Langevin update is local
// to one link cell, so one group of kSeg lanes runs C1, B, A, B, C2 for its
// cell in order. Lane l of a group holds the cell's list entries l, l + kSeg,
// ... (kSegSlots slots; bcc Fe has about six atoms per cell, so most lanes
// hold one): eight cells per wavefront.

constexpr int kSegSlots = kCellCap / kSeg;
static_assert(kCellCap % kSeg == 0, "a cell's list fills whole slots");

// sum over a cell: each lane's slots in order, then a butterfly over the group
__device__ __forceinline__ double seg_sum(const double (&v)[kSegSlots]) {
    double t = v[0];
#pragma unroll
    for (int s = 1; s < kSegSlots; ++s) t += v[s];
#pragma unroll
    for (int m = kSeg / 2; m > 0; m >>= 1) t += __shfl_xor(t, m, kSeg);
    return t;
}

__device__ __forceinline__ double3 seg_sum(const double3 (&v)[kSegSlots]) {
    double x[kSegSlots], y[kSegSlots], z[kSegSlots];
#pragma unroll
    for (int s = 0; s < kSegSlots; ++s) {
        x[s] = v[s].x; y[s] = v[s].y; z[s] = v[s].z;
    }
    return make_double3(seg_sum(x), seg_sum(y), seg_sum(z));
}

// Local collective motion step: walking the list (head to tail, or tail to
// head), each atom gets p += g dt/n (sum_p - p) with sum_p over the cell's
// current momenta (core_dp_CPU.cpp:211-264). The cell sum is carried along:
// after atom k changes by d, the sum changes by d (the reference re-adds the
// list each time; same value up to rounding).
__device__ __forceinline__ void dp_colmot(double3 (&p)[kSegSlots], int l, int n, double factor, bool backward) {
    double3 sp = seg_sum(p);
    const int base = (threadIdx.x & 63) & ~(kSeg - 1);
    for (int q = 0; q < n; ++q) {
        const int k = backward ? n - 1 - q : q;
        const int kl = k % kSeg, ks = k / kSeg;
        double3 d = make_double3(0.0, 0.0, 0.0);
#pragma unroll
        for (int s = 0; s < kSegSlots; ++s) {
            if (l == kl && s == ks) {
                const double3 pn = add3(p[s], mul3(factor, sub3(sp, p[s])));
                d = sub3(pn, p[s]);
                p[s] = pn;
            }
        }
        const int src = base + kl;
        d.x = __shfl(d.x, src, 64);
        d.y = __shfl(d.y, src, 64);
        d.z = __shfl(d.z, src, 64);
        sp = add3(sp, d);
    }
}

// the force of the momentum update: with extforce the reference adds fext to
// the stored force in place first (core_dp_CPU.cpp:69-71,130-132), so a
// second core_dp before the next force evaluation adds it again
__device__ __forceinline__ double3 dp_force(const Phys& P, const Dev& D, int a) {
    double3 f = d3(D.f[a]);
    if (P.extforce) {
        f = add3(f, d3(D.fext[a]));
        D.f[a] = make_double4(f.x, f.y, f.z, 0.0);
    }
    return f;
}

// ---------------------------------------------------------------------------
// quantum thermostat (quantum_noise_CPU.cpp). History element e of an atom's
// three degrees of freedom is normal3 at pass kQnCall0 + e, a range that no
// lattice or spin pass reaches; element e lives in ring slot e % 2Nf.
constexpr uint64_t kQnCall0 = 1ull << 62;

// initial_quantum_noise (:115-119): elements 0 .. 2Nf-1, one thread per atom
__global__ __launch_bounds__(256) void k_qn_init(Phys P, Dev D) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= D.N || D.arep[a] < 0) return;
    const Rep& R = D.rep[D.arep[a]];
    const size_t stride = 3 * (size_t)D.N;
    for (int j = 0; j < P.qnf2; ++j) {
        const double3 z = normal3(R.seed, R.replica, a - R.atom0, kQnCall0 + (uint64_t)j);
        double* m = D.qring + (size_t)j * stride + 3 * (size_t)a;
        m[0] = z.x;
        m[1] = z.y;
        m[2] = z.z;
    }
}

// quantum_noise (:60-81) for the r-th redraw of every degree of freedom at
// once: the noise is sum_i H[i] * element (r + 2Nf - 1 - i), newest first;
// element 2Nf + r then replaces element r, the oldest, in its slot. Each
// lane reads its atom's three doubles of a slot, so a wave reads 1.5 KB
// contiguous per tap.
__global__ __launch_bounds__(256) void k_qn_refresh(Phys P, Dev D, uint64_t r) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= D.N || D.arep[a] < 0) return;
    const int rr = D.arep[a];
    const Rep& R = D.rep[rr];
    const int nf2 = P.qnf2;
    const double* H = D.qH + (size_t)rr * nf2;
    const size_t stride = 3 * (size_t)D.N;
    const double* base = D.qring + 3 * (size_t)a;
    int slot = (int)((r + (uint64_t)nf2 - 1) % (uint64_t)nf2);
    double n0 = 0.0, n1 = 0.0, n2 = 0.0;
    for (int i = 0; i < nf2; ++i) {
        const double* m = base + (size_t)slot * stride;
        const double h = H[i];
        n0 += h * m[0];
        n1 += h * m[1];
        n2 += h * m[2];
        slot = slot == 0 ? nf2 - 1 : slot - 1;
    }
    const double3 z = normal3(R.seed, R.replica, a - R.atom0, kQnCall0 + (uint64_t)nf2 + r);
    double* m = D.qring + (size_t)(r % (uint64_t)nf2) * stride + 3 * (size_t)a;
    m[0] = z.x;
    m[1] = z.y;
    m[2] = z.z;
    double* q = D.qval + 3 * (size_t)a;
    q[0] = n0;
    q[1] = n1;
    q[2] = n2;
}

// One group of kSeg lanes per link cell, eight cells per 64-thread block (a
// replica's cells start on an 8-cell boundary, so each block's partial sums
// belong to one replica).
__global__ __launch_bounds__(64) void k_dp_cells(double dt, Phys P, Dev D, int pass_off, double* partials) {
    const int l = threadIdx.x & (kSeg - 1);
    const int c = (blockIdx.x * blockDim.x + threadIdx.x) / kSeg;
    const int rr = c < D.C ? D.crep[c] : -1;
    const bool valid = rr >= 0;
    const int n = valid ? D.cn[c] : 0;
    bool has[kSegSlots];
    int a[kSegSlots];
    double3 p[kSegSlots];
#pragma unroll
    for (int s = 0; s < kSegSlots; ++s) {
        has[s] = l + kSeg * s < n;
        a[s] = has[s] ? D.cl[c * kCellCap + l + kSeg * s] : 0;
        p[s] = has[s] ? d3(D.p[a[s]]) : make_double3(0.0, 0.0, 0.0);
    }
    if (valid) {
        const double gm = P.gamma_L / P.atmass;
        if (P.lattlang) {
            const double h = dt / 2.0;
            if (P.localcolmot && n > 0) dp_colmot(p, l, n, gm * h / n, false);
            const double eb = P.localcolmot ? exp(-gm * h * (1.0 - 1.0 / n)) : exp(-gm * h);
#pragma unroll
            for (int s = 0; s < kSegSlots; ++s) p[s] = mul3(eb, p[s]);
            const Rep& R = D.rep[rr];
            const double Tk = P.eltemp ? D.Te[c] : R.temperature;
            double3 ff[kSegSlots];
#pragma unroll
            for (int s = 0; s < kSegSlots; ++s) {
                ff[s] = make_double3(0.0, 0.0, 0.0);
                if (has[s]) {
                    if (P.quantumnoise) {
                        // core_dp_CPU.cpp:137-146: coloured noise scaled by sqrt(2 gamma / h), h = M dt
                        const double hq = dt * P.qm;
                        const double len = sqrt(2.0 * P.gamma_L / hq);
                        const double* q = D.qval + 3 * (size_t)a[s];
                        ff[s] = mul3(len, make_double3(q[0], q[1], q[2]));
                    } else {
                        const double len = sqrt(2.0 * Tk * P.gamma_L / dt);
                        const uint64_t pass = D.pass_base[0] + (uint64_t)pass_off;
                        ff[s] = mul3(len, normal3(R.seed, R.replica, a[s] - R.atom0, pass));
                    }
                    p[s] = add3(p[s], mul3(dt, add3(dp_force(P, D, a[s]), ff[s])));
                }
            }
            if (P.localcolmot && n > 0) {
                const double3 fs = seg_sum(ff);
                const double3 ave = make_double3(fs.x / n, fs.y / n, fs.z / n);
#pragma unroll
                for (int s = 0; s < kSegSlots; ++s)
                    if (has[s]) p[s] = sub3(p[s], mul3(dt, ave));
            }
#pragma unroll
            for (int s = 0; s < kSegSlots; ++s) p[s] = mul3(eb, p[s]);
            if (P.localcolmot && n > 0) dp_colmot(p, l, n, gm * h / n, true);
        } else {
#pragma unroll
            for (int s = 0; s < kSegSlots; ++s)
                if (has[s]) p[s] = add3(p[s], mul3(dt, dp_force(P, D, a[s])));
        }
#pragma unroll
        for (int s = 0; s < kSegSlots; ++s)
            if (has[s]) D.p[a[s]] = make_double4(p[s].x, p[s].y, p[s].z, 0.0);
    }
    double acc[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < kSegSlots; ++s) {
        if (has[s]) {
            acc[0] += p[s].x;
            acc[1] += p[s].y;
            acc[2] += p[s].z;
        }
    }
    block_partials<3>(acc, partials);
}

// The NK sums of the block's replica (a block of 256 slots holds one replica's
// atoms, the first slot one of them): scal[0..NK) of its scalar block, or, given
// seg, the sum of the rows seg[rr]..seg[rr + 1) of the nrow partial sums, at most
// kFewRows, by every block for itself and to the bit what k_reduce_seg makes of
// them. In replicas of 2,000 atoms that spares a step four launches of 4 us.
template <int NK>
__device__ __forceinline__ void replica_sums(const Dev& D, const double* scal, const double* in, const int* seg,
                                             int nrow, double (&out)[NK]) {
    const int rr = D.arep[(size_t)blockIdx.x * blockDim.x];
#pragma unroll
    for (int k = 0; k < NK; ++k) out[k] = 0.0;
    if (rr < 0) return;
    if (!seg) {
#pragma unroll
        for (int k = 0; k < NK; ++k) out[k] = scal[(size_t)rr * kScal + k];
        return;
    }
    __shared__ double sh[kFewRows / 64][NK];
    const int t = threadIdx.x, end = seg[rr + 1];
#pragma unroll
    for (int u = 0; u < kFewRows; u += 256) {
        const int b = seg[rr] + u + t;
#pragma unroll
        for (int k = 0; k < NK; ++k) {
            const double v = wave_sum(b < end ? in[(size_t)k * nrow + b] : 0.0);
            if ((t & 63) == 0) sh[(u + t) >> 6][k] = v;
        }
    }
    __syncthreads();
    for (int w = 0; w < kFewRows / 64; ++w)
#pragma unroll
        for (int k = 0; k < NK; ++k) out[k] += sh[w][k];
}

// rescale_momentum, part 1: remove the mean momentum (core_dp_CPU.cpp:270-302)
__global__ __launch_bounds__(256) void k_dp_center(Phys P, Dev D, const double* scal, const double* in,
                                                   const int* seg, int nrow, double* partials) {
    double psum[3];  // the replica's momentum
    replica_sums(D, scal, in, seg, nrow, psum);
    int a = blockIdx.x * blockDim.x + threadIdx.x;
    double acc[2] = {0.0, 0.0};
    const int rr = a < D.N ? D.arep[a] : -1;
    if (rr >= 0) {
        const double inv_n = 1.0 / D.rep[rr].natom;
        double3 mean = make_double3(psum[0] * inv_n, psum[1] * inv_n, psum[2] * inv_n);
        double3 p = d3(D.p[a]);
        acc[0] = sq3(p) / 2.0 / P.atmass;
        p = sub3(p, mean);
        acc[1] = sq3(p) / 2.0 / P.atmass;
        D.p[a] = make_double4(p.x, p.y, p.z, 0.0);
    }
    block_partials<2>(acc, partials);
}

// rescale_momentum, part 2, and the kinetic energies (core_dp_CPU.cpp:78-84,304-310)
__global__ __launch_bounds__(256) void k_dp_scale(Phys P, Dev D, const double* scal, const double* in, const int* seg,
                                                  int nrow) {
    double ke2[2];  // the replica's kinetic energies before and after centring
    replica_sums(D, scal, in, seg, nrow, ke2);
    int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= D.N) return;
    const int rr = D.arep[a];
    if (rr < 0) return;
    double factor = sqrt(ke2[0] / ke2[1]);
    if (ke2[1] < 1e-10) factor = 1.0;
    double3 p = mul3(factor, d3(D.p[a]));
    D.p[a] = make_double4(p.x, p.y, p.z, 0.0);
    D.ke[a] = sq3(p) / 2.0 / P.atmass;
}

// core_dr_CPU.cpp:33-44
__global__ __launch_bounds__(256) void k_dr(double dt, Phys P, Dev D) {
    int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= D.N) return;
    const int rr = D.arep[a];
    if (rr < 0) return;
    double k = dt / P.atmass;
    double3 r = add3(d3(D.r[a]), mul3(k, d3(D.p[a])));
    r = wrap(D.rep[rr].box, r);
    D.r[a] = make_double4(r.x, r.y, r.z, 0.0);
}

// ---------------------------------------------------------------------------
// electron subsystem

// calculate_temperature_CPU.cpp:35-148: one group of kSeg lanes per link
// cell, lane l taking the cell's list entries l, l + kSeg, ...; the cell sums
// are each lane's entries in order, then a butterfly over the group.
__device__ __forceinline__ double seg_reduce(double t) {
#pragma unroll
    for (int m = kSeg / 2; m > 0; m >>= 1) t += __shfl_xor(t, m, kSeg);
    return t;
}

__global__ __launch_bounds__(256) void k_temperature(Tables T, Phys P, Dev D) {
    const int l = threadIdx.x & (kSeg - 1);
    const int lb = xcd_block((D.C * kSeg + blockDim.x - 1) / blockDim.x);
    if (lb < 0) return;
    const int c = (lb * blockDim.x + threadIdx.x) / kSeg;
    if (c >= D.C || D.crep[c] < 0) return;
    const int n = D.cn[c];
    double ke = 0.0, rup = 0.0, rdn = 0.0, lup = 0.0, ldn = 0.0, px = 0.0, py = 0.0, pz = 0.0;
    for (int k = l; k < n; k += kSeg) {
        const int a = D.cl[c * kCellCap + k];
        ke += D.ke[a];
        const double3 pa = d3(D.p[a]);
        px += pa.x; py += pa.y; pz += pa.z;
        double3 H;
        double S;
        exchange_field(a, D, P, H, S);
        double3 s = d3(D.s[a]);
        rup += sq3(cross3(s, H));
        rdn += dot3(s, H);
        const double4 lan = D.lan[a];
        const double A = lan.x, B = lan.y, C = lan.z, Dd = lan.w;
        double s2 = sq3(s), s4 = s2 * s2;
        double s0 = sqrt(s2);
        double kk = -(2.0 * A + 4.0 * B * s2 + 6.0 * C * s4 + 8.0 * Dd * s4 * s2);
        double hc = -S / s0;
        double3 L = make_double3((kk + hc) * s.x, (kk + hc) * s.y, (kk + hc) * s.z);
        lup += sq3(add3(H, L));
        ldn += 6.0 * A + 20.0 * B * s2 + 42.0 * C * s4 + 72.0 * Dd * s4 * s2 + 2.0 * S / s0;
        // s0 stays local: the reference stores it (calculate_temperature_CPU.cpp:100),
        // but here .w is read by the other cells' lanes of this launch through
        // exchange_field, so writing it would race with those reads. The spin
        // sweep and the uploads already keep .w = spin_len(s).
        D.hh[a] = make_double4(H.x, H.y, H.z, 0.0);
        D.hl[a] = make_double4(L.x, L.y, L.z, 0.0);
        D.sjs[a] = S;
    }
    double sum_ke = seg_reduce(ke);
    double3 ap = make_double3(seg_reduce(px), seg_reduce(py), seg_reduce(pz));
    rup = seg_reduce(rup);
    rdn = seg_reduce(rdn);
    lup = seg_reduce(lup);
    ldn = seg_reduce(ldn);
    if (l != 0) return;
    const Rep& R = D.rep[D.crep[c]];
    const double apc = (double)R.natom / (double)R.ncell;
    const double gm = P.gamma_L / P.atmass;
    if (P.localcolmot) {
        ap = make_double3(ap.x / n, ap.y / n, ap.z / n);
        sum_ke -= n * sq3(ap) / 2.0 / P.atmass;
        D.Tl[c] = 2.0 / 3.0 * sum_ke / (n - 1.0) / kBoltz;
        D.Gel[c] = 3.0 * (n - 1.0) * kBoltz * gm / apc;
        D.cellv[c] = make_double4(ap.x, ap.y, ap.z, 0.0);
    } else {
        D.Tl[c] = sum_ke * 2.0 / 3.0 / n / kBoltz;
        D.Gel[c] = 3.0 * n * kBoltz * gm / apc;
    }
    D.TsR[c] = rup / rdn / 2.0 / kBoltz;
    D.TsL[c] = lup / ldn / kBoltz;
    D.Ges[c] = kBoltz * P.gamma_S * ldn / apc;
    D.sRup[c] = rup; D.sRdn[c] = rdn; D.sLup[c] = lup; D.sLdn[c] = ldn;
}

// ---------------------------------------------------------------------------
// barostats: positions follow the box (scale_pressure_CPU.cpp:59,
// scale_stress_CPU.cpp:67-80)

// PRESSURE: r = factor r
__global__ __launch_bounds__(256) void k_scale_r(Dev D, double factor) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= D.N || D.arep[a] < 0) return;
    const double4 r = D.r[a];
    D.r[a] = make_double4(factor * r.x, factor * r.y, factor * r.z, r.w);
}

// STRESS: fractional coordinates of the old box, real ones of the new box
__global__ __launch_bounds__(256) void k_rebox_r(Dev D, Box old_box, Box new_box) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= D.N || D.arep[a] < 0) return;
    const double4 r = D.r[a];
    const double* iv = old_box.inv;
    const double* d = new_box.d;
    const double qx = iv[0] * r.x + iv[1] * r.y + iv[3] * r.z;
    const double qy = iv[2] * r.y + iv[4] * r.z;
    const double qz = iv[5] * r.z;
    D.r[a] = make_double4(d[0] * qx + d[1] * qy + d[3] * qz, d[2] * qy + d[4] * qz, d[5] * qz, r.w);
}

// ---------------------------------------------------------------------------
// scale_step (scale_step_CPU.cpp:35-70): the largest |p|^2 and |Heff_H|^2

__global__ __launch_bounds__(256) void k_step_max(Dev D, double* partials) {
    __shared__ double sh[2][256];
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    const int t = threadIdx.x;
    double pm = 0.0, hm = 0.0;
    if (a < D.N && D.arep[a] >= 0) {
        pm = sq3(d3(D.p[a]));
        hm = sq3(d3(D.hh[a]));
    }
    sh[0][t] = pm;
    sh[1][t] = hm;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if (t < s) {
            sh[0][t] = fmax(sh[0][t], sh[0][t + s]);
            sh[1][t] = fmax(sh[1][t], sh[1][t + s]);
        }
        __syncthreads();
    }
    if (t == 0) {
        partials[2 * blockIdx.x] = sh[0][0];
        partials[2 * blockIdx.x + 1] = sh[1][0];
    }
}

// out[0..1] = the largest of the pair partials (exact in any order)
__global__ __launch_bounds__(256) void k_reduce_max2(const double* partials, int nblk, double* out) {
    __shared__ double sh[2][256];
    const int t = threadIdx.x;
    double a = 0.0, b = 0.0;
    for (int k = t; k < nblk; k += 256) {
        a = fmax(a, partials[2 * k]);
        b = fmax(b, partials[2 * k + 1]);
    }
    sh[0][t] = a;
    sh[1][t] = b;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (t < s) {
            sh[0][t] = fmax(sh[0][t], sh[0][t + s]);
            sh[1][t] = fmax(sh[1][t], sh[1][t + s]);
        }
        __syncthreads();
    }
    if (t == 0) {
        out[0] = sh[0][0];
        out[1] = sh[1][0];
    }
}

// ---------------------------------------------------------------------------
// observables (check_energy_CPU.cpp, check_temperature_CPU.cpp, check_spin_CPU.cpp)

__global__ __launch_bounds__(256) void k_obs_atoms(Tables T, Phys P, Dev D, double* partials,
                                                   int scan_spin) {
    int a = blockIdx.x * blockDim.x + threadIdx.x;
    double acc[kObsAtomK + 1];
#pragma unroll
    for (int k = 0; k <= kObsAtomK; ++k) acc[k] = 0.0;
    if (a < D.N && D.arep[a] >= 0) {
        acc[0] = D.pe[a];
        acc[1] = D.ke[a];
        acc[2] = D.me[a];
        acc[3] = D.me0[a];
        double3 s = d3(D.s[a]);
        acc[4] = s.x; acc[5] = s.y; acc[6] = s.z;
        acc[11] = D.vir[a];
#pragma unroll
        for (int k = 0; k < 6; ++k) acc[12 + k] = D.stress[(size_t)k * D.N + a];
        if (scan_spin) {
            // check_temperature_CPU.cpp:64-77,97-128 (no eltemp)
            double3 H;
            double S;
            exchange_field(a, D, P, H, S);
            acc[7] = sq3(cross3(s, H));
            acc[8] = dot3(s, H);
            const double4 lan = D.lan[a];
            const double A = lan.x, B = lan.y, C = lan.z, Dd = lan.w;
            double s2 = sq3(s), s4 = s2 * s2;
            double s0 = sqrt(s2);
            double k = -(2.0 * A + 4.0 * B * s2 + 6.0 * C * s4 + 8.0 * Dd * s4 * s2);
            double hc = -S / s0;
            double3 L = make_double3((k + hc) * s.x, (k + hc) * s.y, (k + hc) * s.z);
            acc[9] = sq3(add3(H, L));
            acc[10] = 2.0 * S / s0 + (6.0 * A + 20.0 * B * s2 + 42.0 * C * s4 + 72.0 * Dd * s4 * s2);
            D.hh[a] = make_double4(H.x, H.y, H.z, 0.0);
            D.hl[a] = make_double4(L.x, L.y, L.z, 0.0);
            D.sjs[a] = S;
        }
    }
    block_partials<kObsAtomK + 1>(acc, partials);
}

__global__ __launch_bounds__(256) void k_obs_cells(Dev D, double* partials) {
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    double acc[kObsCellK] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (c < D.C) {
        double ee = te_to_ee(D.Te[c]);
        D.Ee[c] = ee;
        acc[0] = ee;
        acc[1] = D.sRup[c]; acc[2] = D.sRdn[c]; acc[3] = D.sLup[c]; acc[4] = D.sLdn[c];
        acc[5] = D.Te[c];
    }
    block_partials<kObsCellK>(acc, partials);
}

// renormalizeEnergy feedback (check_energy_CPU.cpp:103-110); the printed mean
// Te is taken afterwards (check_temperature_CPU.cpp:130-134), so the new
// temperatures are summed here.
__global__ __launch_bounds__(256) void k_renorm(Dev D, const double* err, double* partials) {
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    double acc[1] = {0.0};
    if (c < D.C) {
        double ee = D.Ee[c] - err[0];
        D.Ee[c] = ee;
        double te = ee_to_te(ee);
        D.Te[c] = te;
        acc[0] = te;
    }
    block_partials<1>(acc, partials);
}

// Ee = E(Te) of cells [c0, c0 + n) (map_cells.cpp:128-159)
__global__ __launch_bounds__(256) void k_ee_of_te(Dev D, int c0, int n) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) D.Ee[c0 + k] = te_to_ee(D.Te[c0 + k]);
}

// One run of a piece per blockIdx.y, one thread per element. The buffer is
// pinned host memory: a vector's three doubles are written through LDS as
// contiguous lines (a block's 6 KB), so the bus sees whole bursts.
__global__ __launch_bounds__(256) void k_pack(XferArgs A, int N, double* buf) {
    __shared__ double sh[6 * 256];
    const XferSeg& g = A.seg[blockIdx.y];
    const int t = threadIdx.x;
    const size_t e0 = (size_t)blockIdx.x * 256;
    if (e0 >= g.n) return;
    const int m = (int)(g.n - e0 < 256 ? g.n - e0 : 256);
    const size_t i = g.first + e0 + t;
    const int w = g.kind == kXferVec ? 3 : g.kind == kXferStress ? 6 : 1;
    if (t < m) {
        if (g.kind == kXferVec) {
            const double4 v = static_cast<const double4*>(g.dev)[i];
            sh[3 * t] = v.x; sh[3 * t + 1] = v.y; sh[3 * t + 2] = v.z;
        } else if (g.kind == kXferStress) {
            const double* d = static_cast<const double*>(g.dev);
            for (int k = 0; k < 6; ++k) sh[6 * t + k] = d[(size_t)k * N + i];
        } else {
            sh[t] = static_cast<const double*>(g.dev)[i];
        }
    }
    __syncthreads();
    double* out = buf + g.offset + e0 * w;
    for (int k = t; k < m * w; k += 256) out[k] = sh[k];
}

__global__ __launch_bounds__(256) void k_unpack(XferArgs A, int N, const double* buf) {
    __shared__ double sh[6 * 256];
    const XferSeg& g = A.seg[blockIdx.y];
    const int t = threadIdx.x;
    const size_t e0 = (size_t)blockIdx.x * 256;
    if (e0 >= g.n) return;
    const int m = (int)(g.n - e0 < 256 ? g.n - e0 : 256);
    const size_t i = g.first + e0 + t;
    const int w = g.kind == kXferVec ? 3 : g.kind == kXferStress ? 6 : 1;
    const double* in = buf + g.offset + e0 * w;
    for (int k = t; k < m * w; k += 256) sh[k] = in[k];
    __syncthreads();
    if (t >= m) return;
    void* dev = const_cast<void*>(g.dev);
    if (g.kind == kXferVec) {
        static_cast<double4*>(dev)[i] = make_double4(sh[3 * t], sh[3 * t + 1], sh[3 * t + 2], 0.0);
    } else if (g.kind == kXferStress) {
        for (int k = 0; k < 6; ++k) static_cast<double*>(dev)[(size_t)k * N + i] = sh[6 * t + k];
    } else {
        static_cast<double*>(dev)[i] = sh[t];
    }
}

// .w = |s| over the atom slots [a0, a0 + n), after the host uploaded spins
__global__ __launch_bounds__(256) void k_spin_len(Dev D, int a0, int n) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    D.s[a0 + k].w = spin_len(d3(D.s[a0 + k]));
}

// magmom: the spins from the moments, s = m / (-g), with |s| in .w
// (core_ds_CPU.cpp:37-45, read_config.cpp:136-139), for atom slots
// [a0, a0 + n)
__global__ __launch_bounds__(256) void k_magmom_s(Dev D, int a0, int n) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const double4 m = D.m[a0 + k];
    const double3 s = make_double3(m.x / -kElG, m.y / -kElG, m.z / -kElG);
    D.s[a0 + k] = make_double4(s.x, s.y, s.z, spin_len(s));
}

// magmom: the moments from the spins, m = -g s (core_ds_CPU.cpp:73-81)
__global__ __launch_bounds__(256) void k_magmom_m(Dev D) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= D.N) return;
    const double4 s = D.s[a];
    D.m[a] = make_double4(-kElG * s.x, -kElG * s.y, -kElG * s.z, 0.0);
}

__global__ __launch_bounds__(256) void k_check_nonfinite(Dev D) {
    int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= D.N) return;
    double4 r = D.r[a], p = D.p[a], s = D.s[a];
    double x = r.x + r.y + r.z + p.x + p.y + p.z + s.x + s.y + s.z;
    if (!isfinite(x)) atomicOr(D.err, kErrNonFinite);
}

}  // namespace sld
