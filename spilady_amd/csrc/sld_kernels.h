// Device state and kernel declarations of the spin-lattice engine.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sld_device.h"
#include "sld_dte_plan.h"
#include "sld_model.h"

namespace sld {

// One independent system of a batch: its geometry, thermostat temperature
// and noise stream, and where its atoms and link cells sit in the
// concatenated arrays. A replica's atom slots start on a 256-slot boundary and
// its cells on an 8-cell boundary, so that every block of the per-atom and
// per-cell reductions belongs to one replica; slots and cells in the padding
// have replica -1.
struct Rep {
    Box box;
    double temperature;   // k_B T, eV
    double box_volume;
    uint64_t seed;
    int replica;          // noise stream id
    int natom, atom0;     // atoms [atom0, atom0 + natom)
    int ncell, cell0;     // link cells [cell0, cell0 + ncell)
};

// Per-atom arrays are indexed by atom slot (replica atom0 + the caller's atom
// index); vectors are double4 with .w used as a payload (s.w = |s|, others 0).
struct Dev {
    int N, C;                  // atom slots and cells over all replicas, padding included
    const Rep* rep;            // [R]
    const int* arep;           // replica of each atom slot, -1 for padding [N]
    const int* crep;           // replica of each cell, -1 for padding [C]
    double4 *r, *p, *f, *s, *hh, *hl;
    double4* zn;               // Langevin normals of the current spin pass [N]
    double4 *hext, *fext;      // external field (eV) and force (eV/A) [N]; null when off
    uint64_t* pass_base;       // noise passes consumed before the current step [1]
    // quantum thermostat: noise history ring [2 Nf][3N] (slot e % 2Nf holds
    // history element e), current noise [3N], filter of each replica [R][2 Nf];
    // null when off
    double *qring, *qval;
    const double* qH;
    double *rho, *pe, *ke, *me, *me0, *vir, *sjs;
    double4* lan;              // Landau A, B, C, D at each atom's density [N] (kept current with rho)
    double* stress;            // [6][N]: 11 22 33 12 23 31
    double* lvol;              // localvol: each atom's local volume
    double4* m;                // magmom: the moments m = -g s, the state between spin passes
    int* cell;                 // link cell of each atom (new_cell_index)
    int* cell_prev;            // link cell before the last links()
    int* cslot;                // cell * kCellCap + position in the cell's list
    int *cl, *cn;              // cell lists [C][kCellCap] head->tail, counts [C]
    int *inc, *inc_n;          // atoms that moved into each cell this step, any order [C][kCellCap], counts [C]
                               // (zero between steps: the relink that consumes them clears them)
    int *nb, *nbn;             // neighbours within rcut_max [N][kMaxNb]
    int *nbm, *nbmn;           // neighbours within rcut_mag [N][kMaxMag]
    double* nbJ;               // J(r) of the rcut_mag neighbours [N][kMaxMag]
    // electron subsystem, per link cell
    double *Te, *Ee, *Tl, *Gel, *Ges, *TsR, *TsL, *sRup, *sRdn, *sLup, *sLdn;
    double4* cellv;            // per cell: x,y,z = mean p (localcolmot)
    int* err;                  // error flag bits
};

// The electron mesh as the core_dTe sub-step kernels read it.
struct Mesh {
    double *Te, *Ee;
    const double *Gel, *Ges, *Tl, *TsL;
    double2* src;  // per cell: h (Gel Tl + Ges TsL), and -(Gel + Ges) h / (3 b k_B)
    int C, lattlang, spinlang;
};

// Parameters shared by every replica of a batch.
struct Phys {
    double atmass, gamma_L, gamma_S;
    double rcut_pot, rcut_mag, rcut_pot_sq, rcut_mag_sq, rcut_max_sq;
    int spinlang, lattlang, eltemp, localcolmot;
    int extfield, extforce;
    int quantumnoise, qm, qnf2;  // quantum thermostat: on, redraw period M, filter taps 2 Nf
    int localvol;                // stress over per-atom local volumes
    int magmom;                  // moments as the spin variable
    double rcut_vol;             // their cut-off, A
};

// per-replica block of reduced scalars
constexpr int kScal = 64;
constexpr int kScalLvol = 56;  // localvol: the replica's sum of local volumes
// lanes per link cell in the momentum and temperature passes (a lane takes
// the cell's list entries l, l + kSeg, ...)
constexpr int kSeg = 8;

// ---- kernels ----
__global__ void k_bin(Dev D);
__global__ void k_relink(const int* cl_old, const int* cn_old, Dev D);
// dynamic LDS of k_nbuild, bytes a wave
constexpr int kNbLds = 256 * 16 + 27 * kCellCap * 4;
__global__ void k_nbuild(Tables T, Phys P, Dev D, int write_rho);
__global__ void k_fp(Tables T, Dev D);
__global__ void k_force(Tables T, Phys P, Dev D);
__global__ void k_lvol_sum(Dev D, double* partials);
__global__ void k_lvol_apply(Dev D, const double* scal);
__global__ void k_magmom_s(Dev D, int a0, int n);
__global__ void k_magmom_m(Dev D);
__global__ void k_spin_noise(Dev D, int pass_off);
__global__ void k_landau(Tables T, Dev D);
__global__ void k_step_max(Dev D, double* partials);
__global__ void k_scale_r(Dev D, double factor);
__global__ void k_rebox_r(Dev D, Box old_box, Box new_box);
__global__ void k_reduce_max2(const double* partials, int nblk, double* out);
__global__ void k_pass_advance(Dev D, int n);
__global__ void k_qn_init(Phys P, Dev D);
__global__ void k_qn_refresh(Phys P, Dev D, uint64_t r);
// ncw <= 16 cells a wave; store_fields: write Heff_H, Heff_L and sum J|s_j|
// (the backward sweep of a core_ds call)
template <bool kLang>
__global__ void k_spin_phase(const int* cells, int ncell, int ncw, int backward, int store_fields, double dt,
                             Phys P, Dev D);
__global__ void k_dp_cells(double dt, Phys P, Dev D, int pass_off, double* partials);
// partial sums of a replica that every block of a kernel may add for itself
constexpr int kFewRows = 512;
__global__ void k_dp_center(Phys P, Dev D, const double* scal, const double* in, const int* seg, int nrow,
                            double* partials);
__global__ void k_dp_scale(Phys P, Dev D, const double* scal, const double* in, const int* seg, int nrow);
__global__ void k_dr(double dt, Phys P, Dev D);
__global__ void k_temperature(Tables T, Phys P, Dev D);
__global__ void k_dte_ab(double h, Mesh M, double* partials);
// the C diffusion sweeps over the tiles of a schedule. Tout (may be null),
// Eout: the tile's own cells; ends (may be null): their final energies, one
// partial per tile; start (may be null): receives the sum of the na
// starting-energy partials pa, made by a block past the tiles.
// px, py, pz: the step's prefactor over the squared cell edges
struct DteTiles {
    const DteTile* tile;
    const uint4* upd;        // DteUpdate
    const int32_t* slot;
    const int32_t* lev;
    int ntile, max_slot;
};
struct DteSweepArgs {
    double px, py, pz;
    const double *Tin, *Ein;
    double *Tout, *Eout, *ends;
    const double* pa;
    int na;
    double* start;
};
// cells of a mesh that one workgroup sweeps on its own: 32 bytes of LDS a cell
constexpr int kDteSmall = 1024;
constexpr int kDteSmallBlock = 512;
__global__ void k_dte_small(DteTiles S, Mesh M, double h, double px, double py, double pz, int nloop);
template <int U>
__global__ void k_dte_sweep(DteTiles S, DteSweepArgs A);
// E: the energies the sweeps left; start: the sub-step's starting energy;
// ends: nend partials of its final one
__global__ void k_dte_finish(Mesh M, const double* E, const double* start, const double* ends, int nend);
__global__ void k_dte_finish_ab(Mesh M, const double* E, const double* start, const double* ends, int nend,
                                double* partials);
__global__ void k_obs_atoms(Tables T, Phys P, Dev D, double* partials, int scan_spin);
__global__ void k_obs_cells(Dev D, double* partials);
__global__ void k_renorm(Dev D, const double* err, double* partials);
__global__ void k_reduce(const double* partials, int nblk, double* out);
__global__ void k_reduce_seg(const double* partials, const int* seg, int nk, double* out, int out_off);
__global__ void k_check_nonfinite(Dev D);
__global__ void k_ee_of_te(Dev D, int c0, int n);
// Transfers between device arrays and dense host arrays: run k of a piece is n
// elements of seg[k].dev from element `first` on, at `offset` doubles of the
// pinned buffer. kXferVec: double4 to 3 doubles (.w = 0 on the way in);
// kXferStress: component-major [6][N] to 6 doubles an atom.
enum { kXferScalar = 0, kXferVec = 1, kXferStress = 2 };
constexpr int kXferSegs = 16;
struct XferSeg {
    const void* dev;
    size_t first, n, offset;
    int kind;
};
struct XferArgs {
    XferSeg seg[kXferSegs];
    int nseg;
};
__global__ void k_pack(XferArgs A, int N, double* buf);
__global__ void k_unpack(XferArgs A, int N, const double* buf);
__global__ void k_spin_len(Dev D, int a0, int n);

// ---- parametric potential model (sld_model.hip) ----
constexpr int kAdjBlocks = 2048;  // most blocks of the adjoint
constexpr int kFwdAtoms = 256;    // atoms of a block of the forward pass
struct ModelTab {
    const double* r;    // [N][kMRStride]
    const double *f, *df;  // [N]
    const double* h;    // [N][kMHStride]
    double in_over_rmax, in_over_rhomax;
    double L[4];        // Landau A B C D
    double JA, Jrc;
    double rmax, step;     // entry e of the r tables is at step * (e + 1)
    const double* bridge;  // ModelBridge
    int row0;
};
__global__ void k_model_tab_r(ModelCoef m, const double* bridge, double* out, double* out_f, double* out_df);
__global__ void k_model_tab_h(ModelCoef m, double* out);
template <bool kQ>
__global__ void k_model_rho(ModelTab M, Phys P, Dev D, double* rho_out, double* fp_out, const int* coff,
                            const double* gF, double* Q);
__global__ void k_model_forward(ModelTab M, Phys P, Dev D, const double* rho, const double* fp, const int* coff,
                                double* F, double* H, double* partials);
__global__ void k_model_adjoint(ModelTab M, Phys P, Dev D, int per_block, const double* rho, const double* fp, const double* Q,
                                const int* coff, const double* gE, const double* gF, const double* gH,
                                double* partials);

constexpr int kObsAtomK = 17;  // pe ke me me0 sx sy sz rup rdn lup ldn, then (vir) stress[6]
constexpr int kObsCellK = 6;   // Ee sRup sRdn sLup sLdn Te

}  // namespace sld
