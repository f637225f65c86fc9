// The tile schedules of the electron diffusion (spilady_amd/csrc/sld_dte_plan.h)
// against the group-by-group sweep they stand for: a made-up cell update that
// depends on every neighbour in another way is swept in both, and each cell
// has to be written once and to the same bits.
//   dte_plan_check nx0 nx1 edge...   every mesh with sides in [nx0, nx1]
#include "sld_dte_plan.h"

#include <cmath>
#include <cstdio>
#include <cstdlib>

using namespace sld;

static std::vector<int> greedy(int nx, int ny, int nz) {
    const int C = nx * ny * nz;
    std::vector<int> type(C, 0), group(C, -1);
    for (int left = C, g = 0; left > 0; ++g) {
        for (int i = 0; i < C; ++i) {
            if (type[i] != 0) continue;
            type[i] = 1;
            group[i] = g;
            --left;
            const int x = i % nx, y = (i / nx) % ny, z = i / (nx * ny);
            for (int d = 0; d < 27; ++d) {
                const int n = (x + d % 3 - 1 + nx) % nx + ((y + d / 3 % 3 - 1 + ny) % ny) * nx +
                              ((z + d / 9 - 1 + nz) % nz) * nx * ny;
                if (type[n] != 1) type[n] = -1;
            }
        }
        for (int& t : type)
            if (t == -1) t = 0;
    }
    return group;
}

static double update(double c, const double* n) {
    return 0.9 * c + 0.01 * (n[0] + 1.1 * n[1] + 1.2 * n[2] + 1.3 * n[3] + 1.4 * n[4] + 1.5 * n[5]) + 1e-3 * std::sin(c);
}

static int check(int nx, int ny, int nz, int e, DteSweeps sweeps, bool must) {
    const std::vector<int> group = greedy(nx, ny, nz);
    const int C = nx * ny * nz;
    DteSchedule S;
    if (!dte_schedule(nx, ny, nz, group, sweeps, e, e, e, kDteMaxLev, S)) return must ? 1 : 0;
    std::vector<double> T(C), R, O(C, 0.0);
    for (int c = 0; c < C; ++c) T[c] = std::sin(1.7 * c) + 1e-5 * c;
    R = T;
    int ngroup = 0;
    for (int g : group) ngroup = g + 1 > ngroup ? g + 1 : ngroup;
    for (int back = 0; back < 2; ++back) {
        if (sweeps != kDteBoth && back != (sweeps == kDteBackward)) continue;
        for (int k = 0; k < ngroup; ++k)
            for (int c = 0; c < C; ++c) {
                if (group[c] != (back ? ngroup - 1 - k : k)) continue;
                const int x = c % nx, y = (c / nx) % ny, z = c / (nx * ny);
                auto at = [&](int i, int j, int l) {
                    return R[(i + nx) % nx + ((j + ny) % ny) * nx + ((l + nz) % nz) * nx * ny];
                };
                const double n[6] = {at(x + 1, y, z), at(x - 1, y, z), at(x, y + 1, z),
                                     at(x, y - 1, z), at(x, y, z + 1), at(x, y, z - 1)};
                R[c] = update(R[c], n);
            }
    }
    std::vector<int> written(C, 0);
    int bad = 0;
    for (const DteTile& t : S.tile) {
        std::vector<double> v(t.nslot);
        for (int s = 0; s < t.nslot; ++s) {
            const int c = t.origin + (S.slot[t.slot0 + s] >> 1);
            if (c < 0 || c >= C) return 1;
            v[s] = T[c];
        }
        bad += t.nslot > S.max_slot || t.nupd > S.max_upd || t.nent > S.max_ent || t.nslot > kDteMaxSlot;
        bad += S.lev[t.lev0] != 0 || S.lev[t.lev0 + t.nlev] != t.nent ||
               t.lev0 + kDteMaxLev + 1 > (int)S.lev.size() || t.nlev > kDteMaxLev;
        for (int l = 0; l < t.nlev; ++l) {
            const std::vector<double> old = v;  // the updates of a level may run in any order
            for (int k = S.lev[t.lev0 + l]; k < S.lev[t.lev0 + l + 1]; ++k) {
                const DteUpdate& u = S.upd[t.upd0 + k];
                double n[6];
                for (int q = 0; q < 6; ++q) n[q] = old[u.nb[q] / 8];
                bad += u.self / 8 >= t.nupd;
                v[u.self / 8] = update(old[u.self / 8], n);
            }
        }
        for (int s = 0; s < t.nupd; ++s) {
            const int r = S.slot[t.slot0 + s];
            if (!(r & 1)) continue;
            O[t.origin + (r >> 1)] = v[s];
            ++written[t.origin + (r >> 1)];
        }
    }
    for (int c = 0; c < C; ++c) bad += written[c] != 1 || O[c] != R[c];
    return bad;
}

int main(int argc, char** argv) {
    const int lo = std::atoi(argv[1]), hi = std::atoi(argv[2]);
    int bad = 0;
    for (int x = lo; x <= hi; ++x)
        for (int y = lo; y <= hi; ++y)
            for (int z = lo; z <= hi; ++z)
                for (int a = 3; a < argc; ++a)
                    for (DteSweeps s : {kDteForward, kDteBackward, kDteBoth}) {
                        const int b = check(x, y, z, std::atoi(argv[a]), s, s != kDteBoth);
                        if (b) std::printf("%d %d %d tiles of %s sweeps %d: %d\n", x, y, z, argv[a], (int)s, b);
                        bad += b;
                    }
    std::printf("bad %d\n", bad);
    return bad != 0;
}
