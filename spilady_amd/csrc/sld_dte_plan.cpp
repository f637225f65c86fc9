// Tile schedules of the electron diffusion sweeps (sld_dte_plan.h).
#include "sld_dte_plan.h"

#include <algorithm>
#include <unordered_map>

#include "sld_threads.h"

namespace sld {
namespace {

struct Mesh {
    int nx, ny, nz;
    // +x -x +y -y +z -z
    void faces(int c, int out[6]) const {
        const int sl = nx * ny;
        const int x = c % nx, y = (c / nx) % ny, z = c / sl;
        out[0] = c + (x + 1 == nx ? 1 - nx : 1);
        out[1] = c + (x == 0 ? nx - 1 : -1);
        out[2] = c + (y + 1 == ny ? nx - sl : nx);
        out[3] = c + (y == 0 ? sl - nx : -nx);
        out[4] = c + (z + 1 == nz ? sl - nz * sl : sl);
        out[5] = c + (z == 0 ? nz * sl - sl : -sl);
    }
};

// the lists of one tile
struct Lists {
    std::vector<DteUpdate> upd;
    std::vector<int32_t> slot, lev;
    int nupd = 0;
    bool operator==(const Lists& o) const {
        auto same = [](const DteUpdate& a, const DteUpdate& b) {
            return a.self == b.self && std::equal(a.nb, a.nb + 6, b.nb);
        };
        return nupd == o.nupd && slot == o.slot && lev == o.lev && upd.size() == o.upd.size() &&
               std::equal(upd.begin(), upd.end(), o.upd.begin(), same);
    }
    size_t hash() const {
        size_t h = 1469598103934665603ull + (size_t)nupd;
        for (int32_t v : slot) h = (h ^ (size_t)(uint32_t)v) * 1099511628211ull;
        for (int32_t v : lev) h = (h ^ (size_t)(uint32_t)v) * 1099511628211ull;
        return h;
    }
};

struct Made {  // the tiles one thread makes
    std::vector<int> origin, which;
    std::vector<Lists> lists;
    bool ok = true;
};

int find_or_add(std::vector<Lists>& all, std::unordered_multimap<size_t, int>& by, Lists&& L) {
    const size_t h = L.hash();
    const auto r = by.equal_range(h);
    for (auto it = r.first; it != r.second; ++it)
        if (all[it->second] == L) return it->second;
    all.push_back(std::move(L));
    by.emplace(h, (int)all.size() - 1);
    return (int)all.size() - 1;
}

}  // namespace

bool dte_schedule(int nx, int ny, int nz, const std::vector<int>& group, DteSweeps sweeps, int ex, int ey, int ez,
                  int most_levels, DteSchedule& out) {
    const Mesh M{nx, ny, nz};
    const int C = nx * ny * nz;
    const int tx = (nx + ex - 1) / ex, ty = (ny + ey - 1) / ey, tz = (nz + ez - 1) / ez;
    const int ntile = tx * ty * tz;
    const bool fwd = sweeps != kDteBackward, bwd = sweeps != kDteForward;

    // level of each cell's forward and backward update: 1 + the highest level
    // among the updates whose values it reads
    int ngroup = 0;
    for (int g : group) ngroup = std::max(ngroup, g + 1);
    std::vector<int> order(C), first(ngroup + 1, 0), lf(C, -1), lb(C, -1);
    for (int g : group) ++first[g + 1];
    for (int g = 0; g < ngroup; ++g) first[g + 1] += first[g];
    {
        std::vector<int> fill(first.begin(), first.end() - 1);
        for (int c = 0; c < C; ++c) order[fill[group[c]]++] = c;
    }
    int nb[6], maxlev = 0;
    if (fwd)
        for (int c : order) {
            M.faces(c, nb);
            int lv = 0;
            for (int n : nb)
                if (group[n] < group[c]) lv = std::max(lv, lf[n] + 1);
            lf[c] = lv;
            maxlev = std::max(maxlev, lv + 1);
        }
    if (bwd)
        for (int k = C - 1; k >= 0; --k) {
            const int c = order[k];
            M.faces(c, nb);
            int lv = lf[c] + 1;
            for (int n : nb) lv = std::max(lv, (group[n] > group[c] ? lb[n] : lf[n]) + 1);
            lb[c] = lv;
            maxlev = std::max(maxlev, lv + 1);
        }
    if (maxlev > std::min(most_levels, kDteMaxLev)) return false;

    auto work = [&](int t0, int t1, Made& P) {
        // slot of a cell in the current tile; bits of its updates in the closure
        std::vector<int> slot(C, -1);
        std::vector<uint8_t> has(C, 0);
        std::vector<std::vector<int>> lev(maxlev);
        std::vector<int64_t> keys;
        std::vector<std::pair<int, int>> todo;  // (cell, backward)
        std::vector<int> cells, reads;
        std::unordered_multimap<size_t, int> by;
        for (int t = t0; t < t1; ++t) {
            const int a = t % tx, b = (t / tx) % ty, c3 = t / (tx * ty);
            const int x0 = a * ex, x1 = std::min(nx, x0 + ex);
            const int y0 = b * ey, y1 = std::min(ny, y0 + ey);
            const int z0 = c3 * ez, z1 = std::min(nz, z0 + ez);
            const int origin = x0 + y0 * nx + z0 * nx * ny;
            todo.clear();
            cells.clear();
            reads.clear();
            auto need = [&](int c, int back) {
                const uint8_t bit = (uint8_t)(1 << back);
                if (has[c] & bit) return;
                if (!(has[c] & 3)) cells.push_back(c);
                has[c] |= bit;
                todo.emplace_back(c, back);
            };
            for (int z = z0; z < z1; ++z)
                for (int y = y0; y < y1; ++y)
                    for (int x = x0; x < x1; ++x) {
                        const int c = x + y * nx + z * nx * ny;
                        has[c] |= 4;
                        need(c, bwd ? 1 : 0);
                    }
            int f[6];
            for (size_t k = 0; k < todo.size(); ++k) {
                const int c = todo[k].first, back = todo[k].second;
                M.faces(c, f);
                if (back && fwd) need(c, 0);
                for (int n : f) {
                    if (!back && group[n] < group[c]) need(n, 0);
                    if (back && group[n] > group[c]) need(n, 1);
                    if (back && fwd && group[n] < group[c]) need(n, 0);
                }
            }
            // slots by the level of a cell's first update, then by cell: the
            // cells of a level, and mostly their neighbours, are then
            // consecutive in LDS
            auto order_cells = [&](std::vector<int>& v) {
                keys.clear();
                for (int c : v) keys.push_back((int64_t)(fwd ? lf[c] : lb[c]) * C + c);
                std::sort(keys.begin(), keys.end());
                for (size_t k = 0; k < v.size(); ++k) v[k] = (int)(keys[k] % C);
            };
            order_cells(cells);
            Lists L;
            L.nupd = (int)cells.size();
            for (int c : cells) {
                slot[c] = (int)L.slot.size();
                L.slot.push_back(2 * (c - origin) + ((has[c] & 4) ? 1 : 0));
            }
            for (int c : cells) {
                M.faces(c, f);
                for (int n : f)
                    if (slot[n] < 0) {
                        slot[n] = 0;  // mark
                        reads.push_back(n);
                    }
            }
            order_cells(reads);
            for (int n : reads) {
                slot[n] = (int)L.slot.size();
                L.slot.push_back(2 * (n - origin));
            }
            if ((int)L.slot.size() > kDteMaxSlot) {
                P.ok = false;
                return;
            }
            for (auto& v : lev) v.clear();
            for (int c : cells) {  // in slot order
                if (has[c] & 1) lev[lf[c]].push_back(c);
                if (has[c] & 2) lev[lb[c]].push_back(c);
            }
            L.upd.reserve(todo.size());
            for (const auto& v : lev) {
                if (v.empty()) continue;
                L.lev.push_back((int32_t)L.upd.size());
                for (int c : v) {
                    DteUpdate d{};
                    d.self = (uint16_t)(8 * slot[c]);
                    M.faces(c, f);
                    for (int q = 0; q < 6; ++q) d.nb[q] = (uint16_t)(8 * slot[f[q]]);
                    L.upd.push_back(d);
                }
            }
            L.lev.push_back((int32_t)L.upd.size());
            for (int c : cells) {
                slot[c] = -1;
                has[c] = 0;
            }
            for (int n : reads) slot[n] = -1;
            P.origin.push_back(origin);
            P.which.push_back(find_or_add(P.lists, by, std::move(L)));
        }
    };
    int nt = (int)std::min(std::max(std::thread::hardware_concurrency(), 1u), 16u);
    nt = std::max(1, std::min(nt, ntile / 8));
    std::vector<Made> made(nt);
    run_parts(nt, [&](int k) { work((int)((long)ntile * k / nt), (int)((long)ntile * (k + 1) / nt), made[k]); });

    out = DteSchedule();
    std::vector<Lists> all;
    std::vector<DteTile> head;  // of each distinct set of lists
    std::unordered_multimap<size_t, int> by;
    for (Made& P : made) {
        if (!P.ok) return false;
        std::vector<int> id;
        for (Lists& L : P.lists) id.push_back(find_or_add(all, by, std::move(L)));
        for (size_t k = head.size(); k < all.size(); ++k) {
            const Lists& L = all[k];
            DteTile T{};
            T.upd0 = (int32_t)out.upd.size();
            T.nent = (int32_t)L.upd.size();
            T.slot0 = (int32_t)out.slot.size();
            T.nupd = L.nupd;
            T.nslot = (int32_t)L.slot.size();
            T.lev0 = (int32_t)out.lev.size();
            T.nlev = (int32_t)L.lev.size() - 1;
            out.upd.insert(out.upd.end(), L.upd.begin(), L.upd.end());
            out.slot.insert(out.slot.end(), L.slot.begin(), L.slot.end());
            out.lev.insert(out.lev.end(), L.lev.begin(), L.lev.end());
            out.max_ent = std::max(out.max_ent, T.nent);
            out.max_upd = std::max(out.max_upd, T.nupd);
            out.max_slot = std::max(out.max_slot, T.nslot);
            head.push_back(T);
        }
        for (size_t k = 0; k < P.which.size(); ++k) {
            DteTile T = head[id[P.which[k]]];
            T.origin = P.origin[k];
            out.updates += T.nent;
            out.tile.push_back(T);
        }
    }
    out.lev.resize(out.lev.size() + kDteMaxLev + 1, 0);  // a wave reads 64 level bounds at once
    return true;
}

}  // namespace sld
