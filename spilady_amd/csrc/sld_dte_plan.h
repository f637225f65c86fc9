// Tile schedules of the electron diffusion sweeps (host side, no device calls).
//
// A sweep updates every cell of the electron mesh once, in the order of the
// link-cell groups: a cell reads the new temperatures of its face neighbours
// of earlier groups and the old ones of later groups. The new value of a cell
// therefore depends on a small set of others, its closure: the cell, its
// earlier neighbours, theirs, and so on. It ends after at most as many steps
// as there are levels (4 on even meshes, up to about 20 on odd ones), and
// since each step goes down the group order it stays thin. A tile of the mesh
// together with the closure of its cells can be swept by one workgroup on its
// own, level by level, from the old temperatures alone; cells outside the
// tile are computed again by the tiles that own them, to the same bits. The
// same holds for a forward and a backward sweep taken together, with a larger
// closure.
//
// Cells are held relative to the tile's first cell, wrapped over the mesh's
// faces, so tiles alike in their surroundings (all but those near a face)
// share one set of lists.
#pragma once

#include <cstddef>
#include <cstdint>
#include <vector>

namespace sld {

enum DteSweeps { kDteForward = 0, kDteBackward = 1, kDteBoth = 2 };

// One update of a tile: byte offsets (8 x slot) of the cell and of its +x,
// -x, +y, -y, +z, -z neighbours.
struct DteUpdate {
    uint16_t self, nb[6], pad;
};
constexpr int kDteMaxLev = 63;       // levels of a schedule
constexpr int kDteMaxSlot = 8191;    // so that 8 x slot fits 16 bits

// A tile's cells live in numbered slots: first the updated ones, then those
// only read. slot lists hold 2 x (cell - origin), plus 1 if the tile owns the
// cell and writes it back.
struct DteTile {
    int32_t origin;
    int32_t upd0, nent;      // updates, level by level
    int32_t slot0, nupd, nslot;
    int32_t lev0, nlev;      // level l runs updates [lev[lev0 + l], lev[lev0 + l + 1])
};

struct DteSchedule {
    std::vector<DteTile> tile;
    std::vector<DteUpdate> upd;
    std::vector<int32_t> slot;
    std::vector<int32_t> lev;
    int max_ent = 0, max_upd = 0, max_slot = 0;
    long updates = 0;        // of all tiles
};

// The schedule over tiles of at most ex x ey x ez cells. group: link-cell
// group of each cell; the backward sweep takes the groups in descending
// order. False if the mesh needs more than most_levels
// levels or a tile exceeds the limits above.
bool dte_schedule(int nx, int ny, int nz, const std::vector<int>& group, DteSweeps sweeps, int ex, int ey, int ez,
                  int most_levels, DteSchedule& out);

}  // namespace sld
