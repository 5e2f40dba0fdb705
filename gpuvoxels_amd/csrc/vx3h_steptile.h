// vx3h_steptile.h -- cutting a simulation into tiles for the fused per-step kernel.
#ifndef VX3H_STEPTILE_H
#define VX3H_STEPTILE_H
#include <cstddef>
#include <cstdint>
#include <vector>
#include "vx3_types.h"

namespace vx3 {

// The tiles of one simulation, one workgroup of VX3_TS_BLOCK threads each.  A tile owns up
// to VX3_TS_BLOCK voxels, one per thread, or a whole body of up to VX3_TS_OWN (at most
// VX3_TS_BLOCK of them on the surface); its slots are the owned voxels (surface voxels first,
// each group body by body and ascending) and then the halo: the other ends of their links.  stat holds per tile
// the rows of TsStat up to ST_END, with voxels, links and tiles counted within the simulation
// (row ST is the caller's to fill); each link belongs to the slot of its negative end.
struct StepTilePlan {
    std::vector<TsTile> tiles;   // tile, nTiles, nOwn, nSurf, nHalo, nIn; the rest is the caller's to fill
    std::vector<char> stat;
    int maxSlots = 0, maxOwn = 0;
    template <typename E> E* row(int tile, int off) { return (E*)(stat.data() + (size_t)tile * TsStat::ST_END + off); }
};

// Cuts the voxels [0, nv) (lattice indices ijk; vlinks: six link indices per voxel, -1 =
// none; interior per voxel) joined by links into tiles: connected bodies that fit a tile
// stay whole, near ones together where they are many and small; larger ones are cut into compact lattice blocks.  False
// for an empty simulation or a lattice of more than 2^16 along an axis.
bool planStepTiles(int nv, const int* ijk, int nl, const int* lneg, const int* lpos, const int* vlinks,
                   const char* interior, StepTilePlan* out);

// The numbers under which the fused kernel's steps report (TsReport).  Report words are matched
// by number and never cleared one by one, so a number is used once: when a call's would pass the
// largest, all words have to be cleared and the numbers start over.
struct TsNumbers {
    unsigned next = 1;   // (0: a cleared word's)
    // the first of n numbers (1 <= n <= 2^31), one after another; *restart: clear the words first
    unsigned take(unsigned n, bool* restart) {
        *restart = next == 0 || n - 1 > UINT32_MAX - next;
        if (*restart) next = 1;
        const unsigned first = next;
        next += n;
        return first;
    }
};

}  // namespace vx3
#endif
