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
// stay whole, near ones together where they are many and small; larger ones are cut into compact lattice blocks.
// beside: voxels that other simulations step beside these in the same launches.  False
// for an empty simulation or a lattice of more than 2^16 along an axis.
bool planStepTiles(int nv, const int* ijk, int nl, const int* lneg, const int* lpos, const int* vlinks,
                   const char* interior, StepTilePlan* out, long long beside = 0);

// Whether a launch of `tiles` tiles with `voxels` voxels in them steps faster than the per-step
// kernels, whose time follows the voxels, not the tiles: small bodies that are far apart hardly
// share tiles.  Measured on MI355X, us per step, lists rebuilt every 8 steps, per-step kernels
// and fused, FP64 and FP32:
//                                      tiles   voxels         FP64           FP32
//   2,000 lone voxels, 8 apart           979    2,000    24.2   20.1    23.0   20.2
//   4,000                              2,000    4,000    24.7   31.4    23.1   32.0
//   2,000 cubes of 2^3, 12 apart         865   16,000    41.8   37.2    38.3   34.6
//   4,000                              1,740   32,000    47.9   55.2    41.5   51.0
//   4,000 cubes of 3^3, 20 apart       1,876  108,000    88.7   66.5    72.2   61.4
//   8,000 balls of 33, 16 apart        3,980  264,000   139.4  130.4   105.8  118.5
//   8,000 cubes of 4^3, 24 apart       4,494  512,000   310.9  163.5   216.7  139.1
inline bool stepTilesPay(long long tiles, long long voxels, size_t realBytes) {
    return tiles <= 1000 || voxels >= (realBytes == 8 ? 80 : 96) * (tiles - 1000);
}

// Whether the fused kernel's list rebuilds pay too: each tile with surface voxels (`surface` of a
// simulation's `tiles`) reads the bounds of all, where the per-step kernels hash the voxels.
// Measured on MI355X, us per step, balls of 257 voxels in FP32, one a tile, rebuilt every 8 steps,
// per-step kernels and fused: 16,384 balls 1,727 and 1,074, 32,768 balls 3,556 and 2,338, 65,536
// balls 7,193 and 6,475.
inline bool stepRebuildsPay(long long tiles, long long surface) { return surface <= (1LL << 32) / (tiles > 0 ? tiles : 1); }

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
