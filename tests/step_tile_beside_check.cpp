// tests/step_tile_check.cpp for a plan made beside a million voxels of other simulations.
#include "../gpuvoxels_amd/csrc/vx3h_steptile.h"

#define planStepTiles(nv, ijk, nl, neg, pos, vlinks, interior, out) planStepTiles(nv, ijk, nl, neg, pos, vlinks, interior, out, 1000000)
#include "step_tile_check.cpp"
