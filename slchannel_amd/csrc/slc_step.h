// slc_step.h -- tile shape and budgets of the single-run step kernels
// (slc_step.hip: one component per launch; slc_step3.hip: three).
#pragma once

#include "slc_tile.h"

namespace slc {

// Tile of the step kernels: 4 x 4 x 16 arrival points, one per thread (measured
// at 256^3 order 6 against 4x4x32, 2x8x16, 8x4x8 and 4x8x8 tiles).  Compile-time
// overridable with -DSLC_TILE_TI=... for tile-shape sweeps.  The box budgets
// fill a CU's 160 KB of LDS at the occupancy the registers allow: four
// workgroups per CU (four waves per SIMD), less the workgroup's other LDS.
#ifndef SLC_TILE_TI
#define SLC_TILE_TI 4
#define SLC_TILE_TJ 4
#define SLC_TILE_TK 16
#endif
constexpr int kTI = SLC_TILE_TI, kTJ = SLC_TILE_TJ, kTK = SLC_TILE_TK;
constexpr int kTileLds = 40576;
constexpr int kTileLdsBdf2 = 31104;  // beside the near stencils' 9 KB
constexpr int kTileWavesPerSimd = 4;
// The gather at given feet and the near pass at order 4 fit seven waves per
// SIMD (72 VGPRs) with a 21 KB budget (an order-4 box of a 4x4x16 tile at the
// usual CFL takes 16-20 KB); at order 6 five or more spill.
constexpr int kGatherWaves4 = 7;
constexpr int kGatherLds4 = 21504;

}  // namespace slc
