// Tile shapes of the split-bf16 kernels.
//
// Tiles (workgroup of C, waves, LDS): large 256 x 128, 8 waves of 64 x 64,
// 147 KB; medium 128 x 128, 8 waves of 32 x 64, 98 KB; small 64 x 64, 4 waves
// of 32 x 32, 49 KB (three workgroups per CU); for grids of at most one small
// tile per CU, two groups of 4 waves share its K (98 KB).  On full grids the large
// tile reaches 215 to 220 TFLOP/s of fp32 products (1.3 PFLOP/s of bf16 MFMA): the
// matrix cores are busy 58 % of the cycles at a clock of 2.09 GHz (Linear backward
// 8192 x 1024 x 4096, counters), the vector instructions of the splitting and the
// barriers fill the rest.
#pragma once
#include "gemm_args.hpp"
#include "split_core.hpp"

namespace gemm {

using LargeTile = split::Shape<4, 4, 4, 2>;
using MediumTile = split::Shape<2, 4, 4, 2, 2>;
using SmallTile = split::Shape<2, 2, 2, 2, 2>;
using PairedTile = split::Shape<2, 2, 2, 2, 2, 2>;
static_assert(LargeTile::TM == kSplitTm[0] && LargeTile::TN == kSplitTn[0] && MediumTile::TM == kSplitTm[1] &&
                  MediumTile::TN == kSplitTn[1] && SmallTile::TM == kSplitTm[2] && SmallTile::TN == kSplitTn[2],
              "tile table");

}  // namespace gemm
