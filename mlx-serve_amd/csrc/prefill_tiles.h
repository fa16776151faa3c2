// Which tile and K split a block of the prefill kernels works on.
#pragma once
#include "mi_common.h"

namespace mi {

struct TileOf {
  int mt, nt, split;
};

// Grid (tiles, splits). Blocks go to the 8 XCDs in turn, so block id b runs on XCD b % 8: the
// tiles are renumbered so that an XCD's blocks are a contiguous range of them, and numbered in
// panels of 4 row tiles, rows fastest. The 32 blocks that an XCD runs at a time then cover
// 4 x 8 tiles and read 4 x tiles and 8 weight tiles through its L2, whatever the grid (with
// ids row-fastest over the chip, 2003 rows gave an XCD 1 x tile and 32 weight tiles, each of
// which all 8 XCDs read). 256-row tiles, 4-bit, us: [14336,4096] 8192 rows 805 -> 750, 2003
// rows 230 -> 217, 512 rows 85 -> 81; [4096,14336] 8192 rows 759 -> 724.
MI_DEV TileOf tile_of_block(int mtiles, int ntiles) {
  constexpr int kPanel = 4;
  const int tiles = mtiles * ntiles, total = tiles * (int)gridDim.y;
  const int b = (int)(blockIdx.y * gridDim.x + blockIdx.x), xcd = b % 8;
  const int lin = xcd * (total / 8) + min(xcd, total % 8) + b / 8;
  const int split = lin / tiles, tile = lin - split * tiles;
  const int panel = tile / (kPanel * ntiles), r = tile - panel * kPanel * ntiles;
  const int h = min(kPanel, mtiles - panel * kPanel);
  return {panel * kPanel + r % h, r / h, split};
}

}  // namespace mi
