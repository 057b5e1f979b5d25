// tile_place.h -- which tile of a prompt's int8-weight product a workgroup takes.
#pragma once

#include "common.h"

#include <algorithm>

namespace bh {

// Ids equal modulo 8 run on the same XCD.  An XCD takes a run of an eighth of all tiles, in
// panels of `panel` (column tile, K slice) pairs by all row tiles: the workgroups that it
// runs at the same time share rows and weights in its L2, and no XCD has more than one tile
// above another.  (Pairs shared out to the XCDs, all of an XCD's pairs for a row tile before
// the next row tile: the weights of many columns leave the L2 between two row tiles.
// 4096 -> 2 x 14336, two planes: 640 rows 252 us so, 182 in panels; 1536 -> 8960, whose 35
// columns made it cut the rows into bands besides, 4096 rows 274 and 160.)
//
// panel == 0: the pairs are shared out to the XCDs after all (false: a padding id).
__device__ __forceinline__ bool place_tile(int units, int rows, int panel, int &unit, int &row) {
  const int id = blockIdx.x;
  if (panel == 0) {
    const int ids = (units + 7) & ~7;
    row = id / ids;
    unit = id - row * ids;
    return unit < units;
  }
  const int total = units * rows, die = id % 8;
  const int t = die * (total / 8) + min(die, total % 8) + id / 8;
  const int p = t / (panel * rows), rest = t - p * panel * rows;
  const int width = min(panel, units - p * panel);
  row = rest / width;
  unit = p * panel + rest - row * width;
  return true;
}
// The 64 workgroups of an XCD are 4 pairs by 16 row tiles at a time, with fewer row tiles
// all of them by as many pairs as it takes, one pair after the other.  Rows of several planes are more bytes than
// the weights of a tile: 6 pairs, whose rows are read for the first and found in L2 by the others (three planes,
// prompts of 600, 1000, 1300 and 1931 tokens 4255, 6307, 7537 and 10592 us with 1 or 2 pairs, 4166, 6175, 7470 and
// 10574 so; two planes, 900 and 2048 tokens 5053 and 9700, 4946 and 9453; of more than 32 row tiles 4096 tokens 21595
// with 4 and 21912 with 6; one plane, 1536 -> 8960, 384 rows 18.7 and 19.0).  Of few row tiles every
// pair should be on one XCD only and workgroups that start one behind the other on different
// weights (100 rows, 1536 -> 2 x 8960, two planes: 17.8 us shared out, 19.5 in panels; 224
// rows 23.5 and 23.0), unless that gives an XCD a second workgroup on a compute unit that its
// share alone does not, or notably more of them.
inline int panel_for(int64_t units, int row_tiles, bool planes) {
  const int64_t most = ceil_div(units, 8) * row_tiles, tiles = units * row_tiles;
  if (row_tiles <= 5 && (most <= 32 || (tiles > 8 * 32 && 100 * 8 * most <= 106 * tiles)))
    return 0;
  if (planes && row_tiles > 5 && row_tiles <= 32)
    return 6;
  return row_tiles <= 16 ? 1 : row_tiles <= 32 ? 2 : 4;
}

} // namespace bh
