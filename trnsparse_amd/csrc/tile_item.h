// Order of the output tiles of a product over the workgroups of a launch.
#pragma once

#include "common.h"

namespace tsp {

// Work item of a tiled launch over `mb` row tiles (ranked heaviest first by
// `order`, or in natural order when it is null) and `nt` column tiles.
// Consecutive workgroup ids go round-robin over the 8 XCDs: ranks are dealt
// to XCDs in boustrophedon order (0..7, 15..8, 16..23, ...) so every XCD
// gets an equal share of heavy and light rows, and the column tiles of one
// row sit in consecutive slots of one XCD (they share its L2 for the A row
// panel). Returns false for padding slots.
__device__ inline bool tile_item(int64_t g, int64_t mb, int64_t nt, const int32_t* __restrict__ order,
                                 int64_t& row, int& ntile) {
  const int64_t xcd = g & 7, slot = g >> 3;
  const int64_t rl = slot / nt;
  ntile = (int)(slot - rl * nt);
  const int64_t k = (rl & 1) ? 8 * rl + 7 - xcd : 8 * rl + xcd;
  if (k >= mb) return false;
  row = order ? (int64_t)order[k] : k;
  return true;
}

}  // namespace tsp
