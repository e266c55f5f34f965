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


// Head and item (block row, or a part of one) of a launch of head_grid(P, H)
// workgroups over H heads of P items each. XCD x walks whole heads x, x + 8,
// ..., whose items share the head's K and V in its L2; the H % 8 heads left
// over are dealt by eighths of their item list, so that the XCDs end together
// (one head alone ran on one of them: 8192, head_dim 128, window 4, 2 global
// blocks, fp32 forward 201 -> 105 us, gradients 487 -> 317).
__host__ __device__ inline int64_t head_grid(int64_t P, int64_t H) {
  return 8 * (H / 8 * P + ceil_div(H % 8 * P, 8));
}
// The grid fits int32, so 32-bit divisions do.
__device__ inline bool head_item(uint32_t g, int64_t P_, int64_t H_, int64_t& head, int64_t& item) {
  const uint32_t P = (uint32_t)P_, H = (uint32_t)H_;
  const uint32_t xcd = g & 7, slot = g >> 3, whole = H / 8 * P;
  const uint32_t rest = H % 8 * P, per = (rest + 7) / 8;
  const bool tail = slot >= whole;
  const uint32_t i = tail ? xcd * per + slot - whole : slot, q = i / P;
  head = tail ? (H & ~7u) + q : xcd + 8 * q;
  item = i - q * P;
  if (tail && (slot - whole >= per || i >= rest)) return false;
  return true;
}

}  // namespace tsp
