// Which tile, and which slice of a split reduction, a workgroup takes.  Plain C++, so that it can be tested on the host.
// Workgroup v of a launch (x fastest) runs on XCD v % 8, and each XCD has an L2 of its own.
#pragma once
#include <cstdint>

#include "lt_steps.h"  // LT_HOST_DEVICE

// In runs: the place workgroup v of n takes in an order in which the workgroups of one XCD follow each other
LT_HOST_DEVICE inline int lt_xcd_order(int v, int n) {
  const int each = n >> 3, more = n & 7, xcd = v & 7;
  return xcd * each + (xcd < more ? xcd : more) + (v >> 3);
}

// In turn where 8 does not divide n: neighbouring places on neighbouring XCDs
LT_HOST_DEVICE inline int lt_turn_order(int v, int n) { return (n & 7) == 0 ? (v & 7) * (n >> 3) + (v >> 3) : v; }

// Whether the workgroups of a copy-based launch can start their walk over k at different offsets: one segment of whole blocks of 64 k
LT_HOST_DEVICE inline bool lt_can_stagger(int nseg, int64_t k) { return nseg == 1 && (k & 63) == 0; }

// Tiles of an unsplit product.  staggered: two k-major operands whose workgroups start their walk over k an eighth apart, XCD by
// XCD.  With few tile rows the tiles of a column then go to the XCDs in turn, so that each starts at another part of that column's
// weights; in runs they share one XCD and start together.  Weights from memory, rows x columns of tiles, in runs and in turn: 7 x 49 over
// 3072 142 us, 138; 6 x 47 over 3008 131, 123; 9 x 33 over 2048 98, 92; 10 x 47 over 3008 168, 162.  The other way round with more rows (14 x 25
// over 1600 81, 83; 11 x 47 over 3008 with an activation 243, 250) or without the stagger (7 x 33 over 2064 with an activation 72, 93).
constexpr int LT_TURN_ROWS = 10;
LT_HOST_DEVICE inline int lt_tile_order(int v, int tiles_m, int tiles_n, bool staggered) {
  return staggered && tiles_m <= LT_TURN_ROWS ? lt_turn_order(v, tiles_m * tiles_n) : lt_xcd_order(v, tiles_m * tiles_n);
}
