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

struct lt_split_place { int tile, slice; };

// A split reduction, slice by slice: an XCD's workgroups are neighbouring tiles of one slice or two and read the same rows of k through
// its L2.  Weight gradient [768, 3072] over 16384 (36 tiles, 7 slices), tiles dealt to the XCDs in turn against this: 95 us, 85.
LT_HOST_DEVICE inline lt_split_place lt_split_by_slice(int v, int tiles, int slices) {
  const int place = lt_xcd_order(v, tiles * slices);
  return {place % tiles, place / tiles};
}

// Tile by tile: an XCD's workgroups are the whole reductions of neighbouring tiles
LT_HOST_DEVICE inline lt_split_place lt_split_by_tile(int v, int tiles, int slices) {
  const int place = lt_xcd_order(v, tiles * slices);
  return {place / slices, place % slices};
}

// 128 x 128 tiles, k-major A: tile by tile where one operand is streamed, with next to nothing of it used by two tiles (one tile column,
// or two tile rows), and that operand is over 64 MiB.  By slices an XCD would read a narrow band of k of all its rows.  Slice by
// slice and tile by tile: [4096, 128] over 16384 56 us, 50; [4096, 64] over 16384 57, 48; [129, 4096] over 32768 106, 94; [129, 4096] over
// 16384 58, 54.  Below that size slice by slice is the faster one ([1000, 128] over 16384 16.8, 18.8), and by far where both operands are
// used again ([4096, 256] over 16384 40, 52).
LT_HOST_DEVICE inline bool lt_split_tiles_first(int64_t M, int64_t N, int64_t K) {
  const bool thin = N <= 128 || M <= 256;
  return thin && (M > N ? M : N) * K > (int64_t)1 << 25;
}
