// Offsets of buffer loads that may point past their operand, as plain constexpr functions: tests/test_load_ranges.py
// checks them on the CPU. Whether the hardware counts a load's scalar offset when it compares with the resource's size
// (offset >= size - scalar, which wraps for an empty resource, or offset >= size) differs between descriptions, so no
// load relies on either: a load that must not reach memory has a scalar offset of 0 and a vector offset at or past the
// size.
#pragma once

struct LoadRange {
  int bytes, at;  // the resource's size and the loads' scalar offset
};

// Tile t of `tiles`, `step` bytes apart along the rows of an operand of `bytes`. Past the last tile: an empty resource,
// so that the loads count but touch no memory.
constexpr LoadRange tile_range(int t, int tiles, int bytes, int step) {
  return t < tiles ? LoadRange{bytes, t * step} : LoadRange{0, 0};
}

// What a load of column `col` (of `cols`) adds to its row's offset: `bytes`, or past every operand whose rows span less
// than 2^30 bytes (row offsets stay below that too, so the sum fits 31 bits).
constexpr int column_offset(int col, int cols, int bytes) { return col < cols ? bytes : 1 << 30; }
