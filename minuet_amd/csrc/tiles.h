// Tiles of targets that share their live offsets: what tile_sort_kernel and
// tile_emit_kernel (tiles.hip) leave of a dense kernel map and
// tiled_forward_kernel (tiled_kernel.h) walks.
#pragma once

#include <algorithm>
#include <cstdint>

#include "common.h"

namespace mnt {

constexpr int kTileTargets = 128;
constexpr int kTileWindow = 4096;             // most targets sorted together
constexpr int kTileMaxOffsets = 128;
constexpr int kTileXcds = 8;                  // windows are dealt to the compute dies in turn

// Targets are sorted within windows of consecutive ones.  The windows' number
// is a multiple of the compute dies', and tile p belongs to window
// (p / 8 / tiles_per_window) * 8 + p % 8: workgroups go to the dies in turn, so
// that the tiles of a window stay on one die and find each other's source rows
// in its L2.
struct TileLayout {
  int windows, window, per_window;            // window: targets of one (a multiple of kTileTargets)
  int64_t tiles;                              // windows * per_window
  int slots;                                  // rows of `sources` and `offsets` per tile: one per offset
  int64_t counts_at, offsets_at, sources_at, ints;

  TileLayout(int64_t targets, int64_t num_offsets) {
    windows = static_cast<int>(kTileXcds * std::max<int64_t>(1, div_ceil(targets, int64_t{kTileXcds} * kTileWindow)));
    window = static_cast<int>(div_ceil(std::max<int64_t>(1, div_ceil(targets, windows)), kTileTargets) * kTileTargets);
    per_window = window / kTileTargets;
    tiles = static_cast<int64_t>(windows) * per_window;
    slots = static_cast<int>(num_offsets);
    counts_at = tiles * kTileTargets;         // (rows at 0)
    offsets_at = counts_at + div_ceil(tiles, 4) * 4;
    sources_at = offsets_at + div_ceil(tiles * slots, 4) * 4;
    ints = sources_at + tiles * slots * kTileTargets;
  }
};

struct TileView {
  const int *rows;      // [tiles][128] target of a tile's place, -1 for none
  const int *counts;    // [tiles] live offsets; 0: no targets at all
  const int *offsets;   // [tiles][slots] their numbers
  const int *sources;   // [tiles][slots][128] source rows, -1 for none; rows from `counts` on are not written
};

}  // namespace mnt
