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
// is a multiple of the compute dies' and workgroups go to the dies in turn, so
// window w's tiles, all at numbers of w % 8 modulo 8, stay on one die and find
// each other's source rows in its L2.
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

// The number of the `place`-th longest tile of a window, which is when it runs.
// The longest tiles of all windows go first: one of a map's rare tiles of 27
// live offsets takes three times the average, and the chip waited for those of
// the last windows.  Then the next longest of a band of windows at a time, as
// many as leave their rows in a die's L2 (seven of 4096 128-byte rows), and not
// window after window, whose long tiles leave gaps.  us a layer with 8 windows
// after the other and so: 64 -> 64 channels of 16 bits over 200 000 LiDAR voxels
// 34.4 and 28.6, over a room of 150 000 26.3 and 20.4; over a million, where the last
// windows are a small part, under 5x5x5 415 to 422 and 401 to 411, 32 -> 32 under 3x3x3
// 85.7 and 84.2.
constexpr int kTileFirst = 2, kTileBand = 7;
__device__ __forceinline__ int tile_number(int windows, int per_window, int window, int place) {
  const int rows = windows / kTileXcds, row = window / kTileXcds;      // windows of a die
  const int first = per_window < kTileFirst ? per_window : kTileFirst;
  int at = place * rows + row;                                         // among the die's tiles
  if (place >= first) {
    const int band = row / kTileBand * kTileBand;
    const int in_band = rows - band < kTileBand ? rows - band : kTileBand;
    at = first * rows + band * (per_window - first) + (place - first) * in_band + row - band;
  }
  return at * kTileXcds + window % kTileXcds;
}

struct TileView {
  const int *rows;      // [tiles][128] target of a tile's place, -1 for none
  const int *counts;    // [tiles] live offsets; 0: no targets at all
  const int *offsets;   // [tiles][slots] their numbers
  const int *sources;   // [tiles][slots][128] source rows, -1 for none; rows from `counts` on are not written
};

}  // namespace mnt
