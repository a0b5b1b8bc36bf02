// The query plan of a stride-1 kernel map worked out on the device: packing
// frame, key deltas of the offsets in ascending order and their groups, as
// make_plan() in query.hip builds them on the host from coordinate bounds
// that it had to wait for.  A chain of launches that never returns to the
// host (sort -> query -> lists) lets one wavefront of an earlier kernel write
// this block instead; the query kernel reads it from device memory.
#pragma once

#include <algorithm>
#include <cstring>

#include "device_utils.h"

namespace mnt {

constexpr int kPlanGroupSpan = 4;                // key span of one offset group (kGroupSpan of the query)
constexpr int kPlanMaxOffsets = 128;
constexpr int kPlanMaxKept = 64;                 // offsets that are looked up: one lane each
constexpr int kPlanInts = 6 * kPlanMaxKept;      // 4 words per group + 2 per member
constexpr int kPlanEach = kPlanMaxOffsets / kWave;

// Kernel offsets as launch arguments, and what can be said about them before the
// bounds of the cloud (which is mapped onto itself) are known.  halves != 0 when
// the offsets come in pairs d / -d (no offset named twice, at least one pair);
// kind[o] is then 0 for the offset of a pair that is looked up (the one whose
// first non-zero coordinate is positive, i.e. whose key delta is), 1 for its
// mirror image, 2 for the zero offset, and mirror[o] the index of the offset's
// mirror image.  The offsets that are looked up (all of them without halves) are
// listed in ascending order of their coordinates, equal ones by index.  That is
// the order of their key deltas: a field of the key has room for the difference
// of any two offsets, so the first coordinate that differs decides.
template <int MOST>
struct OffsetTableOf {
  int v[MOST][MNT_MAX_NDIM];              // the looked-up offsets in that order
  int reach_lo[MNT_MAX_NDIM];             // least and largest step along each axis, over all offsets
  int reach_hi[MNT_MAX_NDIM];
  int num_kept;                           // offsets that are looked up
  int halves;
  signed char origin[MOST];               // which offset each looked-up one is
  signed char kind[MOST];
  signed char mirror[MOST];
};
struct OffsetTable : OffsetTableOf<kPlanMaxOffsets> {};      // what a chain's kernels take

// The table of num_offsets <= MOST offsets, rows of ndim coordinates.
template <typename Table>
inline Table make_offset_table(const int64_t *offsets, int num_offsets, int ndim, bool allow_halves) {
  Table table;
  memset(&table, 0, sizeof(table));
  memset(table.mirror, -1, sizeof(table.mirror));
  int order[sizeof(table.kind)];
  for (int o = 0; o < num_offsets; ++o) {
    for (int k = 0; k < ndim; ++k) {
      const int step = static_cast<int>(offsets[o * ndim + k]);
      table.reach_lo[k] = std::min(table.reach_lo[k], step);
      table.reach_hi[k] = std::max(table.reach_hi[k], step);
    }
    order[o] = o;
  }
  const auto compare = [&](int a, int b) {
    for (int k = 0; k < ndim; ++k) {
      const int64_t u = offsets[a * ndim + k], v = offsets[b * ndim + k];
      if (u != v) return u < v ? -1 : 1;
    }
    return 0;
  };
  std::sort(order, order + num_offsets, [&](int a, int b) {
    const int c = compare(a, b);
    return c != 0 ? c < 0 : a < b;
  });
  // ascending and without repeats, the mirror image of the i-th is the i-th from the end
  bool paired = allow_halves && num_offsets > 1;
  for (int i = 0; i < num_offsets && paired; ++i) {
    const int64_t *d = offsets + static_cast<int64_t>(order[i]) * ndim;
    const int64_t *m = offsets + static_cast<int64_t>(order[num_offsets - 1 - i]) * ndim;
    for (int k = 0; k < ndim; ++k) paired = paired && d[k] == -m[k];
    paired = paired && (i == 0 || compare(order[i - 1], order[i]) != 0);
  }
  table.halves = paired ? 1 : 0;
  for (int i = 0; i < num_offsets; ++i) {
    const int o = order[i];
    if (paired) {
      const int other = num_offsets - 1 - i;
      table.kind[o] = static_cast<signed char>(i > other ? 0 : i == other ? 2 : 1);
      table.mirror[o] = static_cast<signed char>(order[other]);
      if (i <= other) continue;
    }
    for (int k = 0; k < ndim; ++k) table.v[table.num_kept][k] = static_cast<int>(offsets[o * ndim + k]);
    table.origin[table.num_kept++] = static_cast<signed char>(o);
  }
  return table;
}

struct DevicePlan {
  Frame frame;
  long long delta_min, delta_max;
  int num_groups;
  int groups_in_rows;       // every group's offsets differ in the last coordinate only
  int verdict;              // 0: go; otherwise the chain stops (sort declined, or keys beyond 63 bits)
  int num_members;          // offsets that are looked up
  int tables[kPlanInts];    // groups (first delta low / high, first member, members), then members (step, offset)
  // A cloud mapped onto itself under offsets that come in pairs d / -d: the
  // hits of -d are those of d with source and target exchanged, in the same
  // order (source positions rise with target positions), so only the offsets
  // of positive key delta are looked up.  halves != 0: kind[o] says what
  // offset o is (0 looked up, 1 the mirror image of offset mirror[o], 2 the
  // zero offset: every voxel is its own hit).
  int halves;
  int kind[kPlanMaxOffsets];
  int mirror[kPlanMaxOffsets];
  // the offsets that have rows of their own to write (all but the mirror
  // images), in offset order: offset | kind << 8 | (mirror + 1) << 16
  int rows[kPlanMaxOffsets];
  // Upper end of a tile's source window from the sort's bucket starts instead
  // of a search (a chain whose dealing launch worked by slabs; 0 buckets:
  // search).  The sort's key has coordinate 0 in its top field, so the rows
  // with coordinate 0 below x end where bucket ((x - lo) << shift) >> bucket_shift
  // starts (its next bucket when a bucket holds parts of two such planes).
  int window_buckets;
  int window_shift;               // of coordinate 0 in the sort's key
  int window_bucket_shift;        // sort key >> this = bucket
  int window_reach;               // largest offset along coordinate 0
  long long window_lo, window_hi; // range of coordinate 0 in the cloud
  const unsigned *window_starts;  // [window_buckets + 1]
};

__device__ __forceinline__ int plan_bits(unsigned long long range) {
  return range == 0 ? 0 : 64 - __builtin_clzll(range);
}

// What lane l of the planning wavefront takes from the launch arguments: looked-up
// offset l and what is said about offsets l and 64 + l.  Read with the lane's index (a load
// per lane; picking them out of scalar registers took some 400 instructions) and
// before the bounds are there.
struct PlanLane {
  int d[MNT_MAX_NDIM];
  int origin, kind[kPlanEach], mirror[kPlanEach];
};

__device__ __forceinline__ PlanLane load_plan_lane(const OffsetTable &offsets) {
  const int lane = lane_id();
  PlanLane in;
#pragma unroll
  for (int k = 0; k < MNT_MAX_NDIM; ++k) in.d[k] = offsets.v[lane][k];
  in.origin = offsets.origin[lane];
#pragma unroll
  for (int e = 0; e < kPlanEach; ++e) {
    in.kind[e] = offsets.kind[e * kWave + lane];
    in.mirror[e] = offsets.mirror[e * kWave + lane];
  }
  return in;
}

// Run by ONE whole wavefront.  bounds = lo[4], hi[4] of the cloud (sources and
// targets are the same rows); the frame leaves room for every offset on both
// sides of every field, so key(q + offset) == key(q) + delta(offset).
// `declined` is the verdict of the launches before (non-zero: stop).
// The launch that carries it waits for it, so everything that needs no bounds is
// in `offsets` already and no step here is a loop over cross-lane reads (with
// the ordering and the ranges worked out here it took 10 us, of 28 us for
// sorting 2 000 rows).
__device__ __forceinline__ void make_plan_on_device(const long long *__restrict__ bounds, const PlanLane &in,
                                                    const OffsetTable &offsets, int num_offsets,
                                                    int ndim, unsigned declined, DevicePlan *__restrict__ out,
                                                    const unsigned *__restrict__ bucket_starts = nullptr,
                                                    int msd_cap = 0) {
  const int lane = lane_id();
  Frame f;
  int bits = 0;
  bool fits = true;
#pragma unroll
  for (int k = MNT_MAX_NDIM - 1; k >= 0; --k) {
    f.lo[k] = 0;
    f.shift[k] = 0;
    f.width[k] = 0;
    if (k < ndim) {
      // coordinates are at most 64-bit and the reach is small: a range that wraps is caught below
      const long long lo = bounds[k] + offsets.reach_lo[k];
      const long long hi = bounds[MNT_MAX_NDIM + k] + offsets.reach_hi[k];
      const unsigned long long range = static_cast<unsigned long long>(hi) - static_cast<unsigned long long>(lo);
      fits = fits && hi >= lo && lo <= bounds[k] && hi >= bounds[MNT_MAX_NDIM + k] && range < (1ull << 63);
      f.lo[k] = lo;
      f.width[k] = plan_bits(range);
      f.shift[k] = bits < 63 ? bits : 63;
      bits += f.width[k];
    }
  }
  f.batch_width = 0;
  f.batch_shift = bits < 63 ? bits : 63;
  f.ndim = ndim;
  f.total_bits = bits;
  fits = fits && bits <= 63;

  long long mine = 0;
#pragma unroll
  for (int k = 0; k < MNT_MAX_NDIM; ++k) {
    if (k < ndim) {
      mine += static_cast<long long>(static_cast<unsigned long long>(static_cast<long long>(in.d[k])) << f.shift[k]);
    }
  }
  const bool halves = offsets.halves != 0;
  const int num_kept = offsets.num_kept;
  const bool placed = lane < num_kept;
  // first place whose delta lies beyond this one's group span (num_kept if
  // none), and never more than kPlanGroupSpan + 1 members (repeated offsets)
  int next = lane + kPlanGroupSpan + 1 < num_kept ? lane + kPlanGroupSpan + 1 : num_kept;
#pragma unroll
  for (int j = kPlanGroupSpan; j >= 1; --j) {
    const long long other = __shfl(mine, lane + j < kWave ? lane + j : kWave - 1);
    next = lane + j < num_kept && other - mine > kPlanGroupSpan ? lane + j : next;
  }
  // the greedy grouping follows those links from place 0
  unsigned long long starts = 0;
  int num_groups = 0;
  for (int cur = 0; cur < num_kept; cur = __builtin_amdgcn_readlane(next, cur)) {
    starts |= 1ull << cur;
    ++num_groups;
  }
  const unsigned long long upto = starts & ((2ull << lane) - 1ull);
  const int group = __popcll(upto) - 1;
  const int first_place = placed ? 63 - __builtin_clzll(upto) : 0;
  const long long first_delta = __shfl(mine, first_place);
  bool same_row = true;
#pragma unroll
  for (int k = 0; k < MNT_MAX_NDIM; ++k) {
    const int other = __shfl(in.d[k], first_place);
    same_row = same_row && (k + 1 >= ndim || other == in.d[k]);
  }
  const bool in_rows = __ballot(placed && !same_row) == 0ull;
  if (placed) {
    out->tables[4 * num_groups + 2 * lane + 0] = static_cast<int>(mine - first_delta);
    out->tables[4 * num_groups + 2 * lane + 1] = in.origin;
    if ((starts >> lane) & 1ull) {
      const unsigned long long first = static_cast<unsigned long long>(mine);
      out->tables[4 * group + 0] = static_cast<int>(static_cast<unsigned>(first & 0xffffffffull));
      out->tables[4 * group + 1] = static_cast<int>(static_cast<unsigned>(first >> 32));
      out->tables[4 * group + 2] = lane;
      out->tables[4 * group + 3] = next - lane;
    }
  }
  int rows = 0;
#pragma unroll
  for (int e = 0; e < kPlanEach; ++e) {
    const int o = e * kWave + lane;
    const bool live = o < num_offsets;
    const bool writes = live && in.kind[e] != 1;
    const unsigned long long writers = __ballot(writes);
    if (live) {
      out->kind[o] = in.kind[e];
      out->mirror[o] = in.mirror[e];
    }
    if (writes) out->rows[rows + __popcll(writers & lanes_below())] = o | (in.kind[e] << 8) | ((in.mirror[e] + 1) << 16);
    rows += __popcll(writers);
  }
  const long long delta_min = __shfl(mine, 0);
  const long long delta_max = __shfl(mine, num_kept > 0 ? num_kept - 1 : 0);
  if (lane == 0) {
    out->frame = f;
    out->delta_min = num_kept > 0 ? delta_min : 0;
    out->delta_max = num_kept > 0 ? delta_max : 0;
    out->halves = halves ? 1 : 0;
    out->num_groups = num_groups;
    out->groups_in_rows = in_rows ? 1 : 0;
    out->verdict = declined != 0 ? static_cast<int>(declined) : (fits ? 0 : 2);
    out->num_members = num_kept;
    // the sort's key: fields of the cloud's own ranges, coordinate 0 on top
    int sort_bits = 0, below_top = 0;
#pragma unroll
    for (int k = MNT_MAX_NDIM - 1; k >= 0; --k) {
      if (k < ndim) {
        const int w = plan_bits(static_cast<unsigned long long>(bounds[MNT_MAX_NDIM + k]) -
                                static_cast<unsigned long long>(bounds[k]));
        if (k > 0) below_top += w;
        sort_bits += w;
      }
    }
    const int msd_bits = sort_bits < msd_cap ? sort_bits : msd_cap;
    const bool usable = bucket_starts != nullptr && sort_bits >= 1 && sort_bits <= 63 && sort_bits > below_top;
    out->window_buckets = usable ? 1 << msd_cap : 0;
    out->window_shift = below_top;
    out->window_bucket_shift = sort_bits - msd_bits;
    out->window_reach = offsets.reach_hi[0];
    out->window_lo = bounds[0];
    out->window_hi = bounds[MNT_MAX_NDIM];
    out->window_starts = bucket_starts;
  }
}

}  // namespace mnt
