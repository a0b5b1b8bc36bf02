// Sorting the targets of a dense kernel map into tiles that share their live
// offsets.
//
// A matrix instruction multiplies 32 targets under one offset whether they
// have a source there or not.  In the order of a sorted cloud 128 neighbouring
// targets of a surface use 20 of 27 offsets between them but 3 to 5 each; put
// in the order of the SETS of offsets they use, 128 of them use 7 to 11.  The
// reference has one order only (csrc/minuet/cuda/functions/sparse_convolution.cu
// multiplies hit lists per offset, which need no such order, and pays with
// buffer rows for every hit).
#include <algorithm>
#include <type_traits>
#include <vector>

#include "device_utils.h"
#include "tiles.h"

namespace mnt {

constexpr int kTileSortBlock = 1024;
constexpr int kTileSortWaves = kTileSortBlock / kWave;
constexpr int kTileDigitBits = 7;
constexpr int kTileDigits = 1 << kTileDigitBits;
constexpr int kTileKeyBits = 49;              // of the offsets' bits, under the 12 bits of a place in the window
constexpr int kTilePlaceBits = 12;
static_assert(kTileWindow == 1 << kTilePlaceBits && kTileKeyBits % kTileDigitBits == 0, "a key and a place in one word");

// The maps one set of launches takes: a network's pass makes the tiles of all its
// maps at once, because the sort of one keeps 8 to 40 of 256 compute units busy
// (the five maps of a network over 200 000 voxels: 156 us one after the other,
// 51 together).
constexpr int kTileJobs = 8;
struct TileJob {
  const int *dense;
  long long num_targets;
  int num_offsets, slots;
  int windows, window, per_window;
  int first_set, first_window, first_tile;     // workgroups of the jobs before
  int *rows, *counts, *offsets, *sources;
  unsigned *sets, *masks;
};
struct TileJobs {
  TileJob job[kTileJobs];
  int count;
};

__device__ __forceinline__ const TileJob &job_of(const TileJobs &jobs, int TileJob::*first) {
  int j = 0;
  while (j + 1 < jobs.count && static_cast<int>(blockIdx.x) >= jobs.job[j + 1].*first) ++j;
  return jobs.job[j];
}

// The set of offsets of every target, WORDS words of 32 each ([WORDS][T]).  In a
// launch of its own because it reads the whole dense map: the few workgroups
// that sort would take 10 us for it, bound by what one compute unit can load.
template <int WORDS>
__global__ __launch_bounds__(256) void tile_sets_kernel(const TileJobs jobs) {
  constexpr int kFlight = WORDS == 1 ? 27 : 16;
  const TileJob &job = job_of(jobs, &TileJob::first_set);
  const int *__restrict__ dense = job.dense;
  unsigned *__restrict__ sets = job.sets;
  const long long num_targets = job.num_targets;
  const int num_offsets = job.num_offsets;
  const long long t = static_cast<long long>(blockIdx.x - job.first_set) * 256 + threadIdx.x;
  const int *column = dense + min(t, num_targets - 1);
#pragma unroll
  for (int w = 0; w < WORDS; ++w) {
    const int o1 = min(num_offsets, 32 * (w + 1));
    unsigned set = 0;
    for (int o0 = 32 * w; o0 < o1; o0 += kFlight) {
      int entry[kFlight];
#pragma unroll
      for (int u = 0; u < kFlight; ++u) entry[u] = column[min(o0 + u, o1 - 1) * num_targets];
#pragma unroll
      for (int u = 0; u < kFlight; ++u) set |= (entry[u] >= 0 && o0 + u < o1 ? 1u : 0u) << ((o0 + u) & 31);
    }
    if (t < num_targets) sets[w * num_targets + t] = set;
  }
}

// One workgroup per window.  A target's set of offsets becomes a key of up to
// 49 bits, the rarest offset of the window on top: targets that have a rare
// neighbour stand together and the others need not carry that offset.  (Taken
// most frequent first, tiles of a LiDAR cloud have 1.8 times the live offsets.)
// Of more than 49 offsets those count that split the window most evenly.  The
// keys are sorted by their digits of 7 bits in LDS (stable: ties stay in the
// cloud's order, whose source rows are neighbours), ranks by one ballot per
// digit bit.  Each tile's number of live offsets then ranks the tiles, longest
// first, so that what runs last is short.
template <int WORDS>
struct TileSortLds {
  unsigned long long word[kTileWindow];
  unsigned mask[WORDS][kTileWindow];
  unsigned hist[kTileSortWaves][kTileDigits + 1];    // (+ 1: read down the wavefronts without conflicts)
  unsigned wave[kTileSortWaves];
  int count[kTileMaxOffsets];
  int chosen[kTileMaxOffsets];                       // offset of key bit k, from the top
  unsigned tile[kTileWindow / kTileTargets][WORDS];
  int live[kTileWindow / kTileTargets];
};

// ITEMS: the window's places in units of the block's threads.
template <int WORDS, int ITEMS>
__device__ __forceinline__ void tile_sort_body(const TileJob &job, TileSortLds<WORDS> &lds) {
  constexpr int kTileSortItems = ITEMS;
  const unsigned *__restrict__ sets = job.sets;
  const long long num_targets = job.num_targets;
  const int num_offsets = job.num_offsets, window = job.window, per_window = job.per_window;
  const int this_window = blockIdx.x - job.first_window;
  int *__restrict__ rows = job.rows;
  int *__restrict__ counts = job.counts;
  unsigned *__restrict__ masks = job.masks;
  unsigned long long *const s_word = lds.word;
  unsigned (*const s_mask)[kTileWindow] = lds.mask;
  unsigned (*const s_hist)[kTileDigits + 1] = lds.hist;
  unsigned *const s_wave = lds.wave;
  int *const s_count = lds.count, *const s_chosen = lds.chosen, *const s_live = lds.live;
  unsigned (*const s_tile)[WORDS] = lds.tile;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const long long first = static_cast<long long>(this_window) * window;
  const int here = static_cast<int>(min(static_cast<long long>(window), max(0ll, num_targets - first)));
  for (int i = tid; i < kTileMaxOffsets; i += kTileSortBlock) s_count[i] = 0;
  for (int i = tid; i < kTileWindow / kTileTargets * WORDS; i += kTileSortBlock) (&s_tile[0][0])[i] = 0u;
  __syncthreads();

  // place (wave * ITEMS + i) * 64 + lane of the window
  unsigned mask[kTileSortItems][WORDS];
  int place[kTileSortItems];
#pragma unroll
  for (int i = 0; i < kTileSortItems; ++i) {
    place[i] = wave * (kWave * kTileSortItems) + i * kWave + lane;
    const long long t = min(first + place[i], num_targets - 1);
#pragma unroll
    for (int w = 0; w < WORDS; ++w) mask[i][w] = sets[w * num_targets + t];
  }
#pragma unroll
  for (int i = 0; i < kTileSortItems; ++i) {
#pragma unroll
    for (int w = 0; w < WORDS; ++w) mask[i][w] = place[i] < here ? mask[i][w] : 0u;
  }
  // how many targets of the window use each offset
#pragma unroll
  for (int w = 0; w < WORDS; ++w) {
    int mine = 0;                                // lane b: offset 32 w + b
    for (int b = 0; b < min(32, num_offsets - 32 * w); ++b) {
      int found = 0;
#pragma unroll
      for (int i = 0; i < kTileSortItems; ++i) found += __popcll(__ballot((mask[i][w] >> b) & 1u));
      mine = lane == b ? found : mine;
    }
    if (lane < 32 && mine > 0) atomicAdd(&s_count[32 * w + lane], mine);
  }
#pragma unroll
  for (int i = 0; i < kTileSortItems; ++i) {
#pragma unroll
    for (int w = 0; w < WORDS; ++w) s_mask[w][place[i]] = mask[i][w];
  }
  __syncthreads();
  const int key_bits = min(num_offsets, kTileKeyBits);
  // ranks by comparing all pairs at once: a thread per pair, a vote per offset
  constexpr int kRankLanes = WORDS == 1 ? 32 : kWave;
  constexpr int kRankRows = kTileSortBlock / kRankLanes;
  constexpr int kRankMost = WORDS * 32;
  auto rank_by = [&](auto precedes, auto keep) {
    for (int o0 = 0; o0 < num_offsets; o0 += kRankRows) {
      const int o = o0 + tid / kRankLanes;
      int before = 0;
#pragma unroll
      for (int p0 = 0; p0 < kRankMost; p0 += kRankLanes) {
        const int p = p0 + tid % kRankLanes;
        const unsigned long long votes = __ballot(o < num_offsets && p < num_offsets && precedes(p, o));
        before += kRankLanes == kWave ? __popcll(votes) : __popc(static_cast<unsigned>(lane < 32 ? votes : votes >> 32));
      }
      if (tid % kRankLanes == 0 && o < num_offsets) keep(o, before);
    }
    __syncthreads();
  };
  if (num_offsets > kTileKeyBits) {
    auto off_half = [&](int o) { return abs(2 * s_count[o] - here); };
    rank_by([&](int p, int o) { return off_half(p) < off_half(o) || (off_half(p) == off_half(o) && p < o); },
            [&](int o, int before) { s_chosen[o] = before < key_bits ? s_count[o] : INT32_MAX; });
    if (tid < num_offsets) s_count[tid] = s_chosen[tid];
    __syncthreads();
  }
  rank_by([&](int p, int o) { return s_count[p] < s_count[o] || (s_count[p] == s_count[o] && p < o); },
          [&](int o, int before) { if (before < key_bits) s_chosen[before] = o; });

  unsigned long long word[kTileSortItems];
  {
    typedef typename std::conditional<WORDS == 1, unsigned, unsigned long long>::type Key;
    Key key[kTileSortItems];
#pragma unroll
    for (int i = 0; i < kTileSortItems; ++i) key[i] = 0;
    const int chosen = s_chosen[lane < key_bits ? lane : 0];
    for (int k = 0; k < key_bits; ++k) {
      const int o = __builtin_amdgcn_readlane(chosen, k);
#pragma unroll
      for (int i = 0; i < kTileSortItems; ++i) {
        unsigned m = mask[i][0];
#pragma unroll
        for (int w = 1; w < WORDS; ++w) m = (o >> 5) == w ? mask[i][w] : m;
        key[i] = (key[i] << 1) | ((m >> (o & 31)) & 1u);
      }
    }
    // ascending order of the inverted key; places past the window's end go last
#pragma unroll
    for (int i = 0; i < kTileSortItems; ++i) {
      const unsigned long long inverted = ~static_cast<unsigned long long>(key[i]) & ((1ull << key_bits) - 1ull);
      word[i] = place[i] < here ? (inverted << kTilePlaceBits) | static_cast<unsigned>(place[i]) : ~0ull;
    }
  }
  const int passes = (key_bits + kTileDigitBits - 1) / kTileDigitBits;
  for (int pass = 0; pass < passes; ++pass) {
    const int shift = kTilePlaceBits + pass * kTileDigitBits;
    for (int d = lane; d < kTileDigits; d += kWave) s_hist[wave][d] = 0u;
    __syncthreads();
    unsigned digit[kTileSortItems], at[kTileSortItems];
#pragma unroll
    for (int i = 0; i < kTileSortItems; ++i) {
      digit[i] = static_cast<unsigned>(word[i] >> shift) & (kTileDigits - 1);
      unsigned lo = ~0u, hi = ~0u;
#pragma unroll
      for (int b = 0; b < kTileDigitBits; ++b) {
        const unsigned set = static_cast<unsigned>(static_cast<int>(digit[i] << (31 - b)) >> 31);
        const unsigned long long votes = __ballot(set != 0u);
        lo &= ~(static_cast<unsigned>(votes) ^ set);
        hi &= ~(static_cast<unsigned>(votes >> 32) ^ set);
      }
      const unsigned long long peers = static_cast<unsigned long long>(hi) << 32 | lo;
      unsigned *mine = &s_hist[wave][digit[i]];
      const unsigned long long below = peers & lanes_below();
      at[i] = *mine + static_cast<unsigned>(__popcll(below));
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (below == 0ull) *mine += static_cast<unsigned>(__popcll(peers));
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    static_assert(kTileDigits * kTileSortWaves == 2 * kTileSortBlock && kTileSortWaves == 16, "two counts per thread");
    unsigned *const two_at = &s_hist[2 * (tid % 8)][tid / 8];
    const uint2 two = make_uint2(two_at[0], two_at[kTileDigits + 1]);
    unsigned inclusive = two.x + two.y;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const unsigned u = __shfl_up(inclusive, d);
      if (lane >= d) inclusive += u;
    }
    if (lane == kWave - 1) s_wave[wave] = inclusive;
    __syncthreads();
    unsigned before = 0;
#pragma unroll
    for (int w = 0; w < kTileSortWaves; ++w) before += w < wave ? s_wave[w] : 0u;
    const unsigned start = before + inclusive - two.x - two.y;
    two_at[0] = start;
    two_at[kTileDigits + 1] = start + two.x;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kTileSortItems; ++i) s_word[s_hist[wave][digit[i]] + at[i]] = word[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kTileSortItems; ++i) word[i] = s_word[place[i]];
  }

  // live offsets of every tile: place[i] is now the place in the sorted window
  int target[kTileSortItems];
#pragma unroll
  for (int i = 0; i < kTileSortItems; ++i) {
    target[i] = word[i] == ~0ull ? -1 : static_cast<int>(word[i] & (kTileWindow - 1));
#pragma unroll
    for (int w = 0; w < WORDS; ++w) {
      unsigned m = target[i] >= 0 ? s_mask[w][target[i]] : 0u;
#pragma unroll
      for (int d = 1; d < kWave; d <<= 1) m |= __shfl_xor(m, d);
      if (lane == 0 && m != 0u) atomicOr(&s_tile[place[i] / kTileTargets][w], m);
    }
  }
  __syncthreads();
  if (tid < per_window) {
    int live = 0;
#pragma unroll
    for (int w = 0; w < WORDS; ++w) live += __popc(s_tile[tid][w]);
    // targets without a single source still want their row written
    s_live[tid] = tid * kTileTargets < here ? max(live, 1) : 0;
  }
  __syncthreads();
  static_assert(kTileWindow / kTileTargets == 32 && kTileSortBlock == 32 * 32, "a thread per pair of tiles");
  {
    const int j = tid / 32, p = tid % 32;
    const bool in = j < per_window && p < per_window;
    const int mine = in ? s_live[j] : 0, theirs = in ? s_live[p] : 0;
    const unsigned long long votes = __ballot(in && (theirs > mine || (theirs == mine && p < j)));
    if (p == 0 && j < per_window) {
      const int longer = __popc(static_cast<unsigned>(lane < 32 ? votes : votes >> 32));
      const int tile = tile_number(job.windows, per_window, this_window, longer);
      counts[tile] = mine;
#pragma unroll
      for (int w = 0; w < WORDS; ++w) masks[tile * WORDS + w] = s_tile[j][w];
      s_count[j] = tile;
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kTileSortItems; ++i) {
    if (place[i] < window) {
      rows[static_cast<long long>(s_count[place[i] / kTileTargets]) * kTileTargets + place[i] % kTileTargets] =
          target[i] >= 0 ? static_cast<int>(first) + target[i] : -1;
    }
  }
}

template <int WORDS>
__global__ __launch_bounds__(kTileSortBlock) void tile_sort_kernel(const TileJobs jobs) {
  __shared__ TileSortLds<WORDS> lds;
  const TileJob &job = job_of(jobs, &TileJob::first_window);
  if (job.window <= kTileSortBlock) {
    tile_sort_body<WORDS, 1>(job, lds);
  } else if (job.window <= 2 * kTileSortBlock) {
    tile_sort_body<WORDS, 2>(job, lds);
  } else {
    tile_sort_body<WORDS, kTileWindow / kTileSortBlock>(job, lds);
  }
}

// The source rows of a tile's live offsets, one row of 128 entries after the
// other: a workgroup per tile, a thread per (target, every second live offset).
template <int WORDS>
__global__ __launch_bounds__(256) void tile_emit_kernel(const TileJobs jobs) {
  __shared__ int s_offset[kTileMaxOffsets];
  const TileJob &job = job_of(jobs, &TileJob::first_tile);
  const int *__restrict__ dense = job.dense;
  const long long num_targets = job.num_targets;
  const int num_offsets = job.num_offsets, slots = job.slots;
  const int *__restrict__ rows = job.rows;
  const int *__restrict__ counts = job.counts;
  const unsigned *__restrict__ masks = job.masks;
  int *__restrict__ offsets = job.offsets;
  int *__restrict__ sources = job.sources;
  const long long tile = blockIdx.x - job.first_tile;
  const int tid = threadIdx.x;
  const int live = counts[tile];
  const int row = rows[tile * kTileTargets + tid % kTileTargets];
  if (live == 0) return;
  if (tid < num_offsets) {
    int before = 0;
    bool set = false;
#pragma unroll
    for (int w = 0; w < WORDS; ++w) {
      const unsigned m = masks[tile * WORDS + w];
      if (w < (tid >> 5)) {
        before += __popc(m);
      } else if (w == (tid >> 5)) {
        before += __popc(m & ((1u << (tid & 31)) - 1u));
        set = (m >> (tid & 31)) & 1u;
      }
    }
    if (set) {
      s_offset[before] = tid;
      offsets[tile * slots + before] = tid;
    }
  }
  if (tid == 0 && live == 1) {                   // the one offset may be nobody's
    unsigned any = 0;
#pragma unroll
    for (int w = 0; w < WORDS; ++w) any |= masks[tile * WORDS + w];
    if (any == 0) {
      s_offset[0] = 0;
      offsets[tile * slots] = 0;
    }
  }
  __syncthreads();
  int *to = sources + tile * slots * kTileTargets + tid % kTileTargets;
  constexpr int kFlight = 8;
  for (int s0 = tid / kTileTargets; s0 < live; s0 += 2 * kFlight) {
    int v[kFlight];
#pragma unroll
    for (int u = 0; u < kFlight; ++u) {
      const int s = s0 + 2 * u;
      v[u] = -1;
      if (s < live && row >= 0) v[u] = dense[static_cast<long long>(s_offset[s]) * num_targets + row];
    }
#pragma unroll
    for (int u = 0; u < kFlight; ++u) {
      if (s0 + 2 * u < live) to[(s0 + 2 * u) * kTileTargets] = v[u];
    }
  }
}

struct TileRequest {
  const int *dense;
  int64_t num_targets, num_offsets;
  int *out;
};

// The requests' maps have all up to 32 offsets, or all more.
template <int WORDS>
static void build_tiles(const TileRequest *requests, int count, hipStream_t stream) {
  Scope scope(stream);
  for (int from = 0; from < count; from += kTileJobs) {
    TileJobs jobs = {};
    jobs.count = std::min(kTileJobs, count - from);
    int64_t set_blocks = 0, windows = 0, tiles = 0;
    for (int j = 0; j < jobs.count; ++j) {
      const TileRequest &r = requests[from + j];
      const TileLayout l(r.num_targets, r.num_offsets);
      TileJob &job = jobs.job[j];
      job.dense = r.dense;
      job.num_targets = r.num_targets;
      job.num_offsets = static_cast<int>(r.num_offsets);
      job.slots = l.slots;
      job.windows = l.windows;
      job.window = l.window;
      job.per_window = l.per_window;
      job.first_set = static_cast<int>(set_blocks);
      job.first_window = static_cast<int>(windows);
      job.first_tile = static_cast<int>(tiles);
      job.rows = r.out;
      job.counts = r.out + l.counts_at;
      job.offsets = r.out + l.offsets_at;
      job.sources = r.out + l.sources_at;
      job.sets = scope.alloc<unsigned>(static_cast<size_t>(r.num_targets) * WORDS);
      job.masks = scope.alloc<unsigned>(static_cast<size_t>(l.tiles) * WORDS);
      set_blocks += div_ceil(r.num_targets, int64_t{256});
      windows += l.windows;
      tiles += l.tiles;
    }
    MNT_CHECK(set_blocks <= INT32_MAX, "tiles of %lld targets at once", (long long)(set_blocks * 256));
    tile_sets_kernel<WORDS><<<static_cast<unsigned>(set_blocks), 256, 0, stream>>>(jobs);
    check_launch("tile_sets_kernel");
    tile_sort_kernel<WORDS><<<static_cast<unsigned>(windows), kTileSortBlock, 0, stream>>>(jobs);
    check_launch("tile_sort_kernel");
    tile_emit_kernel<WORDS><<<static_cast<unsigned>(tiles), 256, 0, stream>>>(jobs);
    check_launch("tile_emit_kernel");
  }
}

static void check_tiles(const TileRequest &r) {
  MNT_CHECK(r.num_targets >= 1 && r.num_targets <= INT32_MAX && r.num_offsets >= 1 && r.num_offsets <= kTileMaxOffsets,
            "no tiles for %lld targets under %lld offsets (at most %d)", (long long)r.num_targets,
            (long long)r.num_offsets, kTileMaxOffsets);
  MNT_CHECK(r.dense != nullptr && r.out != nullptr, "null operand");
  MNT_CHECK(reinterpret_cast<uintptr_t>(r.out) % 16 == 0, "tiles are not 16-byte aligned");
}

}  // namespace mnt

using namespace mnt;

extern "C" int mnt_kernel_map_tiles_size(int64_t num_targets, int64_t num_offsets, int64_t *ints_out) {
  return guarded([&] {
    MNT_CHECK(num_targets >= 0 && num_targets <= INT32_MAX && num_offsets >= 1 && num_offsets <= kTileMaxOffsets,
              "no tiles for %lld targets under %lld offsets (at most %d)", (long long)num_targets,
              (long long)num_offsets, kTileMaxOffsets);
    *ints_out = TileLayout(num_targets, num_offsets).ints;
  });
}

extern "C" int mnt_kernel_map_tiles_batch(int64_t num_maps, const int32_t *const *kernel_maps,
                                          const int64_t *num_targets, const int64_t *num_offsets,
                                          int32_t *const *tiles_out, void *stream_) {
  return guarded([&] {
    MNT_CHECK(num_maps >= 0 && num_maps <= 65536, "tiles of %lld maps", (long long)num_maps);
    std::vector<TileRequest> few, many;
    for (int64_t i = 0; i < num_maps; ++i) {
      const TileRequest r = {kernel_maps[i], num_targets[i], num_offsets[i], tiles_out[i]};
      check_tiles(r);
      (r.num_offsets <= 32 ? few : many).push_back(r);
    }
    build_tiles<1>(few.data(), static_cast<int>(few.size()), static_cast<hipStream_t>(stream_));
    build_tiles<4>(many.data(), static_cast<int>(many.size()), static_cast<hipStream_t>(stream_));
  });
}

extern "C" int mnt_kernel_map_tiles(const int32_t *kernel_map, int64_t num_targets, int64_t num_offsets,
                                    int32_t *tiles_out, void *stream_) {
  return mnt_kernel_map_tiles_batch(1, &kernel_map, &num_targets, &num_offsets, &tiles_out, stream_);
}
