// The coordinate levels and kernel maps of a whole pass in one build.
//
// A network's maps are many and small: of the UNet on two LiDAR scans, four
// strided levels, nine maps, three sets of offset groups and two sets of rank
// tables were 66 launches of 2 to 30 us with a wait on the host per level and
// per table, each behind every layer enqueued before it.  Built together they
// are about ten launches and one wait at the start of the pass (measured with
// the layers that follow: 2.16 -> 1.69 ms for that network):
//
//   pass_mark_kernel     every source row sets its bit in the bitmap of every
//                        level (a level's cell is floor(c / stride) of the
//                        input row itself: nested floors of multiples agree);
//   pass_sums_kernel     set bits per tile of 2 048 bitmap words, all levels;
//   pass_scan_kernel     their prefix, the level counts go to the host;
//   -- the host lays out the results --
//   pass_emit_kernel     rows and batch boundaries of all levels in key order;
//                        clears the bitmaps; further workgroups fill with -1
//                        what the next launches write only in part;
//   pass_parents_kernel  maps of strided layers whose offsets tile the cell
//                        (a 2 x 2 x 2 kernel of stride 2): every source has one
//                        parent, whose row is the rank of its bit; dense map
//                        and inverse are written by the source, no search;
//   query_kernel         all other maps in one launch (enqueue_queries);
//   then offset groups and rank tables, each step once for all maps.
#include <algorithm>

#include "device_utils.h"
#include "pass.h"
#include "sort.h"
#include "target_keys.h"

namespace mnt {

constexpr int kPassLevels = 6;            // strided levels
constexpr int kPassFills = 2 * kPassMaps;
constexpr int kPassParents = 8;           // parent maps of one launch
constexpr int kParentOffsets = 8;
constexpr int kPassCarried = 640;         // table ints that ride the marking launch
constexpr int kPassTableInts = 4096;      // room for tables in the pass block

struct PassSpecs {
  int count;
  TargetSpec spec[kPassLevels];
  int tile_start[kPassLevels + 1];        // first bitmap tile of each level
};
struct PassCarried {
  int count;
  int v[kPassCarried];
};

// A level per row of the grid: one after the other, four levels of 12 000 rows
// took 8.9 us of a launch that is all latency, and side by side 5.3.
template <typename CT, typename IT>
__global__ __launch_bounds__(256) void pass_mark_kernel(const CT *__restrict__ coords, long long n, PassSpecs specs,
                                                        const IT *__restrict__ batch_dims,
                                                        unsigned *__restrict__ bitmap, PassCarried carried,
                                                        int *__restrict__ tables) {
  const int l = blockIdx.y;
  if (blockIdx.x == 0 && l == 0) {
    for (int i = threadIdx.x; i < carried.count; i += 256) tables[i] = carried.v[i];
  }
  if (l >= specs.count) return;
  mark_rows<CT, IT>(coords, n, specs.spec[l], batch_dims,
                    bitmap + static_cast<long long>(specs.tile_start[l]) * kBitmapTile);
}

__global__ __launch_bounds__(kScanBlock) void pass_sums_kernel(const unsigned *__restrict__ bitmap,
                                                               unsigned *__restrict__ tile_sums) {
  const long long base = static_cast<long long>(blockIdx.x) * kBitmapTile + threadIdx.x * 4;
  unsigned count = 0;
#pragma unroll
  for (int r = 0; r < kBitmapWords / 4; ++r) {
    const uint4 w = *reinterpret_cast<const uint4 *>(bitmap + base + r * (kScanBlock * 4));
    count += __popc(w.x) + __popc(w.y) + __popc(w.z) + __popc(w.w);
  }
  unsigned total;
  block_exclusive_scan(count, &total);
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

// One workgroup: exclusive scan of the tile sums of all levels in place (one
// more entry takes the total), then the levels' row counts for the host.
__global__ __launch_bounds__(1024) void pass_scan_kernel(unsigned *__restrict__ tile_sums, PassSpecs specs,
                                                         unsigned *host_counts, unsigned long long *flag,
                                                         unsigned long long sequence) {
  __shared__ unsigned s_start[kPassLevels + 1];
  const int tiles = specs.tile_start[specs.count];
  scan_in_place(tile_sums, tiles);
  __syncthreads();
  const int t = threadIdx.x;
  if (t <= specs.count) s_start[t] = tile_sums[specs.tile_start[t]];
  __syncthreads();
  if (t < specs.count) host_counts[t] = s_start[t + 1] - s_start[t];
  if (t == 0) {
    __threadfence_system();
    __hip_atomic_store(flag, sequence, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

struct PassOut {
  void *coords[kPassLevels];
  void *batch_dims[kPassLevels];
};
struct PassFills {
  int count;
  int *data[kPassFills];                  // 16-byte aligned
  long long n[kPassFills];
  int first_block[kPassFills + 1];
};
constexpr int kFillPerBlock = 8192;
static_assert(kFillPerBlock % (4 * kEmitBlock) == 0, "whole rounds");

// The word's bits and the rank of its first row, for the rank of any set bit.
template <typename CT, typename IT>
__global__ __launch_bounds__(kEmitBlock) void pass_emit_kernel(unsigned *__restrict__ bitmap,
                                                               const unsigned *__restrict__ tile_bases,
                                                               PassSpecs specs, PassOut outs,
                                                               uint2 *__restrict__ word_info, PassFills fills) {
  const int tiles = specs.tile_start[specs.count];
  if (static_cast<int>(blockIdx.x) >= tiles) {
    const int b = static_cast<int>(blockIdx.x) - tiles;
    int f = 0;
    while (f + 1 < fills.count && fills.first_block[f + 1] <= b) ++f;
    int *data = fills.data[f];
    const long long n = fills.n[f];
    const long long from = static_cast<long long>(b - fills.first_block[f]) * kFillPerBlock;
#pragma unroll
    for (int r = 0; r < kFillPerBlock / (4 * kEmitBlock); ++r) {
      const long long i = from + (r * kEmitBlock + threadIdx.x) * 4;
      if (i + 4 <= n) {
        *reinterpret_cast<int4 *>(data + i) = make_int4(-1, -1, -1, -1);
      } else {
        for (int k = 0; k < 4; ++k) {
          if (i + k < n) data[i + k] = -1;
        }
      }
    }
    return;
  }
  int l = 0;
  while (l + 1 < specs.count && specs.tile_start[l + 1] <= static_cast<int>(blockIdx.x)) ++l;
  const int first_tile = specs.tile_start[l];
  const unsigned level_base = tile_bases[first_tile];
  emit_bitmap_tile<CT, IT>(bitmap + static_cast<long long>(first_tile) * kBitmapTile,
                           static_cast<long long>(specs.tile_start[l + 1] - first_tile) * kBitmapTile,
                           static_cast<int>(blockIdx.x) - first_tile, tile_bases[blockIdx.x] - level_base,
                           tile_bases[blockIdx.x + 1] - level_base,
                           tile_bases[specs.tile_start[l + 1]] - level_base, specs.spec[l],
                           static_cast<CT *>(outs.coords[l]), static_cast<IT *>(outs.batch_dims[l]),
                           word_info + static_cast<long long>(first_tile) * kBitmapTile);
}

struct ParentJob {
  const void *sources;
  const void *batch_dims;
  int *dense, *inverse;                   // [O, T] (-1 already), [O, S] (nullable)
  int num_sources, num_targets, first_block, level, num_offsets;
  int offsets[kParentOffsets][MNT_MAX_NDIM];
};
struct ParentJobs {
  int count;
  ParentJob job[kPassParents];
};
constexpr int kParentBlock = 256;

template <typename CT, typename IT>
__global__ __launch_bounds__(kParentBlock) void pass_parents_kernel(ParentJobs jobs, PassSpecs specs,
                                                                    const uint2 *__restrict__ word_info) {
  int j = 0;
  while (j + 1 < jobs.count && jobs.job[j + 1].first_block <= static_cast<int>(blockIdx.x)) ++j;
  const ParentJob &job = jobs.job[j];
  const TargetSpec &spec = specs.spec[job.level];
  const long long s = static_cast<long long>(static_cast<int>(blockIdx.x) - job.first_block) * kParentBlock + threadIdx.x;
  if (s >= job.num_sources) return;
  const CT *row = static_cast<const CT *>(job.sources) + s * spec.ndim;
  long long c[MNT_MAX_NDIM], behind[MNT_MAX_NDIM];
  load_row<CT>(row, spec.ndim, c);
  load_row<CT>(s + 1 < job.num_sources ? row + spec.ndim : row, spec.ndim, behind);
  // of equal rows (a cloud should have none) the last one is the hit, as in query_kernel
  bool repeated = s + 1 < job.num_sources;
  long long rest[MNT_MAX_NDIM];
  unsigned long long key = 0;
#pragma unroll
  for (int k = 0; k < MNT_MAX_NDIM; ++k) {
    rest[k] = 0;
    if (k < spec.ndim) {
      repeated = repeated && behind[k] == c[k];
      const long long cell = cell_of(c[k], spec, k);
      rest[k] = c[k] - cell * spec.stride[k];
      key |= (static_cast<unsigned long long>(cell - spec.base[k]) & spec.mask[k]) << spec.shift[k];
    }
  }
  if (spec.num_batches > 0) {
    const IT *dims = static_cast<const IT *>(job.batch_dims);
    const int batch = batch_of<IT>(s, dims, spec.num_batches);
    key |= static_cast<unsigned long long>(batch) << spec.batch_shift;
    if (repeated) repeated = static_cast<long long>(dims[batch + 1]) != s + 1;
  }
  const uint2 info = word_info[static_cast<long long>(specs.tile_start[job.level]) * kBitmapTile +
                               static_cast<long long>(key >> 5)];
  const int t = static_cast<int>(info.y + __popc(info.x & ((1u << (key & 31u)) - 1u)));
  int hit = -1;
  for (int o = 0; o < job.num_offsets; ++o) {
    bool same = true;
#pragma unroll
    for (int k = 0; k < MNT_MAX_NDIM; ++k) same = same && (k >= spec.ndim || rest[k] == job.offsets[o][k]);
    hit = same ? o : hit;
  }
  if (repeated) hit = -1;
  if (hit >= 0) job.dense[static_cast<long long>(hit) * job.num_targets + t] = static_cast<int>(s);
  if (job.inverse != nullptr) {
    for (int o = 0; o < job.num_offsets; ++o) {
      job.inverse[static_cast<long long>(o) * job.num_sources + s] = o == hit ? t : -1;
    }
  }
}

// inverse of the maps that are looked up: everything -1 before
struct InvertJob {
  const int *dense;
  int *inverse;
  int num_sources, num_targets, first_block;
  long long total;
};
struct InvertJobs {
  int count;
  InvertJob job[kPassMaps];
};

__global__ __launch_bounds__(256) void pass_invert_kernel(InvertJobs jobs) {
  int j = 0;
  while (j + 1 < jobs.count && jobs.job[j + 1].first_block <= static_cast<int>(blockIdx.x)) ++j;
  const InvertJob &job = jobs.job[j];
  const long long i = static_cast<long long>(static_cast<int>(blockIdx.x) - job.first_block) * 256 + threadIdx.x;
  if (i >= job.total) return;
  const int m = job.dense[i];
  if (m >= 0) {
    const long long o = i / job.num_targets;
    job.inverse[o * job.num_sources + m] = static_cast<int>(i - o * job.num_targets);
  }
}

// ------------------------------------------------------------------ host ----

// What mnt_pass_levels leaves for mnt_pass_build (kept in the arena's map
// state: any other map build in between forgets it).
struct PassState {
  const void *coords, *levels, *maps;              // whose state this is
  PassSpecs specs;
  int64_t n, num_batches;
  int ndim, coord_dtype, index_dtype, num_levels, num_maps;
  std::vector<QueryTables> plans;
  std::vector<int> tables_at, plan_of, parent;     // per map: its query plan (-1: none), whether it is a parent map
};

// One state per stream; guarded like the arena it belongs to (one caller thread per stream).
static PassState &pass_state(Arena &arena) {
  if (!arena.pass_state) arena.pass_state = std::make_shared<PassState>();
  return *static_cast<PassState *>(arena.pass_state.get());
}

// device block of the pass builder: tables, then the words' ranks
constexpr size_t kPassTableBytes = kPassTableInts * sizeof(int);

static int64_t take_bytes(int64_t &total, int64_t bytes) {
  const int64_t at = total;
  total += (std::max<int64_t>(bytes, 1) + 255) / 256 * 256;
  return at;
}

static bool offsets_tile_the_cell(const mnt_pass_map &m, const int64_t *target_stride, int ndim) {
  if (m.num_offsets < 1 || m.num_offsets > kParentOffsets) return false;
  for (int64_t o = 0; o < m.num_offsets; ++o) {
    for (int k = 0; k < ndim; ++k) {
      const int64_t d = m.offsets_host[o * ndim + k];
      if (d < 0 || d >= target_stride[k]) return false;
    }
    for (int64_t p = 0; p < o; ++p) {
      bool same = true;
      for (int k = 0; k < ndim; ++k) same = same && m.offsets_host[o * ndim + k] == m.offsets_host[p * ndim + k];
      if (same) return false;
    }
  }
  return true;
}

template <typename CT, typename IT>
static void launch_marks(const CT *coords, const IT *batch_dims, const PassState &state, unsigned *bitmap,
                         unsigned *tile_sums, const PassCarried &carried, int *tables, unsigned *host_counts,
                         unsigned long long *flag, unsigned long long sequence, hipStream_t stream) {
  const int tiles = state.specs.tile_start[state.specs.count];
  const dim3 marks(grid_for(state.n, 256, 2048), std::max(1, state.specs.count));
  pass_mark_kernel<CT, IT><<<marks, 256, 0, stream>>>(coords, state.n, state.specs, batch_dims,
                                                                           bitmap, carried, tables);
  check_launch("pass_mark_kernel");
  pass_sums_kernel<<<tiles, kScanBlock, 0, stream>>>(bitmap, tile_sums);
  check_launch("pass_sums_kernel");
  pass_scan_kernel<<<1, 1024, 0, stream>>>(tile_sums, state.specs, host_counts, flag, sequence);
  check_launch("pass_scan_kernel");
}

static bool levels_supported(const void *coords, const void *batch_dims, const long long *bounds,
                             mnt_pass_level *levels, mnt_pass_map *maps, PassState &state, int64_t *total_out,
                             hipStream_t stream) {
  Arena &arena = Arena::of(stream);
  const int ndim = state.ndim;
  const bool batched = batch_dims != nullptr && state.num_batches > 1;
  PassSpecs &specs = state.specs;
  memset(&specs, 0, sizeof(specs));
  specs.count = state.num_levels;
  std::vector<long long> level_bounds(static_cast<size_t>(state.num_levels + 1) * 8);
  for (int i = 0; i < 8; ++i) level_bounds[i] = bounds[i];
  long long tiles = 0;
  for (int l = 0; l < state.num_levels; ++l) {
    int64_t stride[MNT_MAX_NDIM];
    for (int k = 0; k < ndim; ++k) stride[k] = levels[l].stride[k];
    const int bits = make_target_spec(bounds, stride, ndim, batched ? state.num_batches : 0, specs.spec[l]);
    if (bits > kBitmapMaxBits) return false;
    specs.tile_start[l] = static_cast<int>(tiles);
    tiles += div_ceil(bits <= 5 ? 1 : (1ll << (bits - 5)), kBitmapTile);
    long long *b = &level_bounds[static_cast<size_t>(l + 1) * 8];
    for (int k = 0; k < ndim; ++k) {
      b[k] = host_floor_div(bounds[k], stride[k]) * stride[k];
      b[MNT_MAX_NDIM + k] = host_floor_div(bounds[MNT_MAX_NDIM + k], stride[k]) * stride[k];
    }
  }
  if (tiles > kBitmapMaxTiles) return false;
  for (int l = state.num_levels; l <= kPassLevels; ++l) specs.tile_start[l] = static_cast<int>(tiles);

  // plans of the maps that are looked up
  state.plans.clear();
  state.tables_at.clear();
  state.plan_of.assign(state.num_maps, -1);
  state.parent.assign(state.num_maps, 0);
  std::vector<int> ints;
  int parents = 0;
  for (int i = 0; i < state.num_maps; ++i) {
    const mnt_pass_map &m = maps[i];
    if (m.target_level > 0 && parents < kPassParents &&
        offsets_tile_the_cell(m, levels[m.target_level - 1].stride, ndim)) {
      bool nested = true;
      if (m.source_level > 0) {
        for (int k = 0; k < ndim; ++k) {
          nested = nested && levels[m.target_level - 1].stride[k] % levels[m.source_level - 1].stride[k] == 0;
        }
      }
      if (nested) {
        state.parent[i] = 1;
        ++parents;
        continue;
      }
    }
    QueryTables t = make_query_tables(&level_bounds[static_cast<size_t>(m.source_level) * 8],
                                      &level_bounds[static_cast<size_t>(m.target_level) * 8], m.offsets_host,
                                      m.num_offsets, ndim, batched ? state.num_batches : 1);
    if (t.ints.empty() || t.ints.size() * sizeof(int) > 20 * 1024) return false;
    state.plan_of[i] = static_cast<int>(state.plans.size());
    state.tables_at.push_back(static_cast<int>(ints.size()));
    ints.insert(ints.end(), t.ints.begin(), t.ints.end());
    while (ints.size() % 4 != 0) ints.push_back(0);
    state.plans.push_back(std::move(t));
  }
  if (ints.size() > static_cast<size_t>(kPassTableInts)) return false;

  const size_t words = static_cast<size_t>(tiles) * kBitmapTile;
  char *block = static_cast<char *>(arena.persistent(2, kPassTableBytes + words * sizeof(uint2)));
  int *tables = reinterpret_cast<int *>(block);
  PassCarried carried;
  carried.count = 0;
  if (state.num_levels > 0 && ints.size() <= static_cast<size_t>(kPassCarried)) {
    carried.count = static_cast<int>(ints.size());
    memcpy(carried.v, ints.data(), ints.size() * sizeof(int));
  } else if (!ints.empty()) {
    upload_ints(ints, tables, stream);
  }
  if (state.num_levels > 0) {
    char *keep = static_cast<char *>(arena.persistent(0, kBitmapBasesBytes + words * 4));
    unsigned *tile_sums = reinterpret_cast<unsigned *>(keep);
    unsigned *bitmap = reinterpret_cast<unsigned *>(keep + kBitmapBasesBytes);
    const long long zero_words = arena.zero_bitmap_words;
    if (zero_words < static_cast<long long>(words)) MNT_HIP(hipMemsetAsync(bitmap, 0, words * 4, stream));
    arena.zero_bitmap_words = 0;                   // until the walk of mnt_pass_build is launched
    arena.zero_bitmap_words_after = std::max(zero_words, static_cast<long long>(words));
    volatile unsigned *h = reinterpret_cast<volatile unsigned *>(static_cast<char *>(arena.pinned()) + 256);
    unsigned *d = reinterpret_cast<unsigned *>(static_cast<char *>(arena.pinned_device()) + 256);
    const unsigned long long sequence = arena.next_sequence();
#define MNT_CALL(CT, IT)                                                                                          \
  launch_marks<CT, IT>(static_cast<const CT *>(coords), batched ? static_cast<const IT *>(batch_dims) : nullptr,   \
                       state, bitmap, tile_sums, carried, tables, d, arena.flag_device(2), sequence, stream)
    MNT_DISPATCH_CI(state.coord_dtype, state.index_dtype, MNT_CALL);
#undef MNT_CALL
    arena.wait_flag(2, sequence);
    for (int l = 0; l < state.num_levels; ++l) levels[l].count = static_cast<int64_t>(h[l]);
  }

  // where everything goes
  const int csz = int_size(state.coord_dtype), isz = int_size(state.index_dtype);
  int64_t total = 0;
  for (int l = 0; l < state.num_levels; ++l) {
    levels[l].coords_at = take_bytes(total, levels[l].count * ndim * csz);
    levels[l].batch_dims_at = batched ? take_bytes(total, (state.num_batches + 1) * isz) : -1;
  }
  for (int i = 0; i < state.num_maps; ++i) {
    mnt_pass_map &m = maps[i];
    m.num_sources = m.source_level == 0 ? state.n : levels[m.source_level - 1].count;
    m.num_targets = m.target_level == 0 ? state.n : levels[m.target_level - 1].count;
    const int64_t pairs = m.num_offsets * m.num_targets * 4, back = m.num_offsets * m.num_sources * 4;
    for (int64_t &at : m.at) at = -1;
    m.at[0] = take_bytes(total, pairs);
    if (m.want & MNT_PASS_INVERSE) m.at[1] = take_bytes(total, back);
    if (m.want & MNT_PASS_GROUPS) {
      m.at[2] = take_bytes(total, 9 * m.num_targets * 4);
      m.at[3] = take_bytes(total, 9 * m.num_targets * 16);
      m.at[4] = take_bytes(total, 64);
    }
    if (m.want & MNT_PASS_TABLES) {
      m.at[5] = take_bytes(total, back);
      m.at[6] = take_bytes(total, pairs);
      // a parent map has one hit per source at most
      const int64_t hits = state.parent[i] ? m.num_sources * 4 : pairs;
      m.at[7] = take_bytes(total, hits);
      m.at[8] = take_bytes(total, hits);
      m.at[9] = take_bytes(total, m.num_offsets * 4);
      m.at[10] = take_bytes(total, m.num_offsets * 4);
    }
  }
  *total_out = total;
  return true;
}

template <typename CT, typename IT>
static void launch_levels(const PassState &state, unsigned *bitmap, const unsigned *tile_bases, const PassOut &outs,
                          uint2 *word_info, const PassFills &fills, const ParentJobs &parents, int parent_blocks,
                          hipStream_t stream) {
  const int tiles = state.specs.tile_start[state.specs.count];
  const int blocks = tiles + fills.first_block[fills.count];
  if (blocks > 0) {
    pass_emit_kernel<CT, IT><<<blocks, kEmitBlock, 0, stream>>>(bitmap, tile_bases, state.specs, outs, word_info, fills);
    check_launch("pass_emit_kernel");
  }
  if (parent_blocks > 0) {
    pass_parents_kernel<CT, IT><<<parent_blocks, kParentBlock, 0, stream>>>(parents, state.specs, word_info);
    check_launch("pass_parents_kernel");
  }
}

static void build_pass(const void *coords, const void *batch_dims, mnt_pass_level *levels, mnt_pass_map *maps,
                       char *base, PassState &state, hipStream_t stream) {
  Arena &arena = Arena::of(stream);
  Scope scope(stream);
  const bool batched = batch_dims != nullptr && state.num_batches > 1;
  auto level_coords = [&](int l) -> void * { return l == 0 ? const_cast<void *>(coords) : base + levels[l - 1].coords_at; };
  auto level_dims = [&](int l) -> void * {
    return !batched ? nullptr : l == 0 ? const_cast<void *>(batch_dims) : base + levels[l - 1].batch_dims_at;
  };
  auto ints_at = [&](int64_t at) { return at < 0 ? nullptr : reinterpret_cast<int *>(base + at); };

  PassOut outs;
  memset(&outs, 0, sizeof(outs));
  for (int l = 0; l < state.num_levels; ++l) {
    outs.coords[l] = level_coords(l + 1);
    outs.batch_dims[l] = level_dims(l + 1);
  }
  PassFills fills;
  memset(&fills, 0, sizeof(fills));
  auto fill = [&](int *data, int64_t n) {
    if (data == nullptr || n <= 0) return;
    fills.data[fills.count] = data;
    fills.n[fills.count] = n;
    fills.first_block[fills.count + 1] = fills.first_block[fills.count] + static_cast<int>(div_ceil(n, kFillPerBlock));
    ++fills.count;
  };
  ParentJobs parents;
  memset(&parents, 0, sizeof(parents));
  InvertJobs inverts;
  memset(&inverts, 0, sizeof(inverts));
  int parent_blocks = 0, invert_blocks = 0;
  std::vector<QueryWork> queries;
  std::vector<GroupWork> groups;
  std::vector<TableWork> tables;
  for (int i = 0; i < state.num_maps; ++i) {
    const mnt_pass_map &m = maps[i];
    int *dense = ints_at(m.at[0]);
    if (m.num_targets > 0 && m.num_sources > 0) {
      if (state.parent[i]) {
        fill(dense, m.num_offsets * m.num_targets);
        ParentJob &job = parents.job[parents.count++];
        job.sources = level_coords(m.source_level);
        job.batch_dims = level_dims(m.source_level);
        job.dense = dense;
        job.inverse = ints_at(m.at[1]);
        job.num_sources = static_cast<int>(m.num_sources);
        job.num_targets = static_cast<int>(m.num_targets);
        job.first_block = parent_blocks;
        job.level = m.target_level - 1;
        job.num_offsets = static_cast<int>(m.num_offsets);
        for (int64_t o = 0; o < m.num_offsets; ++o) {
          for (int k = 0; k < state.ndim; ++k) job.offsets[o][k] = static_cast<int>(m.offsets_host[o * state.ndim + k]);
        }
        parent_blocks += static_cast<int>(div_ceil(m.num_sources, kParentBlock));
      } else {
        queries.push_back({level_coords(m.source_level), level_coords(m.target_level), level_dims(m.source_level),
                           level_dims(m.target_level), m.num_sources, m.num_targets, dense, state.plan_of[i]});
        if (m.at[1] >= 0) {
          fill(ints_at(m.at[1]), m.num_offsets * m.num_sources);
          InvertJob &job = inverts.job[inverts.count++];
          job.dense = dense;
          job.inverse = ints_at(m.at[1]);
          job.num_sources = static_cast<int>(m.num_sources);
          job.num_targets = static_cast<int>(m.num_targets);
          job.first_block = invert_blocks;
          job.total = m.num_offsets * m.num_targets;
          invert_blocks += static_cast<int>(div_ceil(job.total, 256));
        }
      }
    }
    if (m.want & MNT_PASS_GROUPS) {
      groups.push_back({dense, static_cast<int>(m.num_targets), m.group_offsets_host, ints_at(m.at[2]),
                        ints_at(m.at[3]), ints_at(m.at[4])});
    }
    if (m.want & MNT_PASS_TABLES) {
      fill(ints_at(m.at[5]), m.num_offsets * m.num_sources);
      tables.push_back({dense, static_cast<int>(m.num_sources), static_cast<int>(m.num_targets),
                        static_cast<int>(m.num_offsets), m.reorder, ints_at(m.at[5]), ints_at(m.at[6]),
                        ints_at(m.at[7]), ints_at(m.at[8]), ints_at(m.at[9]), ints_at(m.at[10]), 0});
    }
  }
  char *block = static_cast<char *>(arena.persistent(2, 0));
  const int *d_tables = reinterpret_cast<const int *>(block);
  uint2 *word_info = reinterpret_cast<uint2 *>(block + kPassTableBytes);
  char *keep = static_cast<char *>(arena.persistent(0, 0));
  const unsigned *tile_bases = reinterpret_cast<const unsigned *>(keep);
  unsigned *bitmap = reinterpret_cast<unsigned *>(keep + kBitmapBasesBytes);
#define MNT_CALL(CT, IT) \
  launch_levels<CT, IT>(state, bitmap, tile_bases, outs, word_info, fills, parents, parent_blocks, stream)
  MNT_DISPATCH_CI(state.coord_dtype, state.index_dtype, MNT_CALL);
#undef MNT_CALL
  if (state.num_levels > 0) arena.zero_bitmap_words = arena.zero_bitmap_words_after;
  profile_mark("pass_levels", stream);
  enqueue_queries(queries, state.plans, state.tables_at, d_tables, state.ndim, state.coord_dtype, state.index_dtype,
                  batched ? state.num_batches : 1, stream);
  if (invert_blocks > 0) {
    pass_invert_kernel<<<invert_blocks, 256, 0, stream>>>(inverts);
    check_launch("pass_invert_kernel");
  }
  profile_mark("pass_queries", stream);
  if (!groups.empty()) enqueue_offset_groups(groups, scope, stream);
  if (!tables.empty()) {
    const unsigned long long sequence = arena.next_sequence();
    enqueue_tables(tables, scope, sequence, stream);
    size_t next = 0;
    for (int i = 0; i < state.num_maps; ++i) {
      if (maps[i].want & MNT_PASS_TABLES) {
        collect_tables(tables[next++], arena, sequence, maps[i].sizes_host, maps[i].order_host);
      }
    }
  }
  profile_mark("pass_tables", stream);
}

}  // namespace mnt

using namespace mnt;

extern "C" int mnt_pass_levels(const void *coords, int64_t n, int ndim, int coord_dtype, const void *batch_dims,
                               int64_t num_batches, int index_dtype, const int64_t *bounds_host,
                               mnt_pass_level *levels, int num_levels, mnt_pass_map *maps, int num_maps,
                               int64_t *bounds_host_out, int64_t *total_bytes_out, int *supported_out,
                               void *stream_) {
  return guarded([&] {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MNT_CHECK(ndim >= 1 && ndim <= MNT_MAX_NDIM, "ndim must be in [1, %d] but found %d", MNT_MAX_NDIM, ndim);
    MNT_CHECK(n > 0 && n <= INT32_MAX, "number of coordinates %lld out of range", static_cast<long long>(n));
    MNT_CHECK(coords != nullptr && total_bytes_out != nullptr && supported_out != nullptr, "null argument");
    MNT_CHECK(num_levels >= 0 && num_maps >= 0 && (num_levels == 0 || levels != nullptr) &&
                  (num_maps == 0 || maps != nullptr),
              "bad lists of levels and maps");
    int_size(coord_dtype);
    int_size(index_dtype);
    if (batch_dims == nullptr) num_batches = 1;
    *supported_out = 0;
    *total_bytes_out = 0;
    Arena &arena = Arena::of(stream);
    PassState &state = pass_state(arena);
    arena.pass_pending = false;
    arena.pending.valid = false;             // (the levels' bitmaps lie where a count's result does)
    int inverses = 0, tables = 0;
    for (int i = 0; i < num_maps; ++i) {
      const mnt_pass_map &m = maps[i];
      MNT_CHECK(m.source_level >= 0 && m.source_level <= num_levels && m.target_level >= 0 &&
                    m.target_level <= num_levels && m.offsets_host != nullptr,
                "map %d of the pass names levels that do not exist", i);
      MNT_CHECK(!(m.want & MNT_PASS_GROUPS) || (m.group_offsets_host != nullptr && m.num_offsets == 27),
                "map %d of the pass has no offset groups", i);
      if (m.num_offsets < 1 || m.num_offsets > 343) return;
      inverses += (m.want & MNT_PASS_INVERSE) ? 1 : 0;
      tables += (m.want & MNT_PASS_TABLES) ? 1 : 0;
    }
    // fills and jobs of one launch
    if (num_levels > kPassLevels || inverses + tables + kPassParents > kPassFills || inverses > kPassMaps ||
        tables > kPassMaps) {
      return;
    }
    for (int l = 0; l < num_levels; ++l) {
      for (int k = 0; k < ndim; ++k) MNT_CHECK(levels[l].stride[k] > 0, "level stride must be positive");
    }
    long long bounds[16];
    profile_mark("enter:pass", stream);
    if (bounds_host != nullptr) {
      for (int i = 0; i < 8; ++i) bounds[i] = bounds_host[i];
    } else {
      Scope scope(stream);
      read_bounds(coords, n, nullptr, 0, ndim, coord_dtype, bounds, scope, stream);
    }
    if (bounds_host_out != nullptr) {
      for (int i = 0; i < 8; ++i) bounds_host_out[i] = bounds[i];
    }
    state.coords = coords;
    state.levels = levels;
    state.maps = maps;
    state.n = n;
    state.ndim = ndim;
    state.coord_dtype = coord_dtype;
    state.index_dtype = index_dtype;
    state.num_batches = num_batches;
    state.num_levels = num_levels;
    state.num_maps = num_maps;
    if (!levels_supported(coords, batch_dims, bounds, levels, maps, state, total_bytes_out, stream)) return;
    profile_mark("pass_marks+sync", stream);
    arena.pass_pending = true;
    *supported_out = 1;
  });
}

extern "C" int mnt_pass_build(const void *coords, const void *batch_dims, mnt_pass_level *levels, mnt_pass_map *maps,
                              void *base, void *stream_) {
  return guarded([&] {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    Arena &arena = Arena::of(stream);
    MNT_CHECK(arena.pass_pending, "mnt_pass_build called without a preceding mnt_pass_levels");
    PassState &state = pass_state(arena);
    // (two threads that take turns on one stream: the first to come back finds the other's state)
    MNT_CHECK(state.coords == coords && state.levels == levels && state.maps == maps,
              "mnt_pass_build called for another cloud or other lists than the mnt_pass_levels before it on this stream");
    arena.pass_pending = false;
    MNT_CHECK(coords != nullptr && base != nullptr && reinterpret_cast<uintptr_t>(base) % 256 == 0,
              "the block of a pass must be 256-byte aligned");
    for (int i = 0; i < state.num_maps; ++i) {
      MNT_CHECK(!(maps[i].want & MNT_PASS_TABLES) || (maps[i].sizes_host != nullptr && maps[i].order_host != nullptr),
                "map %d of the pass has nowhere to put its sizes", i);
    }
    build_pass(coords, batch_dims, levels, maps, static_cast<char *>(base), state, stream);
  });
}
