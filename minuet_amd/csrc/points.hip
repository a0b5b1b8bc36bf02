// What stands before the first layer and after the last one: points to voxels,
// the feature rows of a collated batch, and the global pools.  Each took five
// to eight tensor expressions with a read-back among them; here each is one
// library call (minuet/nn/functional/voxelize.py:11-35, pooling.py).  Measured:
// 100 000 points to voxels 148 -> 56 us; mean pools of 8 clouds of 3 000 voxels
// 91 us of kernels and a read-back -> 8 us.
#include <algorithm>
#include <limits>

#include "conv_device.h"
#include "device_utils.h"
#include "sort.h"
#include "target_keys.h"

namespace mnt {

// ------------------------------------------------------------------ voxels ----

struct VoxelSizes {
  double v[MNT_MAX_NDIM];
};

// floor(p / size) in the points' own precision, as the tensor expression has it.
template <typename FT, typename CT>
__global__ __launch_bounds__(256) void voxel_kernel(const FT *__restrict__ points, long long total, int ndim,
                                                    VoxelSizes sizes, CT *__restrict__ out) {
  const long long i = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= total) return;
  const int k = static_cast<int>(i % ndim);
  FT size = static_cast<FT>(sizes.v[0]);
#pragma unroll
  for (int d = 1; d < MNT_MAX_NDIM; ++d) size = k == d ? static_cast<FT>(sizes.v[d]) : size;
  const FT q = points[i] / size;
  out[i] = static_cast<CT>(sizeof(FT) == 4 ? floorf(static_cast<float>(q)) : floor(static_cast<double>(q)));
}

// The same for clouds that the bucket sort takes: the launch that has the rows in
// registers leaves their extremes too, one part a workgroup, and clears the
// sort's counters.  Bound by latency: 4.5 us at 100 003 points, where the two
// launches are 3.2 and 4.6 and the gap between them; the whole call is 55.8
// against 59.7 (5 000: 49 against 53; a million, where 128 workgroups are few
// for the points: 163 both ways).  The chain of sorting launches that waits for
// the host only once is 49 at 100 003 points, but clouds of walls, which crowd
// more than 4 096 rows into one of its buckets from 65 000 points on, pay for
// it and then for this sort: 75 against 55.
constexpr int kVoxelRows = 4;
template <typename FT, typename CT>
__global__ __launch_bounds__(256) void voxel_bounds_kernel(const FT *__restrict__ points, long long n, int ndim,
                                                           VoxelSizes sizes, CT *__restrict__ out,
                                                           long long *__restrict__ partial,
                                                           unsigned *__restrict__ zero, int zero_count) {
  __shared__ CT s_extreme[256 / kWave][2 * MNT_MAX_NDIM];
  const int tid = threadIdx.x;
  for (int i = blockIdx.x * 256 + tid; i < zero_count; i += gridDim.x * 256) zero[i] = 0u;
  FT size[MNT_MAX_NDIM];
#pragma unroll
  for (int k = 0; k < MNT_MAX_NDIM; ++k) size[k] = static_cast<FT>(sizes.v[k < ndim ? k : 0]);
  CT extreme[2 * MNT_MAX_NDIM];                  // ~v turns the order round
#pragma unroll
  for (int k = 0; k < 2 * MNT_MAX_NDIM; ++k) extreme[k] = std::numeric_limits<CT>::max();
  const long long stride = static_cast<long long>(gridDim.x) * 256;
  for (long long i0 = static_cast<long long>(blockIdx.x) * 256 + tid; i0 < n; i0 += kVoxelRows * stride) {
    FT p[kVoxelRows][MNT_MAX_NDIM];
#pragma unroll
    for (int r = 0; r < kVoxelRows; ++r) {
      const long long i = i0 + r * stride;
#pragma unroll
      for (int k = 0; k < MNT_MAX_NDIM; ++k) p[r][k] = points[(i < n ? i : n - 1) * ndim + (k < ndim ? k : 0)];
    }
#pragma unroll
    for (int r = 0; r < kVoxelRows; ++r) {
      const long long i = i0 + r * stride;
#pragma unroll
      for (int k = 0; k < MNT_MAX_NDIM; ++k) {
        const FT q = p[r][k] / size[k];
        const CT v = static_cast<CT>(sizeof(FT) == 4 ? floorf(static_cast<float>(q)) : floor(static_cast<double>(q)));
        if (i < n && k < ndim) out[i * ndim + k] = v;
        extreme[k] = v < extreme[k] ? v : extreme[k];
        const CT turned = static_cast<CT>(~v);
        extreme[MNT_MAX_NDIM + k] = turned < extreme[MNT_MAX_NDIM + k] ? turned : extreme[MNT_MAX_NDIM + k];
      }
    }
  }
  const CT folded = fold_extremes<CT>(extreme);
  if (lane_id() < 2 * MNT_MAX_NDIM) s_extreme[tid / kWave][lane_id()] = folded;
  __syncthreads();
  if (tid < 2 * MNT_MAX_NDIM) {
    CT v = s_extreme[0][tid];
#pragma unroll
    for (int w = 1; w < 256 / kWave; ++w) v = s_extreme[w][tid] < v ? s_extreme[w][tid] : v;
    partial[static_cast<long long>(blockIdx.x) * 8 + tid] = static_cast<long long>(tid < MNT_MAX_NDIM ? v : static_cast<CT>(~v));
  }
}

// Distinct rows of sorted rows.  Each tile counts the rows that start a run; the
// counts before a tile give every run its place; a run's first row is written
// there and every row's place goes to reverse[order[i]].  What bounds these
// passes is latency, so a tile is 512 rows (two per thread: 100 000 points fill
// the chip) and up to kRunSelfTiles tiles the emitting workgroups add up the
// counts before their own instead of waiting for a launch that scans them;
// beyond that reading all counts in every workgroup would cost more than it.
constexpr int kRunItems = 2;
constexpr int kRunTile = kScanBlock * kRunItems;
constexpr int kRunSelfTiles = 2048;

template <typename CT>
__device__ __forceinline__ bool starts_run(const CT *__restrict__ rows, long long i, int ndim) {
  if (i == 0) return true;
  bool same = true;
#pragma unroll
  for (int k = 0; k < MNT_MAX_NDIM; ++k) {
    const int at = k < ndim ? k : 0;
    same = same && rows[i * ndim + at] == rows[(i - 1) * ndim + at];
  }
  return !same;
}

template <typename CT>
__global__ __launch_bounds__(kScanBlock) void run_sums_kernel(const CT *__restrict__ rows, long long n, int ndim,
                                                              unsigned *__restrict__ tile_sums) {
  __shared__ unsigned s_part[kScanBlock / kWave];
  const long long base = static_cast<long long>(blockIdx.x) * kRunTile;
  unsigned count = 0;
#pragma unroll
  for (int r = 0; r < kRunItems; ++r) {
    const long long i = base + r * kScanBlock + threadIdx.x;
    count += __popcll(__ballot(i < n && starts_run<CT>(rows, i, ndim)));
  }
  if (lane_id() == 0) s_part[threadIdx.x / kWave] = count;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned sum = 0;
#pragma unroll
    for (int w = 0; w < kScanBlock / kWave; ++w) sum += s_part[w];
    tile_sums[blockIdx.x] = sum;
  }
}

// Where the host finds the number of runs.
struct RunTell {
  unsigned *count;
  unsigned long long *flag;
  unsigned long long sequence;
  __device__ __forceinline__ void tell(unsigned total) const {
    *count = total;
    __threadfence_system();
    __hip_atomic_store(flag, sequence, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
};

__global__ __launch_bounds__(1024) void run_scan_kernel(unsigned *__restrict__ tile_sums, int tiles, RunTell host) {
  const unsigned total = scan_in_place(tile_sums, tiles);
  if (threadIdx.x == 1023) host.tell(total);
}

template <typename CT>
__global__ __launch_bounds__(kScanBlock) void run_emit_kernel(const CT *__restrict__ rows, long long n, int ndim,
                                                              const unsigned *__restrict__ tile_sums, bool scanned,
                                                              RunTell host, const int *__restrict__ order,
                                                              CT *__restrict__ out, long long *__restrict__ reverse) {
  constexpr int kWaves = kScanBlock / kWave;
  __shared__ unsigned s_count[kRunItems][kWaves], s_before[kWaves];
  const long long base = static_cast<long long>(blockIdx.x) * kRunTile;
  const int wave = threadIdx.x / kWave;
  bool first[kRunItems];
  unsigned long long votes[kRunItems];
  int to[kRunItems];
#pragma unroll
  for (int r = 0; r < kRunItems; ++r) {
    const long long i = base + r * kScanBlock + threadIdx.x;
    first[r] = i < n && starts_run<CT>(rows, i, ndim);
    to[r] = i < n ? order[i] : 0;
    votes[r] = __ballot(first[r]);
    if (lane_id() == 0) s_count[r][wave] = __popcll(votes[r]);
  }
  unsigned earlier = 0;
  if (!scanned) {
    for (unsigned t = threadIdx.x; t < blockIdx.x; t += kScanBlock) earlier += tile_sums[t];
    for (int d = 32; d >= 1; d >>= 1) earlier += __shfl_xor(earlier, d);
    if (lane_id() == 0) s_before[wave] = earlier;
  }
  __syncthreads();
  unsigned run = 0;
  if (scanned) {
    run = tile_sums[blockIdx.x];
  } else {
#pragma unroll
    for (int w = 0; w < kWaves; ++w) run += s_before[w];
  }
#pragma unroll
  for (int r = 0; r < kRunItems; ++r) {
    unsigned before = run, all = run;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      before += w < wave ? s_count[r][w] : 0u;
      all += s_count[r][w];
    }
    run = all;
    const long long i = base + r * kScanBlock + threadIdx.x;
    if (i >= n) continue;
    // rows up to and including this one that start a run, less one: the row of its run
    const unsigned at = before + __popcll(votes[r] & (lanes_below() | (1ull << lane_id()))) - 1u;
    if (first[r]) {
      for (int k = 0; k < ndim; ++k) out[static_cast<long long>(at) * ndim + k] = rows[i * ndim + k];
    }
    if (reverse != nullptr) reverse[to[r]] = static_cast<long long>(at);
  }
  if (!scanned && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) host.tell(run);
}

template <typename FT, typename CT>
static void voxelize_typed(const FT *points, int64_t n, int ndim, const VoxelSizes &sizes, CT *voxels_out,
                           long long *reverse_out, int64_t *count_out, hipStream_t stream) {
  Scope scope(stream);
  Arena &arena = scope.arena();
  CT *voxels = scope.alloc<CT>(static_cast<size_t>(n) * ndim);
  CT *sorted = scope.alloc<CT>(static_cast<size_t>(n) * ndim);
  int *order = scope.alloc<int>(n);
  const int tiles = static_cast<int>(div_ceil(n, kRunTile));
  unsigned *tile_sums = scope.alloc<unsigned>(static_cast<size_t>(tiles) + 1);
  const SortStart start = sort_start(n, scope);
  if (start.parts > 0) {
    voxel_bounds_kernel<FT, CT><<<start.parts, 256, 0, stream>>>(points, n, ndim, sizes, voxels, start.partial,
                                                                 start.clear, start.clear_words);
    check_launch("voxel_bounds_kernel");
  } else {
    voxel_kernel<FT, CT><<<static_cast<unsigned>(div_ceil(n * ndim, 256)), 256, 0, stream>>>(points, n * ndim, ndim,
                                                                                            sizes, voxels);
    check_launch("voxel_kernel");
  }
  sort_started_rows(voxels, n, ndim, sizeof(CT) == 4 ? MNT_INT32 : MNT_INT64, order, sorted, start, stream);
  volatile unsigned *h = reinterpret_cast<volatile unsigned *>(static_cast<char *>(arena.pinned()) + 256);
  unsigned *d = reinterpret_cast<unsigned *>(static_cast<char *>(arena.pinned_device()) + 256);
  const unsigned long long sequence = arena.next_sequence();
  run_sums_kernel<CT><<<tiles, kScanBlock, 0, stream>>>(sorted, n, ndim, tile_sums);
  check_launch("run_sums_kernel");
  const bool scanned = tiles > kRunSelfTiles;
  const RunTell host{d, arena.flag_device(2), sequence};
  if (scanned) {
    run_scan_kernel<<<1, 1024, 0, stream>>>(tile_sums, tiles, host);
    check_launch("run_scan_kernel");
  }
  run_emit_kernel<CT><<<tiles, kScanBlock, 0, stream>>>(sorted, n, ndim, tile_sums, scanned, host, order, voxels_out,
                                                        reverse_out);
  check_launch("run_emit_kernel");
  arena.wait_flag(2, sequence);
  *count_out = static_cast<int64_t>(*h);
}

// ------------------------------------------------------------------- rows ----

// Rows of several tensors, numbered one after the other, in a given order:
// what concatenating them and indexing the result does, without the copy in
// between.
constexpr int kGatherSources = 64;
struct GatherSources {
  const unsigned char *data[kGatherSources];
  int first[kGatherSources + 1];
  int count;
};

template <int VB, typename IT>
__global__ __launch_bounds__(256) void gather_rows_kernel(GatherSources src, const IT *__restrict__ order, long long n,
                                                          int lanes_per_row, unsigned char *__restrict__ out) {
  typedef typename VecOf<VB>::type V;
  const long long i = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  const long long row = i / lanes_per_row;
  if (row >= n) return;
  const int piece = static_cast<int>(i - row * lanes_per_row);
  const int from = static_cast<int>(order[row]);
  int g = 0;
  while (g + 1 < src.count && src.first[g + 1] <= from) ++g;
  const long long at = static_cast<long long>(from - src.first[g]) * lanes_per_row + piece;
  reinterpret_cast<V *>(out)[i] = reinterpret_cast<const V *>(src.data[g])[at];
}

// The coordinate rows of several clouds one after the other and the clouds'
// boundaries, and for their sort what voxel_bounds_kernel leaves it (partial
// null: nothing).  As launches of their own, a concatenation, the boundaries'
// upload and the bounds are 4.4, 1.5 and 4.9 us and the gaps between them (eight
// clouds of 3 000 voxels), in front of a sort that waits for them.  Bound by
// latency, so it has the workgroups and rows per thread of voxel_bounds_kernel.
// With the sort and the feature rows behind it in one call a classifier's pass over
// those clouds takes 349 us, by calls of their own 376.
template <typename CT>
__global__ __launch_bounds__(256) void collate_rows_kernel(GatherSources src, int ndim, CT *__restrict__ out,
                                                           CT *__restrict__ batch_dims,
                                                           long long *__restrict__ partial,
                                                           unsigned *__restrict__ zero, int zero_count) {
  __shared__ CT s_extreme[256 / kWave][2 * MNT_MAX_NDIM];
  const int tid = threadIdx.x;
  const long long n = src.first[src.count];
  for (int i = blockIdx.x * 256 + tid; i < zero_count; i += gridDim.x * 256) zero[i] = 0u;
  if (blockIdx.x == 0) {
    for (int g = tid; g <= src.count; g += 256) batch_dims[g] = static_cast<CT>(src.first[g]);
  }
  CT extreme[2 * MNT_MAX_NDIM];                  // ~v turns the order round
#pragma unroll
  for (int k = 0; k < 2 * MNT_MAX_NDIM; ++k) extreme[k] = std::numeric_limits<CT>::max();
  const long long stride = static_cast<long long>(gridDim.x) * 256;
  for (long long i0 = static_cast<long long>(blockIdx.x) * 256 + tid; i0 < n; i0 += kVoxelRows * stride) {
    CT p[kVoxelRows][MNT_MAX_NDIM];
#pragma unroll
    for (int r = 0; r < kVoxelRows; ++r) {
      const int from = static_cast<int>(min(i0 + r * stride, n - 1));
      int g = 0;
      while (src.first[g + 1] <= from) ++g;      // (from < first[count])
      const CT *row = reinterpret_cast<const CT *>(src.data[g]) + static_cast<long long>(from - src.first[g]) * ndim;
#pragma unroll
      for (int k = 0; k < MNT_MAX_NDIM; ++k) p[r][k] = row[k < ndim ? k : 0];
    }
#pragma unroll
    for (int r = 0; r < kVoxelRows; ++r) {
      const long long i = i0 + r * stride;
#pragma unroll
      for (int k = 0; k < MNT_MAX_NDIM; ++k) {
        const CT v = p[r][k];
        if (i < n && k < ndim) out[i * ndim + k] = v;
        extreme[k] = v < extreme[k] ? v : extreme[k];
        const CT turned = static_cast<CT>(~v);
        extreme[MNT_MAX_NDIM + k] = turned < extreme[MNT_MAX_NDIM + k] ? turned : extreme[MNT_MAX_NDIM + k];
      }
    }
  }
  if (partial == nullptr) return;
  const CT folded = fold_extremes<CT>(extreme);
  if (lane_id() < 2 * MNT_MAX_NDIM) s_extreme[tid / kWave][lane_id()] = folded;
  __syncthreads();
  if (tid < 2 * MNT_MAX_NDIM) {
    CT v = s_extreme[0][tid];
#pragma unroll
    for (int w = 1; w < 256 / kWave; ++w) v = s_extreme[w][tid] < v ? s_extreme[w][tid] : v;
    partial[static_cast<long long>(blockIdx.x) * 8 + tid] = static_cast<long long>(tid < MNT_MAX_NDIM ? v : static_cast<CT>(~v));
  }
}

// The tensors' addresses and the numbers of their first rows; rows: how many there are.
static GatherSources gather_sources(const void *const *sources, const int64_t *source_rows, int num_sources,
                                    int64_t &rows, uintptr_t &align) {
  MNT_CHECK(num_sources >= 1 && num_sources <= kGatherSources, "between 1 and %d tensors but found %d",
            kGatherSources, num_sources);
  MNT_CHECK(sources != nullptr && source_rows != nullptr, "bad argument");
  GatherSources src;
  memset(&src, 0, sizeof(src));
  src.count = num_sources;
  rows = 0;
  for (int g = 0; g < num_sources; ++g) {
    src.data[g] = static_cast<const unsigned char *>(sources[g]);
    src.first[g] = static_cast<int>(rows);
    MNT_CHECK(source_rows[g] >= 0, "bad argument");
    rows += source_rows[g];
    align |= reinterpret_cast<uintptr_t>(sources[g]);
    MNT_CHECK(rows <= INT32_MAX, "too many rows");
  }
  src.first[num_sources] = static_cast<int>(rows);
  return src;
}

static void gather_rows(const GatherSources &src, uintptr_t align, int64_t row_bytes, const void *order,
                        int index_dtype, int64_t n, void *out, hipStream_t stream) {
  align |= reinterpret_cast<uintptr_t>(out) | static_cast<uintptr_t>(row_bytes);
  MNT_CHECK(align % 2 == 0, "rows are not aligned to two bytes");
  const int vb = align % 16 == 0 ? 16 : align % 8 == 0 ? 8 : align % 4 == 0 ? 4 : 2;
  const int lanes = static_cast<int>(row_bytes / vb);
  const unsigned blocks = static_cast<unsigned>(div_ceil(n * lanes, 256));
  unsigned char *to = static_cast<unsigned char *>(out);
#define MNT_GATHER(VB)                                                                                             \
  if (index_dtype == MNT_INT32) {                                                                                  \
    gather_rows_kernel<VB, int32_t><<<blocks, 256, 0, stream>>>(src, static_cast<const int32_t *>(order), n, lanes, to); \
  } else {                                                                                                         \
    gather_rows_kernel<VB, int64_t><<<blocks, 256, 0, stream>>>(src, static_cast<const int64_t *>(order), n, lanes, to); \
  }
  switch (vb) {
    case 16: MNT_GATHER(16) break;
    case 8: MNT_GATHER(8) break;
    case 4: MNT_GATHER(4) break;
    default: MNT_GATHER(2) break;
  }
#undef MNT_GATHER
  check_launch("gather_rows_kernel");
}

// ------------------------------------------------------------------- pools ----

// Sum or mean of the rows of every cloud.  blockIdx.y is the cloud, blockIdx.x
// one of `parts` runs of its rows, blockIdx.z a block of up to 256 lanes of a
// row.  A workgroup takes 256 / lanes rows at a time, eight of them in flight
// per lane, adds in fp32 and folds its lane groups in LDS.  One part: the
// result itself; more: partial sums for pool_fold_kernel.
constexpr int kPoolBlock = 256;
constexpr int kPoolInFlight = 8;

// The rows of a cloud, kept inside the features as a slice of them would be:
// boundaries come from the caller and are not checked on the host.
struct CloudRows {
  long long lo, hi;
};
template <typename IT>
__device__ __forceinline__ CloudRows cloud_rows(const IT *__restrict__ batch_dims, long long cloud, long long n) {
  if (batch_dims == nullptr) return {0, n};
  const long long lo = min(max(static_cast<long long>(batch_dims[cloud]), 0ll), n);
  return {lo, min(max(static_cast<long long>(batch_dims[cloud + 1]), lo), n)};
}

template <typename T, int VB, typename IT>
__global__ __launch_bounds__(kPoolBlock) void pool_kernel(const unsigned char *__restrict__ features,
                                                          const IT *__restrict__ batch_dims, long long n, int channels,
                                                          int lanes, int lanes_per_row, int mean,
                                                          float *__restrict__ partial, T *__restrict__ out) {
  typedef typename VecOf<VB>::type V;
  constexpr int E = VB / static_cast<int>(sizeof(T));
  __shared__ float s_sum[kPoolBlock * E];
  const int groups = kPoolBlock / lanes;
  const int group = threadIdx.x / lanes, lane = threadIdx.x - group * lanes;
  const int piece = blockIdx.z * lanes + lane;
  const CloudRows cloud = cloud_rows<IT>(batch_dims, blockIdx.y, n);
  const long long lo = cloud.lo, hi = cloud.hi;
  const long long share = (hi - lo + gridDim.x - 1) / gridDim.x;
  const long long from = lo + blockIdx.x * share;
  const long long to = from + share < hi ? from + share : hi;
  float sum[E];
#pragma unroll
  for (int e = 0; e < E; ++e) sum[e] = 0.0f;
  if (group < groups && piece < lanes_per_row) {
    for (long long r = from + group; r < to; r += static_cast<long long>(groups) * kPoolInFlight) {
      V v[kPoolInFlight];
#pragma unroll
      for (int u = 0; u < kPoolInFlight; ++u) {
        const long long row = r + static_cast<long long>(u) * groups;
        v[u] = reinterpret_cast<const V *>(features)[(row < to ? row : r) * lanes_per_row + piece];
      }
#pragma unroll
      for (int u = 0; u < kPoolInFlight; ++u) {
        if (r + static_cast<long long>(u) * groups < to) {
          const T *e = reinterpret_cast<const T *>(&v[u]);
#pragma unroll
          for (int x = 0; x < E; ++x) sum[x] += to_float(e[x]);
        }
      }
    }
  }
#pragma unroll
  for (int e = 0; e < E; ++e) s_sum[e * kPoolBlock + threadIdx.x] = sum[e];
  __syncthreads();
  for (int i = threadIdx.x; i < lanes * E; i += kPoolBlock) {
    const int l = i / E, e = i % E;
    if (blockIdx.z * lanes + l >= lanes_per_row) continue;
    float total = 0.0f;
    for (int g = 0; g < groups; ++g) total += s_sum[e * kPoolBlock + g * lanes + l];
    const int channel = (blockIdx.z * lanes + l) * E + e;
    if (partial != nullptr) {
      partial[(static_cast<long long>(blockIdx.y) * gridDim.x + blockIdx.x) * channels + channel] = total;
    } else {
      out[static_cast<long long>(blockIdx.y) * channels + channel] =
          static_cast<T>(mean ? total / static_cast<float>(hi - lo) : total);
    }
  }
}

template <typename T, typename IT>
__global__ __launch_bounds__(256) void pool_fold_kernel(const float *__restrict__ partial,
                                                        const IT *__restrict__ batch_dims, long long n, int parts,
                                                        int channels, long long total, int mean, T *__restrict__ out) {
  const long long i = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= total) return;
  const long long cloud = i / channels;
  const float *at = partial + cloud * parts * channels + (i - cloud * channels);
  float sum = 0.0f;
  for (int p = 0; p < parts; ++p) sum += at[static_cast<long long>(p) * channels];
  const CloudRows of = cloud_rows<IT>(batch_dims, cloud, n);
  const long long rows = of.hi - of.lo;
  out[i] = static_cast<T>(mean ? sum / static_cast<float>(rows) : sum);
}

// out[b][c] = rows[b] . weights[c] + bias[c], a classifier's head: a wavefront per
// output, pieces of VB bytes per lane, sums in fp32.  Bound by its launch alone:
// 8 clouds of 256 fp16 channels to 10 classes take 2.3 us of the device and 7 of
// the host, torch's linear 3.1 and 18.
template <typename T, int VB>
__global__ __launch_bounds__(256) void linear_kernel(const T *__restrict__ rows, const T *__restrict__ weights,
                                                     const T *__restrict__ bias, int channels, int classes,
                                                     int outputs, T *__restrict__ out) {
  typedef typename VecOf<VB>::type V;
  constexpr int E = VB / static_cast<int>(sizeof(T));
  const int at = static_cast<int>(blockIdx.x) * 4 + static_cast<int>(threadIdx.x / kWave);
  if (at >= outputs) return;
  const int b = at / classes, c = at - b * classes;
  const V *x = reinterpret_cast<const V *>(rows + static_cast<long long>(b) * channels);
  const V *w = reinterpret_cast<const V *>(weights + static_cast<long long>(c) * channels);
  float sum = 0.0f;
  for (int p = lane_id(); p < channels / E; p += kWave) {
    const V vx = x[p], vw = w[p];
    const T *ex = reinterpret_cast<const T *>(&vx), *ew = reinterpret_cast<const T *>(&vw);
#pragma unroll
    for (int e = 0; e < E; ++e) sum = fmaf(to_float(ex[e]), to_float(ew[e]), sum);
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) sum += __shfl_xor(sum, d);
  if (lane_id() == 0) out[at] = static_cast<T>(sum + (bias != nullptr ? to_float(bias[c]) : 0.0f));
}

template <typename T>
static void linear_typed(const T *rows, const T *weights, const T *bias, int64_t batches, int64_t channels,
                         int64_t classes, T *out, hipStream_t stream) {
  int vb = 16;
  while (vb > static_cast<int>(sizeof(T)) &&
         (channels * sizeof(T) % vb != 0 || (reinterpret_cast<uintptr_t>(rows) | reinterpret_cast<uintptr_t>(weights)) % vb != 0)) {
    vb /= 2;
  }
  const int outputs = static_cast<int>(batches * classes);
  const unsigned blocks = static_cast<unsigned>(div_ceil(outputs, 4));
#define MNT_LINEAR(VB)                                                                                  \
  linear_kernel<T, VB><<<blocks, 256, 0, stream>>>(rows, weights, bias, static_cast<int>(channels),     \
                                                   static_cast<int>(classes), outputs, out)
  if (vb == 16) MNT_LINEAR(16);
  else if (vb == 8) MNT_LINEAR(8);
  else if (vb == 4) MNT_LINEAR(4);
  else if constexpr (sizeof(T) == 2) MNT_LINEAR(2);
#undef MNT_LINEAR
  check_launch("linear_kernel");
}

template <typename T, typename IT>
static void pool_typed(const void *features, const IT *batch_dims, int64_t n, int64_t batches, int64_t channels,
                       int mean, T *out, hipStream_t stream) {
  Scope scope(stream);
  const int64_t row_bytes = channels * sizeof(T);
  int vb = 16;
  while (vb > static_cast<int>(sizeof(T)) && (row_bytes % vb != 0 || reinterpret_cast<uintptr_t>(features) % vb != 0)) vb /= 2;
  const int lanes_per_row = static_cast<int>(row_bytes / vb);
  const int lanes = std::min(lanes_per_row, kPoolBlock);
  const int groups = kPoolBlock / lanes;
  // as many parts as leave every workgroup about four rounds of loads, and never more than fill the chip
  const int64_t rows = div_ceil(std::max<int64_t>(n, 1), batches);
  const int64_t most = std::max<int64_t>(1, 4 * compute_units() / batches);
  const int parts = static_cast<int>(std::max<int64_t>(
      1, std::min<int64_t>(std::min<int64_t>(most, 256), rows / (static_cast<int64_t>(groups) * kPoolInFlight * 4))));
  float *partial = parts > 1 ? scope.alloc<float>(static_cast<size_t>(batches) * parts * channels) : nullptr;
  const dim3 grid(static_cast<unsigned>(parts), static_cast<unsigned>(batches),
                  static_cast<unsigned>(div_ceil(lanes_per_row, lanes)));
#define MNT_POOL(VB)                                                                                              \
  pool_kernel<T, VB, IT><<<grid, kPoolBlock, 0, stream>>>(static_cast<const unsigned char *>(features), batch_dims, \
                                                          n, static_cast<int>(channels), lanes, lanes_per_row,     \
                                                          mean, partial, out)
  if (vb == 16) MNT_POOL(16);
  else if (vb == 8) MNT_POOL(8);
  else if (vb == 4) MNT_POOL(4);
  else if constexpr (sizeof(T) == 2) MNT_POOL(2);
#undef MNT_POOL
  check_launch("pool_kernel");
  if (parts > 1) {
    const int64_t total = batches * channels;
    pool_fold_kernel<T, IT><<<static_cast<unsigned>(div_ceil(total, 256)), 256, 0, stream>>>(
        partial, batch_dims, n, parts, static_cast<int>(channels), total, mean, out);
    check_launch("pool_fold_kernel");
  }
}

}  // namespace mnt

using namespace mnt;

extern "C" int mnt_voxelize(const void *points, int64_t n, int ndim, int wide_points, const double *voxel_size,
                            int coord_dtype, void *voxels_out, int64_t *reverse_out, int64_t *count_out,
                            void *stream_) {
  return guarded([&] {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MNT_CHECK(ndim >= 1 && ndim <= MNT_MAX_NDIM, "ndim must be in [1, %d] but found %d", MNT_MAX_NDIM, ndim);
    MNT_CHECK(n > 0 && n <= INT32_MAX, "number of points %lld out of range", static_cast<long long>(n));
    MNT_CHECK(points != nullptr && voxel_size != nullptr && voxels_out != nullptr && count_out != nullptr, "null argument");
    int_size(coord_dtype);
    VoxelSizes sizes;
    for (int k = 0; k < MNT_MAX_NDIM; ++k) sizes.v[k] = voxel_size[k < ndim ? k : 0];
    long long *reverse = reinterpret_cast<long long *>(reverse_out);
#define MNT_CALL(FT, CT)                                                                                    \
  voxelize_typed<FT, CT>(static_cast<const FT *>(points), n, ndim, sizes, static_cast<CT *>(voxels_out), reverse, \
                         count_out, stream)
    if (coord_dtype == MNT_INT32) {
      if (wide_points != 0) MNT_CALL(double, int32_t);
      else MNT_CALL(float, int32_t);
    } else {
      if (wide_points != 0) MNT_CALL(double, int64_t);
      else MNT_CALL(float, int64_t);
    }
#undef MNT_CALL
  });
}

extern "C" int mnt_gather_rows(const void *const *sources, const int64_t *source_rows, int num_sources,
                               int64_t row_bytes, const void *order, int index_dtype, int64_t n, void *out,
                               void *stream_) {
  return guarded([&] {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MNT_CHECK(sources != nullptr && source_rows != nullptr && row_bytes >= 1, "bad argument");
    MNT_CHECK(num_sources >= 1 && num_sources <= kGatherSources, "between 1 and %d tensors but found %d",
              kGatherSources, num_sources);
    int_size(index_dtype);
    if (n == 0) return;                            // (of however many rows)
    int64_t rows = 0;
    uintptr_t align = 0;
    const GatherSources src = gather_sources(sources, source_rows, num_sources, rows, align);
    MNT_CHECK(n <= rows, "more rows asked for than there are");
    gather_rows(src, align, row_bytes, order, index_dtype, n, out, stream);
  });
}

extern "C" int mnt_collate(const void *const *clouds, const void *const *features, const int64_t *cloud_rows,
                           int num_clouds, int ndim, int coord_dtype, int64_t row_bytes, void *sorted_out,
                           void *batch_dims_out, void *features_out, int64_t *bounds_host_out, void *stream_) {
  return guarded([&] {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MNT_CHECK(ndim >= 1 && ndim <= MNT_MAX_NDIM, "ndim must be in [1, %d] but found %d", MNT_MAX_NDIM, ndim);
    const int csz = int_size(coord_dtype);
    int64_t n = 0, feature_rows = 0;
    uintptr_t align = 0, feature_align = 0;
    const GatherSources src = gather_sources(clouds, cloud_rows, num_clouds, n, align);
    MNT_CHECK(n >= 1 && align % csz == 0, "clouds without a row, or not aligned to their type");
    MNT_CHECK(sorted_out != nullptr && batch_dims_out != nullptr, "null argument");
    GatherSources rows;
    if (features_out != nullptr) {
      MNT_CHECK(row_bytes >= 1, "bad argument");
      rows = gather_sources(features, cloud_rows, num_clouds, feature_rows, feature_align);
    }
    Scope scope(stream);
    void *stacked = scope.alloc<unsigned char>(static_cast<size_t>(n) * ndim * csz);
    void *order = scope.alloc<unsigned char>(static_cast<size_t>(n) * csz);
    const SortStart start = sort_start(n, scope);
    const unsigned blocks = start.parts > 0 ? start.parts : grid_for(div_ceil(n, int64_t{kVoxelRows}), 256, 4096);
    if (coord_dtype == MNT_INT32) {
      collate_rows_kernel<int32_t><<<blocks, 256, 0, stream>>>(src, ndim, static_cast<int32_t *>(stacked),
                                                               static_cast<int32_t *>(batch_dims_out), start.partial,
                                                               start.clear, start.clear_words);
    } else {
      collate_rows_kernel<int64_t><<<blocks, 256, 0, stream>>>(src, ndim, static_cast<int64_t *>(stacked),
                                                               static_cast<int64_t *>(batch_dims_out), start.partial,
                                                               start.clear, start.clear_words);
    }
    check_launch("collate_rows_kernel");
    sort_started_batches(stacked, n, ndim, coord_dtype, batch_dims_out, num_clouds, order, sorted_out,
                         bounds_host_out, start, stream);
    if (features_out != nullptr) {
      gather_rows(rows, feature_align, row_bytes, order, coord_dtype, n, features_out, stream);
    }
  });
}

extern "C" int mnt_upload_ints(const int64_t *values, int64_t count, int index_dtype, void *out, void *stream_) {
  return guarded([&] {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MNT_CHECK(count >= 0 && (count == 0 || (values != nullptr && out != nullptr)), "bad argument");
    const int words = int_size(index_dtype) / 4;
    std::vector<int> ints(static_cast<size_t>(count) * words);
    if (words == 1) {
      for (int64_t i = 0; i < count; ++i) ints[i] = static_cast<int>(values[i]);
    } else if (count > 0) {
      memcpy(ints.data(), values, sizeof(int64_t) * count);
    }
    upload_ints(ints, static_cast<int *>(out), stream);
  });
}

extern "C" int mnt_global_pool(const void *features, const void *batch_dims, int64_t n, int64_t num_batches,
                               int64_t channels, int float_dtype, int index_dtype, int mean, void *out,
                               void *stream_) {
  return guarded([&] {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MNT_CHECK(n >= 0 && n <= INT32_MAX && num_batches >= 1 && num_batches <= 65535 && channels >= 1 && channels <= 65536,
              "bad shape N=%lld B=%lld C=%lld", (long long)n, (long long)num_batches, (long long)channels);
    MNT_CHECK(out != nullptr && (n == 0 || features != nullptr), "null argument");
    float_size(float_dtype);
    const bool narrow = batch_dims == nullptr || int_size(index_dtype) == 4;
    if (batch_dims == nullptr) num_batches = 1;
#define MNT_CALL(T)                                                                                                   \
  if (narrow) {                                                                                                       \
    pool_typed<T, int32_t>(features, static_cast<const int32_t *>(batch_dims), n, num_batches, channels, mean,         \
                           static_cast<T *>(out), stream);                                                            \
  } else {                                                                                                            \
    pool_typed<T, int64_t>(features, static_cast<const int64_t *>(batch_dims), n, num_batches, channels, mean,         \
                           static_cast<T *>(out), stream);                                                            \
  }
    if (float_dtype == MNT_FLOAT32) {
      MNT_CALL(float)
    } else if (float_dtype == MNT_FLOAT16) {
      MNT_CALL(half_t)
    } else {
      MNT_CALL(bf16_t)
    }
#undef MNT_CALL
  });
}

extern "C" int mnt_linear(const void *rows, const void *weights, const void *bias, int64_t num_rows, int64_t channels,
                          int64_t classes, int float_dtype, void *out, void *stream_) {
  return guarded([&] {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MNT_CHECK(num_rows >= 0 && classes >= 1 && channels >= 1 && channels <= INT32_MAX && num_rows <= INT32_MAX &&
                  classes <= INT32_MAX && num_rows * classes <= INT32_MAX - 4,
              "bad shape N=%lld Cin=%lld Cout=%lld", (long long)num_rows, (long long)channels, (long long)classes);
    if (num_rows == 0) return;
    MNT_CHECK(rows != nullptr && weights != nullptr && out != nullptr, "null argument");
    float_size(float_dtype);
#define MNT_CALL(T)                                                                                              \
  linear_typed<T>(static_cast<const T *>(rows), static_cast<const T *>(weights), static_cast<const T *>(bias), \
                  num_rows, channels, classes, static_cast<T *>(out), stream)
    if (float_dtype == MNT_FLOAT32) {
      MNT_CALL(float);
    } else if (float_dtype == MNT_FLOAT16) {
      MNT_CALL(half_t);
    } else {
      MNT_CALL(bf16_t);
    }
#undef MNT_CALL
  });
}
