// Keys of strided cells, and the bitmap that yields the distinct ones in sorted
// order: shared by the single-level build (unique.hip) and the pass builder
// (pass.hip).
#pragma once

#include <cstring>

#include "device_utils.h"

namespace mnt {

constexpr int kScanBlock = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanBlock * kScanItems;

// Exclusive scan of `flag` over the workgroup; returns this thread's exclusive
// prefix and the workgroup total through *total.
template <int BLOCK = kScanBlock>
__device__ __forceinline__ unsigned block_exclusive_scan(unsigned value, unsigned *total) {
  __shared__ unsigned wave_sums[BLOCK / kWave];
  unsigned inclusive = value;
  for (int off = 1; off < kWave; off <<= 1) {
    unsigned v = __shfl_up(inclusive, off);
    if (static_cast<int>(lane_id()) >= off) inclusive += v;
  }
  const int w = threadIdx.x >> 6;
  if (lane_id() == kWave - 1) wave_sums[w] = inclusive;
  __syncthreads();
  unsigned base = 0, sum = 0;
  for (int ww = 0; ww < BLOCK / kWave; ++ww) {
    if (ww < w) base += wave_sums[ww];
    sum += wave_sums[ww];
  }
  __syncthreads();
  *total = sum;
  return base + inclusive - value;
}

struct TargetSpec {
  long long base[MNT_MAX_NDIM];     // floor(min / stride) per dimension
  long long stride[MNT_MAX_NDIM];
  int log2_stride[MNT_MAX_NDIM];    // -1: the stride is no power of two
  int shift[MNT_MAX_NDIM];
  unsigned long long mask[MNT_MAX_NDIM];
  int batch_shift;
  int ndim;
  int num_batches;                  // 0 when there is no batch field
};

__device__ __forceinline__ long long floor_div(long long a, long long b) {
  long long q = a / b;
  return (a % b != 0 && ((a < 0) != (b < 0))) ? q - 1 : q;
}

// floor(c / stride) along dimension k (a 64-bit division is some 100
// instructions, a shift one; strides of networks are powers of two).
__device__ __forceinline__ long long cell_of(long long c, const TargetSpec &spec, int k) {
  return spec.log2_stride[k] >= 0 ? c >> spec.log2_stride[k] : floor_div(c, spec.stride[k]);
}

inline int bit_width64(unsigned long long range) {
  return range == 0 ? 0 : 64 - __builtin_clzll(range);
}

inline long long host_floor_div(long long a, long long b) {
  const long long q = a / b;
  return (a % b != 0 && ((a < 0) != (b < 0))) ? q - 1 : q;
}

// Key layout of the cells of a cloud with these bounds (minima [0..3], maxima
// [4..7]); num_batches = 0: no batch field.  Returns the key bits (more than 64:
// the spec is of no use).
inline int make_target_spec(const long long *bounds, const int64_t *stride, int ndim, int64_t num_batches,
                            TargetSpec &spec) {
  memset(&spec, 0, sizeof(spec));
  int bits = 0;
  spec.ndim = ndim;
  for (int k = ndim - 1; k >= 0; --k) {
    const long long lo = host_floor_div(bounds[k], stride[k]);
    const long long hi = host_floor_div(bounds[MNT_MAX_NDIM + k], stride[k]);
    const int width = bit_width64(static_cast<unsigned long long>(hi) - static_cast<unsigned long long>(lo));
    spec.base[k] = lo;
    spec.stride[k] = stride[k];
    spec.log2_stride[k] = (stride[k] & (stride[k] - 1)) == 0 ? __builtin_ctzll(stride[k]) : -1;
    spec.shift[k] = bits < 64 ? bits : 63;
    spec.mask[k] = width >= 64 ? ~0ull : ((1ull << width) - 1ull);
    bits += width;
  }
  spec.batch_shift = bits < 64 ? bits : 63;
  spec.num_batches = static_cast<int>(num_batches);
  return bits + (num_batches > 0 ? bit_width64(static_cast<unsigned long long>(num_batches - 1)) : 0);
}

// ---- bitmap form: when the packed keys span at most 2^28 values, the set of
// distinct keys is a bitmap.  Marking it and walking it in key order yields
// the sorted, duplicate-free targets without any sort.

constexpr int kBitmapMaxBits = 28;                   // 32 MiB of bits
constexpr int kBitmapWords = 8;                      // 32-bit words per thread
constexpr int kBitmapTile = kScanBlock * kBitmapWords;
// Threads that write the rows of a tile: 256 leave what is left of its chain (a
// room's densest tile 13.8 us, 11.6, and 10.2 with 1024), 1024 cost a cloud whose
// tiles are mostly empty their launch (18.6 us, and 27.3).
constexpr int kEmitBlock = 512;
constexpr int kBitmapRows = 8192;                    // of a tile whose keys are in LDS together
// persistent block 0 in the bitmap form: the tile bases of the largest bitmap
// first, so that the bitmap itself always starts at the same place
constexpr long long kBitmapMaxTiles = 2 * ((1ll << (kBitmapMaxBits - 5)) / kBitmapTile);   // several bitmaps in one block
constexpr size_t kBitmapBasesBytes = (((kBitmapMaxTiles + 1) * 4 + 255) / 256) * 256;

template <typename CT, typename IT>
__device__ __forceinline__ unsigned long long target_key(const CT *__restrict__ coords, long long i,
                                                         const TargetSpec &spec,
                                                         const IT *__restrict__ batch_dims) {
  unsigned long long key = 0;
#pragma unroll
  for (int k = 0; k < MNT_MAX_NDIM; ++k) {
    if (k < spec.ndim) {
      long long cell = cell_of(static_cast<long long>(coords[i * spec.ndim + k]), spec, k);
      key |= (static_cast<unsigned long long>(cell - spec.base[k]) & spec.mask[k]) << spec.shift[k];
    }
  }
  if (spec.num_batches > 0) {
    key |= static_cast<unsigned long long>(batch_of<IT>(i, batch_dims, spec.num_batches))
           << spec.batch_shift;
  }
  return key;
}

// Sets the bit of every row's key (all threads of the launch share the rows).
template <typename CT, typename IT>
__device__ __forceinline__ void mark_rows(const CT *__restrict__ coords, long long n, const TargetSpec &spec,
                                          const IT *__restrict__ batch_dims, unsigned *__restrict__ bitmap) {
  // Rows that follow each other in a sorted cloud fall into the same word of
  // the bitmap more often than not (their cells differ in the last coordinate
  // only): a run of neighbouring lanes with one word ORs its bits into the
  // run's first lane, which issues the run's only atomic.
  const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
  const int lane = static_cast<int>(lane_id());
  for (long long first = static_cast<long long>(blockIdx.x) * blockDim.x; first < n; first += stride) {
    const long long i = first + threadIdx.x;
    const bool valid = i < n;
    const unsigned long long key = valid ? target_key<CT, IT>(coords, i, spec, batch_dims) : 0ull;
    const unsigned word = valid ? static_cast<unsigned>(key >> 5) : 0xffffffffu;   // no word has this index
    unsigned bits = valid ? 1u << (key & 31u) : 0u;
    for (int off = 1; off < kWave; off <<= 1) {
      const unsigned next_word = __shfl_down(word, off);
      const unsigned next_bits = __shfl_down(bits, off);
      if (lane + off < kWave && next_word == word) bits |= next_bits;
    }
    const unsigned word_before = __shfl_up(word, 1);
    if (valid && (lane == 0 || word_before != word)) atomicOr(&bitmap[word], bits);
  }
}

// Exclusive scan of `tiles` counts in place by one workgroup of 1 024 threads; one
// more entry receives the total, which every thread gets back.
__device__ __forceinline__ unsigned scan_in_place(unsigned *__restrict__ tile_sums, int tiles) {
  __shared__ unsigned wave_sums[1024 / kWave];
  const int t = threadIdx.x;
  const int chunk = (tiles + 1023) / 1024;
  const int lo = t * chunk;
  const int hi = min(tiles, lo + chunk);
  unsigned sum = 0;
  for (int i = lo; i < hi; ++i) sum += tile_sums[i];
  // scan of the 1 024 per-thread sums: inside each wavefront by shuffles, then
  // every thread adds the wavefronts before its own
  unsigned inclusive = sum;
  for (int off = 1; off < kWave; off <<= 1) {
    const unsigned v = __shfl_up(inclusive, off);
    if (static_cast<int>(lane_id()) >= off) inclusive += v;
  }
  const int w = t >> 6;
  if (lane_id() == kWave - 1) wave_sums[w] = inclusive;
  __syncthreads();
  unsigned before = 0, all = 0;
  for (int ww = 0; ww < 1024 / kWave; ++ww) {
    const unsigned v = wave_sums[ww];
    before += ww < w ? v : 0u;
    all += v;
  }
  unsigned run = before + inclusive - sum;
  for (int i = lo; i < hi; ++i) {
    const unsigned v = tile_sums[i];
    tile_sums[i] = run;
    run += v;
  }
  if (t == 1023) tile_sums[tiles] = all;
  return all;
}

// Writes the rows of one bitmap tile (its first row has rank `tile_base`, the
// first behind it rank `tile_end`, the bitmap holds `rows` in all) and the batch
// boundaries that fall into it, and clears its words.  word_info (nullable)
// takes the bits of every non-empty word and the rank of its first row.
template <typename CT, typename IT>
__device__ __forceinline__ void emit_bitmap_tile(unsigned *__restrict__ bitmap, long long words, int tile,
                                                 unsigned tile_base, unsigned tile_end, unsigned rows,
                                                 const TargetSpec &spec, CT *__restrict__ out,
                                                 IT *__restrict__ batch_dims_out, uint2 *__restrict__ word_info) {
  constexpr int kEmitWords = kBitmapTile / kEmitBlock;
  const long long base = static_cast<long long>(tile) * kBitmapTile + threadIdx.x * kEmitWords;
  if (batch_dims_out != nullptr && tile == 0 && threadIdx.x == 0) batch_dims_out[spec.num_batches] = static_cast<IT>(rows);
  // a tile without a set bit has nothing to write but the batch boundaries in it
  if (tile_base == tile_end) {
    if (batch_dims_out != nullptr) {
      for (int g = threadIdx.x; g < spec.num_batches; g += kEmitBlock) {
        const unsigned long long word = (static_cast<unsigned long long>(g) << spec.batch_shift) >> 5;
        if (word / kBitmapTile == static_cast<unsigned long long>(tile)) batch_dims_out[g] = static_cast<IT>(tile_base);
      }
    }
    return;
  }
  unsigned word[kEmitWords];
  unsigned count = 0;
#pragma unroll
  for (int r = 0; r < kEmitWords; ++r) {
    word[r] = base + r < words ? bitmap[base + r] : 0u;
    count += __popc(word[r]);
  }
  // Set bits cluster (cells that differ in the last coordinate share a word):
  // a thread that walked its own 8 words would hold up its wavefront for up to
  // 256 rows while others have none.  The tile's non-empty words, with the rank
  // of their first row, are therefore listed in LDS and dealt round-robin, and
  // what is walked leaves the rows' keys in LDS, in their order: rows written
  // from there are neighbours in neighbouring lanes, where a thread that wrote
  // its word's rows itself sent 64 lanes to 64 lines for every coordinate (pass
  // over 150 000 rows of a room, one level 19.4 us, now 11.6).
  __shared__ unsigned s_word[kBitmapTile], s_rank[kBitmapTile];
  __shared__ unsigned short s_at[kBitmapTile], s_key[kBitmapRows];
  static_assert(kBitmapTile * 32 <= 65536, "a bit's place in the tile in 16 bits");
  unsigned total;
  unsigned run = block_exclusive_scan<kEmitBlock>(count, &total) + tile_base;
  unsigned filled = 0;
#pragma unroll
  for (int r = 0; r < kEmitWords; ++r) filled += word[r] != 0u ? 1u : 0u;
  unsigned listed;
  unsigned slot = block_exclusive_scan<kEmitBlock>(filled, &listed);
#pragma unroll
  for (int r = 0; r < kEmitWords; ++r) {
    const unsigned long long first_key = static_cast<unsigned long long>(base + r) << 5;
    if (batch_dims_out != nullptr && base + r < words) {
      // batch boundaries g << batch_shift that fall into this word
      const unsigned long long step = 1ull << spec.batch_shift;
      for (unsigned long long g = (first_key + step - 1) >> spec.batch_shift;
           g < static_cast<unsigned long long>(spec.num_batches) && (g << spec.batch_shift) < first_key + 32;
           ++g) {
        const unsigned bit = static_cast<unsigned>((g << spec.batch_shift) - first_key);
        batch_dims_out[g] = static_cast<IT>(run + __popc(word[r] & ((1u << bit) - 1u)));
      }
    }
    if (word[r] != 0u) {
      bitmap[base + r] = 0u;                     // the bitmap goes back all zero: the next build clears nothing
      if (word_info != nullptr) word_info[base + r] = make_uint2(word[r], run);
      s_word[slot] = word[r];
      s_rank[slot] = run;
      s_at[slot] = static_cast<unsigned short>(threadIdx.x * kEmitWords + r);
      ++slot;
      run += __popc(word[r]);
    }
  }
  __syncthreads();
  // Keys of the bitmap form have at most 28 bits, and (field + base) * stride
  // worked out in CT wraps exactly as the wide product cut to CT does: the
  // loop stays in 32-bit arithmetic for 32-bit coordinates.
  const unsigned tile_key = static_cast<unsigned>(static_cast<unsigned long long>(tile) * kBitmapTile << 5);
  const unsigned here = tile_end - tile_base;
  for (unsigned from = 0; from < here; from += kBitmapRows) {
    if (from > 0) __syncthreads();
    for (unsigned i = threadIdx.x; i < listed; i += kEmitBlock) {
      unsigned bits = s_word[i];
      unsigned at = s_rank[i] - tile_base - from;            // (below 0: far past the end)
      if (at + 32 < 32 || at < kBitmapRows) {
        const unsigned first_key = static_cast<unsigned>(s_at[i]) << 5;
        while (bits != 0u) {
          const unsigned bit = __ffs(bits) - 1;
          bits &= bits - 1u;
          if (at < kBitmapRows) s_key[at] = static_cast<unsigned short>(first_key | bit);
          ++at;
        }
      }
    }
    __syncthreads();
    const unsigned rows_here = min(here - from, static_cast<unsigned>(kBitmapRows));
    for (unsigned i = threadIdx.x; i < rows_here; i += kEmitBlock) {
      const unsigned key = tile_key | s_key[i];
      CT *row = out + static_cast<long long>(tile_base + from + i) * spec.ndim;
#pragma unroll
      for (int k = 0; k < MNT_MAX_NDIM; ++k) {
        if (k < spec.ndim) {
          const CT cell = static_cast<CT>((key >> spec.shift[k]) & static_cast<unsigned>(spec.mask[k])) +
                          static_cast<CT>(spec.base[k]);
          row[k] = cell * static_cast<CT>(spec.stride[k]);
        }
      }
    }
  }
}

}  // namespace mnt

#define MNT_DISPATCH_CI(coord_dtype, index_dtype, CALL) \
  do {                                                  \
    if (coord_dtype == MNT_INT32 && index_dtype == MNT_INT32) { \
      CALL(int32_t, int32_t);                           \
    } else if (coord_dtype == MNT_INT32) {              \
      CALL(int32_t, int64_t);                           \
    } else if (index_dtype == MNT_INT32) {              \
      CALL(int64_t, int32_t);                           \
    } else {                                            \
      CALL(int64_t, int64_t);                           \
    }                                                   \
  } while (0)
