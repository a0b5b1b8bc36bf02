// Output-stationary forward of a sparse convolution over tiles of targets that
// share their live offsets (tiles.hip): Gather -> GEMM -> Scatter
// (csrc/minuet/cuda/functions/sparse_convolution.cu:504-661) in one kernel
// without buffer rows, multiplying only what a tile has.
#pragma once

#include <algorithm>

#include "conv_device.h"
#include "device_utils.h"
#include "implicit.h"
#include "tiles.h"

namespace mnt {

template <int N>
struct RowSet {
  uint4 v[N];
};

// A lane's share of the source rows of a stage, and the lanes that have one.
template <int N>
struct Rows {
  uint4 v[N];
  unsigned long long takers;
};

typedef unsigned uint4v __attribute__((ext_vector_type(4)));

constexpr unsigned kNowhere = 0xFFFFF000u;     // past the end of every source buffer: reads zeros

// a and b of lanes that differ in one bit of their number change places off the
// diagonal: lanes of `even` keep a and take the other lane's a for their b, the
// others take the other lane's b for their a.  One v_cndmask with a lane
// permutation per word and side; the waits before (a word just written) and
// after (a matrix instruction that reads it) are the hardware's, which no
// compiler sees through inline assembly.
#define MNT_SWAP4(PERM)                                                                              \
  asm("s_mov_b64 vcc, %[even]\n\ts_nop 1\n\t"                                                        \
      "v_cndmask_b32_dpp %0, %12, %8, vcc quad_perm:" PERM " row_mask:0xf bank_mask:0xf\n\t"         \
      "v_cndmask_b32_dpp %1, %13, %9, vcc quad_perm:" PERM " row_mask:0xf bank_mask:0xf\n\t"         \
      "v_cndmask_b32_dpp %2, %14, %10, vcc quad_perm:" PERM " row_mask:0xf bank_mask:0xf\n\t"        \
      "v_cndmask_b32_dpp %3, %15, %11, vcc quad_perm:" PERM " row_mask:0xf bank_mask:0xf\n\t"        \
      "s_not_b64 vcc, vcc\n\t"                                                                       \
      "v_cndmask_b32_dpp %4, %8, %12, vcc quad_perm:" PERM " row_mask:0xf bank_mask:0xf\n\t"         \
      "v_cndmask_b32_dpp %5, %9, %13, vcc quad_perm:" PERM " row_mask:0xf bank_mask:0xf\n\t"         \
      "v_cndmask_b32_dpp %6, %10, %14, vcc quad_perm:" PERM " row_mask:0xf bank_mask:0xf\n\t"        \
      "v_cndmask_b32_dpp %7, %11, %15, vcc quad_perm:" PERM " row_mask:0xf bank_mask:0xf\n\ts_nop 1" \
      : "=&v"(x.x), "=&v"(x.y), "=&v"(x.z), "=&v"(x.w), "=&v"(y.x), "=&v"(y.y), "=&v"(y.z),          \
        "=&v"(y.w)                                                                                   \
      : "v"(a.x), "v"(a.y), "v"(a.z), "v"(a.w), "v"(b.x), "v"(b.y), "v"(b.z), "v"(b.w),              \
        [even] "s"(even)                                                                             \
      : "vcc", "scc")

template <int BIT>
__device__ __forceinline__ void swap_lanes(uint4 &a, uint4 &b) {
  uint4 x, y;
  if constexpr (BIT == 0) {
    const unsigned long long even = 0x5555555555555555ull;
    MNT_SWAP4("[1,0,3,2]");
  } else {
    const unsigned long long even = 0x3333333333333333ull;
    MNT_SWAP4("[2,3,0,1]");
  }
  a = x;
  b = y;
}
#undef MNT_SWAP4

// The row start of the i-th lane of the lane's KS (four or two).
template <int KS>
__device__ __forceinline__ unsigned row_of_lane(unsigned row_at, int i) {
  const int v = static_cast<int>(row_at);
  if (KS == 2) {
    return static_cast<unsigned>(i == 0 ? __builtin_amdgcn_mov_dpp(v, 0xA0, 0xf, 0xf, true)
                                        : __builtin_amdgcn_mov_dpp(v, 0xF5, 0xf, 0xf, true));
  }
  return static_cast<unsigned>(i == 0   ? __builtin_amdgcn_mov_dpp(v, 0x00, 0xf, 0xf, true)
                               : i == 1 ? __builtin_amdgcn_mov_dpp(v, 0x55, 0xf, 0xf, true)
                               : i == 2 ? __builtin_amdgcn_mov_dpp(v, 0xAA, 0xf, 0xf, true)
                                        : __builtin_amdgcn_mov_dpp(v, 0xFF, 0xf, 0xf, true));
}

// The part `step` of turning KS lanes' pieces round: before, piece i of lane j
// is piece j of lane i's row; after all KS steps, piece i of its own.
template <int KS>
__device__ __forceinline__ void turn_rows(uint4 *v, int step) {
  if (step == 0) swap_lanes<0>(v[0], v[1]);
  if constexpr (KS == 4) {
    if (step == 1) swap_lanes<0>(v[2], v[3]);
    if (step == 2) swap_lanes<1>(v[0], v[2]);
    if (step == 3) swap_lanes<1>(v[1], v[3]);
  }
}

struct TiledShape {
  long long num_targets;
  int slots;                   // offsets of the map
  int K, N;
  int chunks;                  // 128-byte pieces of a source row
  int packed_row, packed_rows; // of the packed weights, elements
};

// A workgroup takes a tile of 128 targets (32 per wavefront) and 32 * NB output
// channels, and walks the live offsets, 32 * KS bytes of a source row per stage.
// TILED: the tiles of tiles.hip; otherwise 128 consecutive targets under every
// offset of the dense map.  Tiled sums are those of implicit_forward_kernel bit
// for bit (ascending offsets, the same 16 products per matrix instruction) while
// weights are finite, so that a layer may change from one to the other between
// two calls.  A weight that is not reaches the targets that share a wavefront
// with one that uses its offset, in either kernel; which those are differs.
// KEEP (rows of up to 64 bytes under more than 128 channels): those that have a
// source under its offset only (keep_to_sources), as in the three kernels.
// PAIRED (rows of up to 64 bytes): a stage is two offsets, one per half of the
// wavefront's lanes, which halves what a stage costs besides its products.
// WHOLE: a source row is exactly one stage (or half of one, PAIRED).
// QUADS: KS lanes read neighbouring pieces of one row and turn them round among
// themselves.  The first-level cache looks up one line per clock: 64 lanes on
// 64 lines take 64 clocks per load instruction, in fours 16 (measured: 254 and
// 131 clocks per 32 rows of 128 bytes, indices included).  Without tiles the
// lane permutations make a lone wavefront slower (13.4 against 11.2 us at 25 000
// targets); where they pay with tiles is told at the launch.
// GROUPS = 2: two sets of four wavefronts take every second stage each and
// their sums meet in LDS, for launches of one workgroup per compute unit or
// less, which wait for a tile's longest chain of stages.
//
// What bounds it: on small clouds that chain (0.3 us a stage), on large ones
// the address units and the path from the second-level cache.  At a million
// targets under 125 offsets, 25 M source rows of 128 bytes in 0.42 ms, the
// address units are busy 89 % of the time and the matrix pipes 38 %; of 46 M
// reads of the second-level cache four in five are hits there.  64 -> 64
// channels, 16-bit, us a layer in implicit_forward_kernel and here: 3 000
// targets of an object 14.9 / 8.8, 25 000 of a LiDAR scan 14.9 / 10.3, 60 000
// of a room 18.2 / 17.4; in tiles, LiDAR, 200 000 48.6 / 27, a
// million under 5 x 5 x 5 836 / 403.
template <typename T, int NB, int KS, bool TILED, bool PAIRED, bool WHOLE, bool QUADS, int GROUPS, bool KEEP>
__global__ __launch_bounds__(256 * GROUPS) void tiled_forward_kernel(
    const T *__restrict__ sources, unsigned source_bytes, const T *__restrict__ wt,
    const int *__restrict__ kernel_map, TileView tiles, TiledShape s, unsigned char *__restrict__ out, Epilogue ep) {
  constexpr int ES = static_cast<int>(sizeof(T));
  static_assert(!PAIRED || (!TILED && KS == 4), "tiles keep the order of the offsets");
  constexpr int Np = NB * 32;
  constexpr int kStageBytes = KS * 32;
  constexpr int kRowPieces = 2 * KS;                     // 16-byte pieces of a weight row per stage
  constexpr int kWRows = 256 / kRowPieces;               // weight rows the workgroup loads at a time
  constexpr int kWPieces = (Np + kWRows - 1) / kWRows;   // pieces per thread and stage
  constexpr int kLdsRow = kStageBytes + 16;
  constexpr int kZeros = KS * 32;                        // after the rows of a block of 32 channels
  constexpr int kBlockStride = 32 * kLdsRow + kZeros;
  constexpr int kBufferBytes = NB * kBlockStride;
  constexpr int kSlotsPerStage = PAIRED ? 2 : 1;
  constexpr int kMeetBytes = NB * (GROUPS - 1) * 16384;
  constexpr int kLdsBytes = std::max({2 * GROUPS * kBufferBytes, 4 * std::min(NB, GROUPS) * kTurnBytes, kMeetBytes});
  __shared__ __align__(16) unsigned char lds[kLdsBytes];
  const long long tile = blockIdx.x;
  const int live = TILED ? __builtin_amdgcn_readfirstlane(tiles.counts[tile]) : s.slots;
  if (TILED && live == 0) return;
  const int chunks = PAIRED || WHOLE ? 1 : s.chunks;
  const int first_channel = blockIdx.y * Np;
  const int tid = threadIdx.x & 255;
  const int group = GROUPS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31;
  const int h = lane >> 5;

  // kernel-map entries (a slot past the live ones is read and not used)
  const __amdgpu_buffer_rsrc_t map_buffer = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int *>(TILED ? tiles.sources + tile * s.slots * kTileTargets : kernel_map), 0,
      s.slots * kTileTargets * 4, 0x00020000);
  const unsigned map_at = static_cast<unsigned>(wv * 32 + r) * 4u;
  const long long target = min(tile * kTileTargets + wv * 32 + r, s.num_targets - 1);
  auto load_index = [&](int slot) -> int {
    if (!TILED) return kernel_map[min(PAIRED ? slot + h : slot, s.slots - 1) * s.num_targets + target];
    return __builtin_amdgcn_raw_buffer_load_b32(map_buffer, map_at, min(slot, s.slots - 1) * (kTileTargets * 4), 0);
  };
  // the numbers of a tile's live offsets: lane l holds the l-th and the (64 + l)-th
  const int *offsets_at = tiles.offsets + tile * s.slots;
  const int off_lo = TILED && lane < live ? offsets_at[lane] : 0;
  const int off_hi = TILED && 64 + lane < live ? offsets_at[64 + lane] : 0;
  auto offset_of = [&](int slot) -> unsigned {
    if (!TILED) return static_cast<unsigned>(min(slot, s.slots - 1));
    const int lo = __builtin_amdgcn_readlane(off_lo, slot & 63);
    const int hi = __builtin_amdgcn_readlane(off_hi, slot & 63);
    return static_cast<unsigned>(slot < 64 ? lo : hi);
  };
  // the targets whose output pieces this lane stores (-1: none)
  auto row_of = [&](int place) -> int {
    const long long t = tile * kTileTargets + place;
    return TILED ? tiles.rows[t] : t < s.num_targets ? static_cast<int>(t) : -1;
  };
  constexpr int EPV = 16 / ES;
  constexpr int kOutPieces = 32 / EPV;
  constexpr int kPieces = 32 * kOutPieces / 64;
  int out_row[kPieces];
#pragma unroll
  for (int i = 0; i < kPieces; ++i) out_row[i] = row_of(wv * 32 + (lane + i * 64) / kOutPieces);

  floatx16 acc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[b][j] = 0.0f;
  }

  struct Cursor {
    int slot, chunk;
  };
  auto next = [&](Cursor c) -> Cursor {
    if (PAIRED || WHOLE || ++c.chunk == chunks) {
      c.chunk = 0;
      c.slot += kSlotsPerStage * GROUPS;
    }
    return c;
  };
  const unsigned offset_stride = static_cast<unsigned>(s.packed_rows * s.packed_row * ES);
  const __amdgpu_buffer_rsrc_t weight_buffer = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T *>(wt), 0, static_cast<unsigned>(s.slots) * offset_stride, 0x00020000);
  // piece i of this thread: 16 bytes of weight row tid / kRowPieces + kWRows i
  // (threads past the last row repeat it)
  unsigned w_at[kWPieces], w_put[kWPieces];
  const int w_piece = tid % kRowPieces;
#pragma unroll
  for (int i = 0; i < kWPieces; ++i) {
    const int row = min(tid / kRowPieces + kWRows * i, Np - 1);
    const int channel = min(first_channel + row, s.packed_rows - 1);
    // (in 24 bits where the 64-bit product's register pair came to hold what is being loaded: 4 to 8 % of a layer)
    const int channel_at = KEEP ? static_cast<int>(__umul24(channel, s.packed_row * ES)) : channel * s.packed_row * ES;
    w_at[i] = static_cast<unsigned>(channel_at + (PAIRED ? w_piece & 3 : w_piece) * 16);
    w_put[i] = static_cast<unsigned>(row / 32 * kBlockStride + row % 32 * kLdsRow + w_piece * 16) +
               group * 2 * kBufferBytes;
  }
  auto load_w = [&](const Cursor &c) -> RowSet<kWPieces> {
    RowSet<kWPieces> set;
    unsigned lane_part = 0, all_part = 0;
    if (PAIRED) {
      const unsigned a = offset_of(c.slot) * offset_stride, b = offset_of(c.slot + 1) * offset_stride;
      lane_part = w_piece < 4 ? a : b;
    } else {
      all_part = offset_of(c.slot) * offset_stride + c.chunk * kStageBytes;
    }
#pragma unroll
    for (int i = 0; i < kWPieces; ++i) {
      const uint4v v = __builtin_amdgcn_raw_buffer_load_b128(weight_buffer, w_at[i] + lane_part, all_part, 0);
      set.v[i] = make_uint4(v.x, v.y, v.z, v.w);
    }
    return set;
  };
  auto store_w = [&](int buffer, const RowSet<kWPieces> &set) {
#pragma unroll
    for (int i = 0; i < kWPieces; ++i) {
      *reinterpret_cast<uint4 *>(lds + buffer * kBufferBytes + w_put[i]) = set.v[i];
    }
  };
  const __amdgpu_buffer_rsrc_t source_buffer = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T *>(sources), 0, source_bytes, 0x00020000);
  const unsigned row_bytes = static_cast<unsigned>(s.K) * ES;
  // Half h of the lanes takes the pieces 2 i + h of a row's stage (PAIRED: of its
  // own offset's row all four); with QUADS the i-th lane of KS loads the i-th of
  // them for each of the KS rows.
  constexpr unsigned kPieceStep = PAIRED ? 16u : 32u;
  const unsigned lane_at = (PAIRED ? 0u : h * 16u) + (QUADS ? (lane & (KS - 1)) * kPieceStep : 0u);
  auto load_rows = [&](int index, const Cursor &c) -> Rows<KS> {
    Rows<KS> set;
    const unsigned chunk_at = WHOLE || PAIRED ? 0u : static_cast<unsigned>(c.chunk) * kStageBytes;
    const bool take = index >= 0 && (PAIRED ? c.slot + h : c.slot) < live;
    const unsigned row_at = take ? static_cast<unsigned>(index) * row_bytes : kNowhere;
    set.takers = __ballot(take);
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      unsigned at = (QUADS ? row_of_lane<KS>(row_at, i) : row_at + i * kPieceStep) + lane_at;
      if (!WHOLE && chunk_at + lane_at + (QUADS ? 0u : i * kPieceStep) >= row_bytes) at = kNowhere;
      const uint4v v = __builtin_amdgcn_raw_buffer_load_b128(source_buffer, at, chunk_at, 0);
      set.v[i] = make_uint4(v.x, v.y, v.z, v.w);
    }
    return set;
  };

  // Two register sets of everything.  At stage o the weights of stage o + 1 go
  // to LDS and those of o + 3 are asked for; the rows of o + 2 (QUADS: o + 3,
  // those of o + 1 being turned round between the products) and the map entries
  // two stages later still.  Every load is issued in every stage, lanes without
  // a source reading past the end: what is in flight is the same on every path,
  // so that no wait is longer than it must be.  (With the loads under a branch
  // the compiler had to wait for the youngest one: a trip to memory per stage,
  // 0.5 us of it on clouds that leave one wavefront to a SIMD.)
  const Cursor c0 = {group * kSlotsPerStage, 0};
  const Cursor c1 = next(c0), c2 = next(c1), c3 = next(c2);
  int m0 = load_index(c0.slot), m1 = load_index(c1.slot);
  RowSet<kWPieces> w1 = load_w(c0), w0;
  Rows<KS> a0 = load_rows(m0, c0), a1;
  w0 = load_w(c1);
  m0 = load_index(c2.slot);
  a1 = load_rows(m1, c1);
  store_w(0, w1);
  for (int i = threadIdx.x; i < 2 * GROUPS * NB * kZeros / 16; i += 256 * GROUPS) {
    *reinterpret_cast<uint4 *>(lds + i / (kZeros / 16) * kBlockStride + 32 * kLdsRow + i % (kZeros / 16) * 16) =
        make_uint4(0u, 0u, 0u, 0u);
  }
  w1 = load_w(c2);
  m1 = load_index(c3.slot);
  __syncthreads();
  Cursor at_a = c2, at_w = c3, at_m = next(c3);
  // An offset that none of a wavefront's 32 targets has a source under is
  // multiplied like the others, but by zeros: one infinite or undefined weight
  // there would make all of their sums undefined.  (Leaving the products out
  // needs a branch around them: 36 % slower where QUADS turns rows between them.)
  const unsigned w_here = static_cast<unsigned>(r * kLdsRow + (PAIRED ? h * 64 : h * 16)) + group * 2 * kBufferBytes;
  const unsigned w_none = 32 * kLdsRow + group * 2 * kBufferBytes;
  auto weights_for = [&](unsigned long long takers) -> unsigned {
    const bool any = PAIRED ? (h == 0 ? static_cast<unsigned>(takers) : static_cast<unsigned>(takers >> 32)) != 0u
                            : takers != 0ull;
    return any ? w_here : w_none;
  };
  int left = ((live + kSlotsPerStage * GROUPS - 1) / (kSlotsPerStage * GROUPS) * chunks + 1) >> 1;
  Rows<KS> rows;
#define MNT_STAGE(A, W, M, BUF)                                                                    \
  {                                                                                                \
    store_w(1 - (BUF), W);                                                                         \
    const unsigned w_get = weights_for(QUADS ? rows.takers : A.takers);                            \
    uint4 f[KS][NB];                                                                               \
    _Pragma("unroll") for (int kk = 0; kk < KS; ++kk) {                                            \
      _Pragma("unroll") for (int b = 0; b < NB; ++b) {                                             \
        f[kk][b] = *reinterpret_cast<const uint4 *>(lds + (BUF) * kBufferBytes + w_get +           \
                                                    b * kBlockStride + kk * kPieceStep);           \
      }                                                                                            \
    }                                                                                              \
    __builtin_amdgcn_sched_barrier(0);                                                             \
    W = load_w(at_w);                                                                              \
    Rows<KS> coming = A;                                                                           \
    if (!QUADS) rows = A;                                                                          \
    _Pragma("unroll") for (int kk = 0; kk < KS; ++kk) {                                            \
      _Pragma("unroll") for (int b = 0; b < NB; ++b) acc[b] = Mfma<T>::run(f[kk][b], rows.v[kk], acc[b]); \
      if (QUADS) {                                                                                 \
        __builtin_amdgcn_sched_barrier(0);                                                         \
        turn_rows<KS>(coming.v, kk);                                                                   \
        __builtin_amdgcn_sched_barrier(0);                                                         \
      }                                                                                            \
    }                                                                                              \
    if (QUADS) rows = coming;                                                                      \
    A = load_rows(M, at_a);                                                                        \
    M = load_index(at_m.slot);                                                                     \
    at_w = next(at_w);                                                                             \
    at_a = next(at_a);                                                                             \
    at_m = next(at_m);                                                                             \
    __syncthreads();                                                                               \
  }
  if (QUADS) {
    rows = a0;
#pragma unroll
    for (int i = 0; i < KS; ++i) turn_rows<KS>(rows.v, i);
    a0 = load_rows(m0, at_a);
    m0 = load_index(at_m.slot);
    at_a = next(at_a);
    at_m = next(at_m);
    do {
      MNT_STAGE(a1, w0, m1, 0)
      MNT_STAGE(a0, w1, m0, 1)
    } while (--left != 0);
  } else {
    do {
      MNT_STAGE(a0, w0, m0, 0)
      MNT_STAGE(a1, w1, m1, 1)
    } while (--left != 0);
  }
#undef MNT_STAGE

  // Group g ends with the blocks b of which b % GROUPS == g; the others hand
  // theirs over, in the order of their numbers.
  if (GROUPS > 1) {
    float4 *const meet = reinterpret_cast<float4 *>(lds) + wv * 256 + lane;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int from = (group - b % GROUPS + GROUPS) % GROUPS;        // 0: the owner
      if (from == 0) continue;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        meet[(b * (GROUPS - 1) + from - 1) * 1024 + q * 64] =
            make_float4(acc[b][q * 4], acc[b][q * 4 + 1], acc[b][q * 4 + 2], acc[b][q * 4 + 3]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (b % GROUPS != group) continue;
#pragma unroll
      for (int g = 0; g < GROUPS - 1; ++g) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float4 f = meet[(b * (GROUPS - 1) + g) * 1024 + q * 64];
          acc[b][q * 4] += f.x;
          acc[b][q * 4 + 1] += f.y;
          acc[b][q * 4 + 2] += f.z;
          acc[b][q * 4 + 3] += f.w;
        }
      }
    }
    __syncthreads();
  }
  float seen = 0.0f;                           // the largest of the sums that are stored
  auto keep = [&]() {
    if constexpr (KEEP) {
      keep_to_sources<T, NB, GROUPS>(
          acc, seen, sources, s.K, wt, s.packed_row, s.packed_rows, first_channel, s.N, h, group, live,
          [&](int slot) {
            return TILED ? tiles.sources[(tile * s.slots + slot) * kTileTargets + wv * 32 + r]
                         : kernel_map[slot * s.num_targets + target];
          },
          [&](int slot) { return TILED ? offsets_at[slot] : slot; },
          [&]() { return static_cast<long long>(row_of(wv * 32 + r)); }, ep, out);
    }
  };
  if ((static_cast<long long>(s.N) * ES) % 16 != 0) {      // output rows are no whole 16-byte pieces
    const int row = row_of(wv * 32 + r);
    if (!KEEP && row < 0) return;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (b % GROUPS != group || (KEEP && row < 0)) continue;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int ch = first_channel + b * 32 + q * 8 + h * 4;
        if (ch >= s.N) continue;               // N % 4 == 0: a group of four is all in or all out
        float v[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = acc[b][q * 4 + x];
        if constexpr (KEEP) seen = largest_of<4>(v, seen);
        finish_four<T>(v, ep, row, ch, s.N, out);
      }
    }
    keep();
    return;
  }
  unsigned char *turn = lds + (group * 4 + wv) * kTurnBytes;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if (first_channel + b * 32 >= s.N) break;
    if (b % GROUPS != group) continue;
    if constexpr (KEEP) seen = largest_of<16>(acc[b], seen);
    store_turned_rows<T>(acc[b], turn, lane, r, h, out_row, first_channel + b * 32, s.N, ep, out);
  }
  keep();
}

template <typename T>
void tiled_forward(const T *sources, const T *packed, const int *kernel_map, const int *tiles, int64_t S, int64_t Tn,
                   int64_t O, int64_t K, int64_t N, const Epilogue &ep, T *out, hipStream_t stream) {
  const TileLayout l(Tn, O);
  const bool tiled = tiles != nullptr;
  const TileView view = {tiles, tiles + l.counts_at, tiles + l.offsets_at, tiles + l.sources_at};
  const int kc = kChunkBytes / static_cast<int>(sizeof(T));
  const int row_bytes = static_cast<int>(K * sizeof(T));
  TiledShape s;
  s.num_targets = Tn;
  s.slots = static_cast<int>(O);
  s.K = static_cast<int>(K);
  s.N = static_cast<int>(N);
  s.packed_row = static_cast<int>(div_ceil(K, kc) * kc);
  s.packed_rows = static_cast<int>(div_ceil(N, 32) * 32);
  const bool paired = !tiled && row_bytes <= 64 && O > 1;
  const int stage_bytes = tiled && row_bytes <= 64 ? 64 : 128;
  s.chunks = static_cast<int>(div_ceil(row_bytes, stage_bytes));
  const bool whole = row_bytes == (paired ? 64 : stage_bytes);
  const unsigned source_bytes = static_cast<unsigned>(S * row_bytes);
  // Channel blocks per workgroup: as many as there are, up to four, because a
  // workgroup of its own for other channels reads the source rows again; fewer
  // where that leaves compute units idle (3 000 targets, 64 -> 64 channels: 8.1
  // us with one block, 10.1 with two).
  const int cols = s.packed_rows / 32, cus = compute_units();
  const int64_t filled = div_ceil(Tn, kTileTargets);
  int nb = std::min(4, cols);
  while (nb > 1 && filled * div_ceil(cols, nb - 1) <= cus) --nb;
  const int y = static_cast<int>(div_ceil(cols, nb));
  // Two sets of wavefronts up to a workgroup per compute unit.
  const bool two = !tiled && filled * y <= cus && O * s.chunks > 2;
  // Lanes load together (64 -> 64 channels, 100 000 targets 18.4 against 19.3 us,
  // 59 000 of a LiDAR level 17.7 and 22.5, though 70 000 of a room 17.9 and 16.8);
  // tiles of large kernels have more stages to hide the latency behind and gain
  // from a quarter of a million targets on only.
  const bool quads = nb <= 2 && (O <= 32 || 2 * filled >= 16 * cus);
  const bool keep = row_bytes <= 64 && N > 128;
  const dim3 grid(static_cast<unsigned>(tiled ? l.tiles : filled), static_cast<unsigned>(y));
#define MNT_TILED_K(NB, KS, TILED, PAIRED, WHOLE, QUADS, GROUPS, KEEP)                                            \
  tiled_forward_kernel<T, NB, KS, TILED, PAIRED, WHOLE, QUADS, GROUPS, KEEP><<<grid, 256 * GROUPS, 0, stream>>>(  \
      sources, source_bytes, packed, kernel_map, view, s, reinterpret_cast<unsigned char *>(out), ep)
#define MNT_TILED(NB, KS, TILED, PAIRED, WHOLE, QUADS, GROUPS)                 \
  if ((PAIRED || KS == 2) && keep) {                                           \
    MNT_TILED_K(NB, KS, TILED, PAIRED, WHOLE, QUADS, GROUPS, (PAIRED || KS == 2)); \
  } else {                                                                     \
    MNT_TILED_K(NB, KS, TILED, PAIRED, WHOLE, QUADS, GROUPS, false);           \
  }
#define MNT_TILED_Q(NB, KS, WHOLE)                               \
  if (NB <= 2 && quads) {                                        \
    MNT_TILED(NB, KS, true, false, WHOLE, (NB <= 2), 1)          \
  } else {                                                       \
    MNT_TILED(NB, KS, true, false, WHOLE, false, 1)              \
  }
#define MNT_TILED_G(NB, PAIRED, WHOLE)                           \
  if (two) {                                                     \
    MNT_TILED(NB, 4, false, PAIRED, WHOLE, false, 2)             \
  } else {                                                       \
    MNT_TILED(NB, 4, false, PAIRED, WHOLE, false, 1)             \
  }
#define MNT_TILED_N(NB)                                          \
  if (tiled && stage_bytes == 64) {                              \
    if (whole) {                                                 \
      MNT_TILED_Q(NB, 2, true)                                   \
    } else {                                                     \
      MNT_TILED_Q(NB, 2, false)                                  \
    }                                                            \
  } else if (tiled) {                                            \
    if (whole) {                                                 \
      MNT_TILED_Q(NB, 4, true)                                   \
    } else {                                                     \
      MNT_TILED_Q(NB, 4, false)                                  \
    }                                                            \
  } else if (paired) {                                           \
    if (whole) {                                                 \
      MNT_TILED_G(NB, true, true)                                \
    } else {                                                     \
      MNT_TILED_G(NB, true, false)                               \
    }                                                            \
  } else if (whole) {                                            \
    MNT_TILED_G(NB, false, true)                                 \
  } else {                                                       \
    MNT_TILED_G(NB, false, false)                                \
  }
  switch (nb) {
    case 1: MNT_TILED_N(1) break;
    case 2: MNT_TILED_N(2) break;
    case 3: MNT_TILED_N(3) break;
    default: MNT_TILED_N(4) break;
  }
#undef MNT_TILED_N
#undef MNT_TILED_G
#undef MNT_TILED_Q
#undef MNT_TILED
#undef MNT_TILED_K
  check_launch("tiled_forward_kernel");
}

}  // namespace mnt

