// Output-stationary forward of a sparse convolution whose operands stream
// through LDS: Gather -> GEMM -> Scatter
// (csrc/minuet/cuda/functions/sparse_convolution.cu:504-661) in one kernel
// without buffer rows.
#pragma once

#include <algorithm>

#include "conv_device.h"
#include "device_utils.h"
#include "implicit.h"
#include "tiles.h"

namespace mnt {

typedef int int4v __attribute__((ext_vector_type(4)));

constexpr int kStreamedStage = 128;            // bytes of a row
constexpr int kStreamedLoaders = 4;            // wavefronts of a workgroup that load
constexpr unsigned kPastEnd = 0xFFFFF000u;     // past the end of every source buffer: reads zeros

struct StreamedShape {
  long long num_targets;
  int slots;                   // offsets of the map
  int row_bytes;               // of a source row
  int N;
  int packed_row_bytes, packed_rows;
};

__device__ __forceinline__ int4v buffer_words(const void *base, unsigned bytes) {
  const unsigned long long at = reinterpret_cast<unsigned long long>(base);
  int4v r;
  r.x = __builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<unsigned>(at)));
  r.y = __builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<unsigned>(at >> 32) & 0xffffu));
  r.z = __builtin_amdgcn_readfirstlane(static_cast<int>(bytes));
  r.w = 0x00020000;
  return r;
}

// Loads past the registers: 16 (4) bytes of each lane go to LDS at lds_at + 16
// (4) x lane, zeros where a lane reads past the buffer's end.  In assembly so
// that the compiler does not wait for the youngest of them at the next read of
// LDS: who reads has waited (wait_loads) and met the others (meet) first.
__device__ __forceinline__ void load_lds16(const int4v &buffer, unsigned at, unsigned all, unsigned lds_at) {
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(at), "s"(buffer),
               "s"(all), "s"(lds_at)
               : "memory");
}
__device__ __forceinline__ void load_lds4(const int4v &buffer, unsigned at, unsigned lds_at) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dword %0, %1, 0 offen lds" ::"v"(at), "s"(buffer),
               "s"(lds_at)
               : "memory");
}
template <int LEFT>
__device__ __forceinline__ void wait_loads() {
  static_assert(LEFT >= 0 && LEFT < 64, "the counter has six bits");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LEFT) : "memory");
}
__device__ __forceinline__ void meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// A workgroup of MW x NW x KW wavefronts that multiply and four that load takes TM
// targets and TN output channels; a stage is 128 bytes of the source rows and of
// the weights under one offset, CH stages an offset, RING of them in LDS.
//
// Those that load ask for stage L as soon as all have read stage L - RING, and
// for map entries kAhead offsets before their rows.  Those that multiply read a
// stage's pieces while they multiply those of the stage before; KW of them share
// the pieces of a stage and add up at the end, because 64 x 64 sums a wavefront
// need the fewest reads of LDS per product.
//
// TILED: the tiles of tiles.hip with their live offsets; otherwise consecutive
// targets under every offset of the dense map.  For one shape both add up the
// same products in the same order.
//
// What bounds it, by stamps in a copy of it: a compute unit takes 17.5 clocks for a load of 1 KB, whether
// of one piece or of eight rows of 128 bytes (in the order of the matrix
// instruction, 32 rows of 32 bytes, 70), and a stage of 128 targets and 64
// channels is 24 of them: 0.175 us of the 0.19 it takes.  The rest is how evenly
// the workgroups fill the chip (over a launch of 256 -> 256 over 25 600 of a LiDAR scan
// address units are 20 % busy), and about 5 us to start and end.  The wavefronts
// that load are others than those that multiply because one that did both took
// the sum of the two (0.8 us a stage).  Against grouped products and a
// Scatter, us a layer: 128 -> 128 channels over 6 850 targets of objects 23.0 and
// 11.8, over 18 600 of a LiDAR level 27.7 and 17.3 (in tiles), 256 -> 256 over
// 2 000 27.1 and 16.8, over 25 600 of a LiDAR scan 39.5 and 37.1.
//
// A target without a source under an offset takes part with zeros, which one
// infinite or undefined weight would turn into sums that are undefined.  So
// where sums are not finite the workgroup starts again, and every target keeps
// what it has under an offset that it has no source under (the same sums
// wherever those are finite): a test per stage instead cost 15 % of it.
template <typename T, int MW, int NW, int KW, int WM, int WN, int CH, int RING, bool TILED>
__global__ __launch_bounds__(64 * (MW * NW * KW + kStreamedLoaders))
__attribute__((amdgpu_waves_per_eu((MW * NW * KW + kStreamedLoaders + 3) / 4, 8))) void streamed_forward_kernel(
    const T *__restrict__ sources, unsigned source_bytes, const T *__restrict__ wt,
    const int *__restrict__ kernel_map, TileView tiles, StreamedShape s, unsigned char *__restrict__ out,
    Epilogue ep) {
  constexpr int TM = 32 * MW * WM, TN = 32 * NW * WN, BK = kStreamedStage;
  constexpr int NC = MW * NW * KW, NL = kStreamedLoaders;    // wavefronts that multiply, and that load
  constexpr int kRowLanes = BK / 16;                         // lanes that load a row's stage
  constexpr int kLoadRows = 64 / kRowLanes;                  // rows of a load
  constexpr int kWaveRows = TM / NL;                         // of a wavefront that loads
  constexpr int kRowLoads = kWaveRows / kLoadRows, kWeightLoads = TN / NL / kLoadRows;
  constexpr int kLoads = kRowLoads + kWeightLoads;
  static_assert(kRowLoads * NL * kLoadRows == TM && kWeightLoads * NL * kLoadRows == TN, "whole loads");
  static_assert(!TILED || kTileTargets % TM == 0, "whole parts of a tile");
  constexpr int KS = BK / 32 / KW;                           // products along K a wavefront makes of a stage
  static_assert(KS >= 1 && KS * 32 * KW == BK && BK == 128, "stages are dealt out evenly");
  static_assert(RING % CH == 0 && RING >= 2, "whole offsets in the ring");
  constexpr int kSlots = RING / CH;                          // offsets in the ring
  constexpr int kAhead = kSlots + 1;
  constexpr int kEntries = 2 * kSlots + 1 < 8 ? 8 : 16;      // offsets whose map entries are in LDS
  static_assert(2 * kSlots + 1 < kEntries && kWaveRows <= 64, "entries stay until all have read them");
  constexpr int kStage = (TM + TN) * BK;
  // LDS: the ring, where at the end sums meet and rows are turned round; map entries
  constexpr int kBlocks = WM * WN;
  constexpr int kMeetBlock = MW * NW * (KW - 1) * 4096;
  constexpr int kRingBytes = RING * kStage;
  constexpr int kFit = KW == 1 ? kBlocks : kRingBytes / kMeetBlock;
  constexpr int kAtOnce = kFit < kBlocks ? kFit : kBlocks;   // blocks whose sums meet at a time
  static_assert(kAtOnce >= 1 && NC * kTurnBytes <= kRingBytes, "room for the end in the ring");
  constexpr int kEndMeets = KW == 1 ? 0 : 2 * ((kBlocks + kAtOnce - 1) / kAtOnce);
  constexpr int kEntriesAt = kRingBytes;
  constexpr int kAgainAt = kEntriesAt + kEntries * TM * 4;
  __shared__ __align__(16) unsigned char lds[kAgainAt + 16];
  static_assert(kAgainAt + 16 <= 160 * 1024, "LDS of a compute unit");
  const unsigned lds0 =
      static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char *)(lds)));
  volatile int *const again = reinterpret_cast<volatile int *>(lds + kAgainAt);
  constexpr int kParts = TILED ? kTileTargets / TM : 1;      // workgroups of a tile
  const long long tile = blockIdx.x / kParts;
  const int part = blockIdx.x % kParts * TM;
  const int live = TILED ? __builtin_amdgcn_readfirstlane(tiles.counts[tile]) : s.slots;
  if (TILED && live == 0) return;
  const int first_channel = blockIdx.y * TN;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 31, h = lane >> 5;
  const long long first_target = static_cast<long long>(blockIdx.x) * TM;
  // rows lie in LDS with their pieces exchanged so that eight rows' same piece
  // are in eight different places
  auto place = [](int row, int piece) -> int { return piece ^ (row & 7); };
  if (threadIdx.x == 0) *again = 0;

  // All meet when the first stage is there, once a stage, kEndMeets times at the
  // end and once to hear whether all of it is done again.
  if (wv >= NC) {
    const int lw = wv - NC;
    const int4v source_buffer = buffer_words(sources, source_bytes);
    const unsigned offset_stride = static_cast<unsigned>(s.packed_rows * s.packed_row_bytes);
    const int4v weight_buffer = buffer_words(wt, static_cast<unsigned>(s.slots) * offset_stride);
    // (targets past the last one stand for it)
    const int *const entries = TILED ? tiles.sources + tile * s.slots * kTileTargets : kernel_map;
    const long long entry_stride = TILED ? kTileTargets : s.num_targets;
    const unsigned entry_at =
        TILED ? (part + lw * kWaveRows + lane) * 4u
              : static_cast<unsigned>(min(first_target + lw * kWaveRows + lane, s.num_targets - 1)) * 4u;
    // the numbers of a tile's live offsets: lane l holds the l-th and the (64 + l)-th
    const int *offsets_at = tiles.offsets + tile * s.slots;
    int off_lo = TILED && lane < live ? offsets_at[lane] : 0;
    int off_hi = TILED && 64 + lane < live ? offsets_at[64 + lane] : 0;
    const int load_row = lane / kRowLanes;
    unsigned w_at[kWeightLoads];
#pragma unroll
    for (int i = 0; i < kWeightLoads; ++i) {
      const int row = (lw * kWeightLoads + i) * kLoadRows + load_row;
      w_at[i] = static_cast<unsigned>(min(first_channel + row, s.packed_rows - 1) * s.packed_row_bytes +
                                      place(row, lane % kRowLanes) * 16);
    }
    const unsigned piece_at = place(load_row, lane % kRowLanes) * 16u;     // (of later loads' rows the same)
    // the last stage of a row may be longer than what is left of it
    const bool past_row = (CH - 1) * BK + piece_at >= static_cast<unsigned>(s.row_bytes);
    unsigned chunk_at[CH];                     // (in registers: the instruction takes no such constants)
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      chunk_at[c] = c * BK;
      asm volatile("" : "+s"(chunk_at[c]));
    }
    auto load_entries = [&](int slot) {
      if (slot < live && (kWaveRows == 64 || lane < kWaveRows)) {
        load_lds4(buffer_words(entries + slot * entry_stride, static_cast<unsigned>(entry_stride) * 4u), entry_at,
                  __builtin_amdgcn_readfirstlane(lds0 + kEntriesAt + (slot % kEntries * TM + lw * kWaveRows) * 4));
      }
    };
    int index[kRowLoads];
    unsigned starts[kRowLoads], weights = 0;
    auto read_entries = [&](int slot) {
      const int *at = reinterpret_cast<const int *>(lds + kEntriesAt) + slot % kEntries * TM + lw * kWaveRows + load_row;
#pragma unroll
      for (int i = 0; i < kRowLoads; ++i) index[i] = at[i * kLoadRows];
    };
    auto open_offset = [&](int slot) {
#pragma unroll
      for (int i = 0; i < kRowLoads; ++i) {
        const unsigned at = static_cast<unsigned>(index[i]) * static_cast<unsigned>(s.row_bytes) + piece_at;
        starts[i] = index[i] < 0 ? kPastEnd : at;
      }
      int number = slot;
      if (TILED) {
        const int lo = __builtin_amdgcn_readlane(off_lo, slot & 63);
        const int hi = __builtin_amdgcn_readlane(off_hi, slot & 63);
        number = slot < 64 ? lo : hi;
      }
      weights = static_cast<unsigned>(number) * offset_stride;
    };
    auto load_stage = [&](int c, unsigned to) {
#pragma unroll
      for (int i = 0; i < kRowLoads; ++i) {
        const unsigned at = c == CH - 1 && past_row ? kPastEnd : starts[i];
        load_lds16(source_buffer, at, chunk_at[c], to + (lw * kRowLoads + i) * 1024);
      }
#pragma unroll
      for (int i = 0; i < kWeightLoads; ++i) {
        load_lds16(weight_buffer, w_at[i], weights + chunk_at[c], to + TM * BK + (lw * kWeightLoads + i) * 1024);
      }
    };
    for (int turn = 0; turn < 2; ++turn) {
      for (int slot = 0; slot < kSlots + kAhead; ++slot) load_entries(slot);
      wait_loads<0>();
      asm volatile("" : "+v"(off_lo), "+v"(off_hi));         // (loaded: no wait of the compiler's further down)
      read_entries(0);
      open_offset(0);
#pragma unroll
      for (int slot = 0; slot < kSlots; ++slot) {
        if (slot < live) {
#pragma unroll
          for (int c = 0; c < CH; ++c) load_stage(c, lds0 + (slot * CH + c) * kStage);
          read_entries(slot + 1);
          open_offset(min(slot + 1, live - 1));
        }
      }
      if (live >= kSlots) {
        wait_loads<kLoads *(RING - 1)>();
      } else {
        wait_loads<0>();
      }
      meet();
      // All have read stage L - RING when they meet and stage L - RING + 1 has
      // landed; stage L goes where the former was.
      unsigned at = lds0;
      for (int slot = kSlots; slot < live; ++slot) {
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          wait_loads<kLoads *(RING - 2)>();
          meet();
          load_stage(c, at + c * kStage);
          if (c == 0) {
            load_entries(slot + kAhead);
            read_entries(slot + 1);
          }
        }
        open_offset(min(slot + 1, live - 1));
        at = at + CH * kStage == lds0 + kRingBytes ? lds0 : at + CH * kStage;
      }
      for (int stage = min(live, kSlots) * CH; stage > 0; --stage) {
        wait_loads<0>();
        meet();
      }
#pragma unroll
      for (int i = 0; i < kEndMeets; ++i) meet();
      meet();
      if (*again == 0) return;
    }
    return;
  }

  const int wm = wv % MW, wn = wv / MW % NW, wk = wv / (MW * NW);
  unsigned x_at[KS], w_at[KS];
#pragma unroll
  for (int kk = 0; kk < KS; ++kk) {
    const int piece = 2 * (wk * KS + kk) + h;
    x_at[kk] = (wm * WM * 32 + r) * BK + place(r, piece) * 16;
    w_at[kk] = TM * BK + (wn * WN * 32 + r) * BK + place(r, piece) * 16;
  }
  struct Pieces {
    uint4 x[KS][WM], w[KS][WN];
  };
  // the targets whose output pieces this lane stores (-1: none)
  constexpr int kOutPieces = 4, kPieces = 2;
  auto row_of = [&](int target) -> int {
    if (TILED) return tiles.rows[tile * kTileTargets + part + target];
    return first_target + target < s.num_targets ? static_cast<int>(first_target) + target : -1;
  };
  int out_row[WM][kPieces];
#pragma unroll
  for (int a = 0; a < WM; ++a) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) out_row[a][i] = row_of((wm * WM + a) * 32 + (lane + i * 64) / kOutPieces);
  }
  const int total = live * CH;
  unsigned base = 0;
  floatx16 acc[WM][WN];
  auto clear = [&]() {
    base = 0;
#pragma unroll
    for (int a = 0; a < WM; ++a) {
#pragma unroll
      for (int b = 0; b < WN; ++b) {
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[a][b][j] = 0.0f;
      }
    }
  };
  auto read = [&](Pieces &p, int kk) {
#pragma unroll
    for (int a = 0; a < WM; ++a) p.x[kk][a] = *reinterpret_cast<const uint4 *>(lds + base + x_at[kk] + a * 32 * BK);
#pragma unroll
    for (int b = 0; b < WN; ++b) p.w[kk][b] = *reinterpret_cast<const uint4 *>(lds + base + w_at[kk] + b * 32 * BK);
  };
  auto advance = [&]() { base = base + kStage == kRingBytes ? 0 : base + kStage; };
  // Reads go between the products: a wavefront's instructions leave in order, and
  // products behind the reads of all others cost a third of a stage.
  auto multiply = [&](const Pieces &now, Pieces &next) {
    meet();
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      read(next, kk);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int a = 0; a < WM; ++a) {
#pragma unroll
        for (int b = 0; b < WN; ++b) acc[a][b] = Mfma<T>::run(now.w[kk][b], now.x[kk][a], acc[a][b]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    advance();
  };
  auto add_up = [&]() {                        // block b's sums end in wavefronts wk = b % KW
    if (KW == 1) return;
    float4 *const at = reinterpret_cast<float4 *>(lds) + (wn * MW + wm) * ((KW - 1) * 256) + lane;
#pragma unroll
    for (int b0 = 0; b0 < kBlocks; b0 += kAtOnce) {
#pragma unroll
      for (int b = b0; b < b0 + kAtOnce && b < kBlocks; ++b) {
        const int from = (wk - b % KW + KW) % KW;
        if (from == 0) continue;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const floatx16 &v = acc[b / WN][b % WN];
          at[(b - b0) * (kMeetBlock / 16) + (from - 1) * 256 + q * 64] =
              make_float4(v[q * 4], v[q * 4 + 1], v[q * 4 + 2], v[q * 4 + 3]);
        }
      }
      meet();
#pragma unroll
      for (int b = b0; b < b0 + kAtOnce && b < kBlocks; ++b) {
        if (b % KW != wk) continue;
        floatx16 &v = acc[b / WN][b % WN];
#pragma unroll
        for (int g = 0; g < KW - 1; ++g) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float4 f = at[(b - b0) * (kMeetBlock / 16) + g * 256 + q * 64];
            v[q * 4] += f.x;
            v[q * 4 + 1] += f.y;
            v[q * 4 + 2] += f.z;
            v[q * 4 + 3] += f.w;
          }
        }
      }
      meet();
    }
  };
  {
    Pieces p0, p1;
    clear();
    meet();
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) read(p0, kk);
    advance();
    // (what the last stage reads ahead is not used)
    int stage = 0;
    for (; stage + 2 <= total; stage += 2) {
      multiply(p0, p1);
      multiply(p1, p0);
    }
    if (stage < total) multiply(p0, p1);
  }
  add_up();
  {
    float sum = 0.0f;                          // zero where all are finite
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) {
      if (b % KW != wk) continue;
#pragma unroll
      for (int j = 0; j < 16; ++j) sum = fmaf(acc[b / WN][b % WN][j], 0.0f, sum);
    }
    if (__ballot(sum != 0.0f) != 0ull && lane == 0) *again = 1;
  }
  meet();
  if (*again != 0) {
    clear();
    meet();
    for (int stage = 0; stage < total; ++stage) {
      Pieces p;
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) read(p, kk);
      const int *at = reinterpret_cast<const int *>(lds + kEntriesAt) + stage / CH % kEntries * TM + wm * WM * 32 + r;
      int entry[WM];
#pragma unroll
      for (int a = 0; a < WM; ++a) entry[a] = at[a * 32];
      advance();
      meet();
#pragma unroll
      for (int a = 0; a < WM; ++a) {
        if (__ballot(entry[a] >= 0) != 0ull) {
#pragma unroll
          for (int kk = 0; kk < KS; ++kk) {
#pragma unroll
            for (int b = 0; b < WN; ++b) {
              const floatx16 sum = Mfma<T>::run(p.w[kk][b], p.x[kk][a], acc[a][b]);
#pragma unroll
              for (int j = 0; j < 16; ++j) acc[a][b][j] = entry[a] >= 0 ? sum[j] : acc[a][b][j];
            }
          }
        }
      }
    }
    add_up();
    meet();
  }
  unsigned char *turn = lds + wv * kTurnBytes;
  const bool whole = s.N % 8 == 0;             // output rows are whole 16-byte pieces
#pragma unroll
  for (int a = 0; a < WM; ++a) {
#pragma unroll
    for (int b = 0; b < WN; ++b) {
      const int ch0 = first_channel + (wn * WN + b) * 32;
      if (ch0 >= s.N || (a * WN + b) % KW != wk) continue;
      if (whole) {
        store_turned_rows<T>(acc[a][b], turn, lane, r, h, out_row[a], ch0, s.N, ep, out);
        continue;
      }
      const int row = row_of((wm * WM + a) * 32 + r);
      if (row < 0) continue;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int ch = ch0 + q * 8 + h * 4;
        if (ch >= s.N) continue;               // N % 4 == 0: a group of four is all in or all out
        float v[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = acc[a][b][q * 4 + x];
        finish_four<T>(v, ep, row, ch, s.N, out);
      }
    }
  }
}

}  // namespace mnt

namespace mnt {

template <typename T>
void streamed_forward(const T *sources, const T *packed, const int *kernel_map, const int *tiles, int64_t S, int64_t Tn,
                      int64_t O, int64_t K, int64_t N, const Epilogue &ep, T *out, hipStream_t stream) {
  const TileLayout l(Tn, O);
  const bool tiled = tiles != nullptr;
  const TileView view = {tiles, tiles + l.counts_at, tiles + l.offsets_at, tiles + l.sources_at};
  const int kc = kChunkBytes / static_cast<int>(sizeof(T));
  StreamedShape s;
  s.num_targets = Tn;
  s.slots = static_cast<int>(O);
  s.row_bytes = static_cast<int>(K * sizeof(T));
  s.N = static_cast<int>(N);
  s.packed_row_bytes = static_cast<int>(div_ceil(K, kc) * kc * sizeof(T));
  s.packed_rows = static_cast<int>(div_ceil(N, 32) * 32);
  const unsigned source_bytes = static_cast<unsigned>(S * s.row_bytes);
  const int64_t cus = compute_units();
  // Targets and channels of a workgroup.  What a compute unit loads for a product
  // falls as both grow, but a layer of few workgroups takes as long as the
  // longest of them, so the smallest shape that fits the chip in one go, then
  // the larger ones (us, 128 -> 128 channels, 2 000 targets: 32 x 64 10.0, 64 x
  // 64 10.4; 6 850: 64 x 64 11.8, 64 x 128 14.6; 18 600 in tiles: 64 x 128 17.3,
  // 128 x 128 22.8; 60 000 in tiles: 33.0, 25.6).  The line to the largest lies
  // higher for rows of more than two stages, whose chains are longer (128 -> 256
  // over 18 600 in tiles 33.2, 27.0; 256 -> 256 over 20 000 of a room 40.3, 42.4,
  // over 25 600 of a LiDAR scan even, over 30 000 54.4, 45.0).
  auto workgroups = [&](int64_t tm, int64_t tn) { return div_ceil(Tn, tm) * div_ceil(N, tn); };
#define MNT_STREAMED(MW, NW, KW, WM, WN, CH, RING)                                                                \
  {                                                                                                               \
    constexpr int TM = 32 * MW * WM, TN = 32 * NW * WN, threads = 64 * (kStreamedLoaders + MW * NW * KW);         \
    const dim3 grid(static_cast<unsigned>(tiled ? l.tiles * (kTileTargets / TM) : div_ceil(Tn, int64_t{TM})),     \
                    static_cast<unsigned>(div_ceil(N, int64_t{TN})));                                             \
    if (tiled) {                                                                                                  \
      streamed_forward_kernel<T, MW, NW, KW, WM, WN, CH, RING, true><<<grid, threads, 0, stream>>>(               \
          sources, source_bytes, packed, kernel_map, view, s, reinterpret_cast<unsigned char *>(out), ep);        \
    } else {                                                                                                      \
      streamed_forward_kernel<T, MW, NW, KW, WM, WN, CH, RING, false><<<grid, threads, 0, stream>>>(              \
          sources, source_bytes, packed, kernel_map, view, s, reinterpret_cast<unsigned char *>(out), ep);        \
    }                                                                                                             \
  }
#define MNT_STREAMED_WIDE(MW, NW, KW, WM, WN)                     \
  switch (div_ceil(s.row_bytes, kStreamedStage)) {                \
    case 2: MNT_STREAMED(MW, NW, KW, WM, WN, 2, 4) break;         \
    case 3: MNT_STREAMED(MW, NW, KW, WM, WN, 3, 3) break;         \
    default: MNT_STREAMED(MW, NW, KW, WM, WN, 4, 4) break;        \
  }
#define MNT_STREAMED_K(MW, NW, KW, WM, WN, R1)                    \
  if (s.row_bytes <= kStreamedStage) {                            \
    MNT_STREAMED(MW, NW, KW, WM, WN, 1, R1)                       \
  } else {                                                        \
    MNT_STREAMED_WIDE(MW, NW, KW, WM, WN)                         \
  }
  if (workgroups(32, 64) <= cus) {
    MNT_STREAMED_K(1, 1, 2, 1, 2, 4)
  } else if (workgroups(64, 64) <= cus) {
    MNT_STREAMED_K(1, 2, 2, 2, 1, 4)
  } else if (N <= 64) {                        // (rows of one stage come with more than 128 channels)
    MNT_STREAMED_WIDE(2, 1, 2, 2, 2)
  } else if (20 * workgroups(128, 128) < (s.row_bytes > 256 ? 30 : 21) * cus) {
    MNT_STREAMED_K(1, 2, 2, 2, 2, 3)
  } else {
    MNT_STREAMED_K(2, 2, 1, 2, 2, 3)
  }
#undef MNT_STREAMED_K
#undef MNT_STREAMED_WIDE
#undef MNT_STREAMED
  check_launch("streamed_forward_kernel");
}

}  // namespace mnt
