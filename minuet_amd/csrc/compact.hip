// Output-stationary forward of an fp32 sparse convolution that multiplies hits
// only: Gather -> GEMM -> Scatter
// (csrc/minuet/cuda/functions/sparse_convolution.cu:504-661) in one kernel from
// the dense kernel map, without buffer rows and without rank tables.
#include <algorithm>

#include "conv_device.h"
#include "device_utils.h"
#include "implicit.h"

namespace mnt {

constexpr unsigned kCompactNowhere = 0xFFFFF000u;   // past the end of every buffer: reads zeros

typedef unsigned uint4v __attribute__((ext_vector_type(4)));
typedef unsigned uint2v __attribute__((ext_vector_type(2)));

template <int C>
struct Floats {
  float v[C];
} __attribute__((aligned(4 * C)));

struct CompactShape {
  long long num_targets;
  int num_offsets, K, N;
  int chunks;                  // units of KI * 16 input channels
  int columns;                 // workgroups side by side over the output channels
  int steps;                   // of 16 input channels, in weights given in lane order
};

// A workgroup takes TARGETS targets and 16 * C output channels; its SPLIT wavefronts
// take every SPLIT-th offset each.  fp32 matrix instructions are 16 times dearer
// than 16-bit ones, so nothing but hits is multiplied: a wavefront lists the
// hits of its offsets, 16 rows of one offset at a time are multiplied by
// 16 x 16 x 4 instructions (K in pieces of 16 channels, KI of them per unit),
// and the sums of their targets, which stand in LDS, go in and come out as the
// instruction's accumulators (AFTER: the products are added to them).  Every
// wavefront has sums of its own; they are added up in the order of the wavefronts
// at the end, so that a result is the same whenever it is computed.
//
// LANES: the weights come in the order of the instruction's lanes (pack_lanes),
// one load of 1 KB where [O][K][N] takes four of 256 or 512 bytes.  For callers
// that keep such a copy: a layer's weights are read where they are, because a
// copy would miss what is written through .data or before a graph's replay
// (which costs 8 % on average over 226 layers).
//
// What bounds it: on small clouds one wavefront's chain of map entry, source
// rows, products (the unit after is asked for before one is multiplied), hence
// the split; beyond, fp32 products of 16 rows that are about half hits, and the
// weights, which every 16 rows read again: from some
// targets x input x output channels on (78 million for 3 x 3 x 3) the
// three-kernel form is the faster one again, unless there are few input channels
// (hits_rows_limit and hits_rows_from in nn/functional/convolution.py have the
// lines and both sides of them).  fp32, 3 x 3 x 3, us a layer in
// three kernels and here: 32 -> 32 channels over 3 000 voxels 11.4 / 4.9,
// 20 000 17.9 / 11.2, 200 000 76 / 54; 64 -> 64 over 3 000 12.1 / 8.4, 12 000
// 18.8 / 14.9; 256 -> 256 over 135 28 / 15.6 (in lanes 12.5).  (128 targets per workgroup
// fill the 16 rows better, but their sums leave fewer wavefronts to a compute
// unit: 17 to 40 % slower.  Rows that four lanes load together and turn round:
// 20 000 targets 13.0 -> 14.4; the hits of all wavefronts dealt out evenly: 12.1, but
// 256 -> 256 over 130 targets 13.6 -> 14.9, and sums that go by the targets of a
// workgroup.)
template <int C, int KI, int SPLIT, int TARGETS, bool WHOLE, bool LANES, bool AFTER>
__global__ __launch_bounds__(64 * SPLIT) void compact_forward_kernel(
    const float *__restrict__ sources, unsigned source_bytes, const float *__restrict__ weights,
    unsigned weight_bytes, const int *__restrict__ kernel_map, CompactShape s, unsigned char *__restrict__ out,
    Epilogue ep) {
  constexpr int kCompactBatch = 32 / SPLIT;                // offsets whose hits a wavefront lists together
  constexpr int kTargets = TARGETS;
  constexpr int kAtOnce = 64 / TARGETS;                    // offsets that a wavefront's lanes look at together
  constexpr int kMost = kCompactBatch * kTargets;          // list entries
  constexpr int kAccRow = 16 * C + 4;
  struct Lists {
    int source[kMost];
    int offset[kMost / 16];
    unsigned char target[kMost];
  };
  __shared__ __align__(16) float s_acc[SPLIT][(kTargets + 1) * kAccRow];
  __shared__ __align__(16) Lists s_lists[SPLIT];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15;
  const int q = lane >> 4;
  const long long first = static_cast<long long>(blockIdx.x / s.columns) * kTargets;
  const int channel = static_cast<int>(blockIdx.x % s.columns + blockIdx.y) * 16 * C;
  const int chunks = s.chunks;
  float *const acc = s_acc[wv];
  Lists &lists = s_lists[wv];

  const __amdgpu_buffer_rsrc_t source_buffer = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(sources), 0, source_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t weight_buffer = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(weights), 0, weight_bytes, 0x00020000);
  const unsigned row_bytes = static_cast<unsigned>(s.K) * 4u;
  const unsigned line_bytes = static_cast<unsigned>(s.N) * 4u;
  // lane (r, q) multiplies the C channels r * C .. of the workgroup's 16 * C;
  // with weights in lane order r, 16 + r, ..
  const bool in_width = LANES || channel + r * C < s.N;
  const unsigned w_at = LANES ? lane * 16u
                        : in_width ? static_cast<unsigned>(q) * 4u * line_bytes + static_cast<unsigned>(channel + r * C) * 4u
                                   : kCompactNowhere;
  const unsigned blocks = (static_cast<unsigned>(s.N) + 15u) / 16u;
  struct Unit {
    uint4 a[KI];
    float w[KI][4][C];
    unsigned targets;
  };
  auto fetch = [&](int g, int c, Unit &u) {
    const int source = lists.source[g * 16 + r];
    const int o = __builtin_amdgcn_readfirstlane(lists.offset[g]);
    u.targets = *reinterpret_cast<const unsigned *>(&lists.target[g * 16 + q * 4]);
    const unsigned chunk_at = static_cast<unsigned>(c) * (KI * 64u);
    const unsigned row_at = source >= 0 ? static_cast<unsigned>(source) * row_bytes + q * 16u : kCompactNowhere;
    const unsigned w_base = static_cast<unsigned>(o) * row_bytes * static_cast<unsigned>(s.N) + chunk_at / 4u * line_bytes;
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      const bool inside = WHOLE || chunk_at + i * 64u + q * 16u < row_bytes;
      const uint4v v = __builtin_amdgcn_raw_buffer_load_b128(source_buffer, inside ? row_at : kCompactNowhere,
                                                             chunk_at + i * 64u, 0);
      u.a[i] = make_uint4(v.x, v.y, v.z, v.w);
      if constexpr (LANES) {
        const int step = c * KI + i;
#pragma unroll
        for (int b = 0; b < C; ++b) {
          const unsigned at = WHOLE || step < s.steps ? w_at : kCompactNowhere;
          const unsigned from = ((static_cast<unsigned>(o) * blocks + channel / 16 + b) * s.steps + step) * 1024u;
          const uint4v w = __builtin_amdgcn_raw_buffer_load_b128(weight_buffer, at, from, 0);
          u.w[i][0][b] = __uint_as_float(w.x);
          u.w[i][1][b] = __uint_as_float(w.y);
          u.w[i][2][b] = __uint_as_float(w.z);
          u.w[i][3][b] = __uint_as_float(w.w);
        }
        continue;
      }
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const unsigned at = inside ? w_at : kCompactNowhere;
        const unsigned from = w_base + (i * 16u + x) * line_bytes;
        if constexpr (C == 1) {
          u.w[i][x][0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(weight_buffer, at, from, 0));
        } else if constexpr (C == 2) {
          const uint2v v = __builtin_amdgcn_raw_buffer_load_b64(weight_buffer, at, from, 0);
          u.w[i][x][0] = __uint_as_float(v.x);
          u.w[i][x][1] = __uint_as_float(v.y);
        } else {
          const uint4v v = __builtin_amdgcn_raw_buffer_load_b128(weight_buffer, at, from, 0);
          u.w[i][x][0] = __uint_as_float(v.x);
          u.w[i][x][1] = __uint_as_float(v.y);
          u.w[i][x][2] = __uint_as_float(v.z);
          u.w[i][x][3] = __uint_as_float(v.w);
        }
      }
    }
  };
  auto multiply = [&](const Unit &u) {
    float *row[4];
    Floats<C> before[4];
    floatx4 sum[C];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      row[j] = acc + ((u.targets >> (8 * j)) & 255u) * kAccRow + r * C;
      before[j] = *reinterpret_cast<const Floats<C> *>(row[j]);
#pragma unroll
      for (int b = 0; b < C; ++b) sum[b][j] = AFTER ? 0.0f : before[j].v[b];
    }
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      const float *a = reinterpret_cast<const float *>(&u.a[i]);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
#pragma unroll
        for (int b = 0; b < C; ++b) sum[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[x], u.w[i][x][b], sum[b], 0, 0, 0);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      Floats<C> after;
#pragma unroll
      for (int b = 0; b < C; ++b) after.v[b] = AFTER ? before[j].v[b] + sum[b][j] : sum[b][j];
      *reinterpret_cast<Floats<C> *>(row[j]) = after;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };

  int index[kCompactBatch / kAtOnce];          // (outside the loop over them, which asks for all of them at once)
  auto load_map = [&](int first_offset) {
#pragma unroll
    for (int j = 0; j < kCompactBatch / kAtOnce; ++j) {
      const int o = min(first_offset + (j * kAtOnce + lane / kTargets) * SPLIT, s.num_offsets - 1);
      const long long target = min(first + lane % kTargets, s.num_targets - 1);
      // without a map the offsets are pieces of the target's own row
      index[j] = kernel_map != nullptr ? kernel_map[o * s.num_targets + target] : static_cast<int>(target) * s.num_offsets + o;
    }
  };
  load_map(wv);
  for (int i = lane; i < (kTargets + 1) * kAccRow / 4; i += 64) {
    reinterpret_cast<float4 *>(acc)[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
  for (int first_offset = wv; first_offset < s.num_offsets; first_offset += SPLIT * kCompactBatch) {
    int count = 0;
#pragma unroll
    for (int j = 0; j < kCompactBatch / kAtOnce; ++j) {
      const bool hit = index[j] >= 0 && first + lane % kTargets < s.num_targets &&
                       first_offset + (j * kAtOnce + lane / kTargets) * SPLIT < s.num_offsets;
      const unsigned long long votes = __ballot(hit);
#pragma unroll
      for (int part = 0; part < kAtOnce; ++part) {
        constexpr unsigned long long kOwn = kTargets == 64 ? ~0ull : (1ull << (kTargets & 63)) - 1ull;
        const unsigned long long own = votes & (kOwn << (part * kTargets & 63));
        const int from = count;
        if (hit && lane / kTargets == part) {
          const int p = count + __popcll(own & lanes_below());
          lists.source[p] = index[j];
          lists.target[p] = static_cast<unsigned char>(lane % kTargets);
        }
        count += __popcll(own);
        const int end = (count + 15) & ~15;    // the rest of 16 rows: no source, a target nobody asks for
        if (lane < end - count) {
          lists.source[count + lane] = -1;
          lists.target[count + lane] = static_cast<unsigned char>(kTargets);
        }
        if (lane < (end - from) / 16) lists.offset[from / 16 + lane] = first_offset + (j * kAtOnce + part) * SPLIT;
        count = end;
      }
    }
    count = __builtin_amdgcn_readfirstlane(count);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (first_offset + SPLIT * kCompactBatch < s.num_offsets) load_map(first_offset + SPLIT * kCompactBatch);
    int left = count / 16 * chunks;
    if (left == 0) continue;
    int g = 0, c = 0;
    auto advance = [&]() {
      if (++c == chunks) {
        c = 0;
        ++g;
      }
    };
    // One unit ahead and none past the last: the loads of one that is not
    // multiplied keep the address unit as long as another's (two of the nine a
    // wavefront has over 20 000 targets; 256 -> 256 channels over 130 targets
    // 15.4 -> 13.4 us without them, 128 -> 128 over 3 000 20.8 -> 19.8).  Three
    // units in flight are no faster (14.6, 24.3).
    Unit u0, u1;
    fetch(0, 0, u0);
    for (; left > 2; left -= 2) {
      advance();
      fetch(g, c, u1);
      multiply(u0);
      advance();
      fetch(g, c, u0);
      multiply(u1);
    }
    if (left == 2) {
      advance();
      fetch(g, c, u1);
      multiply(u0);
      multiply(u1);
    } else {
      multiply(u0);
    }
  }

  __syncthreads();
  for (int p = tid; p < kTargets * 4 * C; p += 64 * SPLIT) {
    const int t = p / (4 * C), part = p % (4 * C);
    if (first + t >= s.num_targets || channel + part * 4 >= s.N) continue;     // N % 4 == 0
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < SPLIT; ++w) {
      if constexpr (LANES && C > 1) {
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const int ch = part * 4 + x;
          v[x] += s_acc[w][t * kAccRow + ch % 16 * C + ch / 16];
        }
      } else {
        const float4 f = *reinterpret_cast<const float4 *>(&s_acc[w][t * kAccRow + part * 4]);
        v[0] += f.x;
        v[1] += f.y;
        v[2] += f.z;
        v[3] += f.w;
      }
    }
    finish_piece<float, 4>(v, ep, first + t, channel + part * 4, s.N, out);
  }
}

// lanes[o][block][step][lane][x] = w[o][16 step + 4 (lane / 16) + x][16 block + lane % 16]
__global__ __launch_bounds__(256) void pack_lanes_kernel(const float *__restrict__ w, int K, int N, int blocks,
                                                         int steps, long long pieces, uint4 *__restrict__ lanes) {
  const long long stride = static_cast<long long>(gridDim.x) * 256;
  for (long long i = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x; i < pieces; i += stride) {
    const int lane = static_cast<int>(i & 63);
    const long long group = i >> 6;
    const int step = static_cast<int>(group % steps), block = static_cast<int>(group / steps % blocks);
    const long long o = group / steps / blocks;
    const int k0 = 16 * step + 4 * (lane >> 4), n = 16 * block + (lane & 15);
    unsigned v[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) v[x] = k0 + x < K && n < N ? __float_as_uint(w[(o * K + k0 + x) * N + n]) : 0u;
    lanes[i] = make_uint4(v[0], v[1], v[2], v[3]);
  }
}

int64_t lane_weight_floats(int64_t O, int64_t K, int64_t N) { return O * div_ceil(N, int64_t{16}) * div_ceil(K, int64_t{16}) * 256; }

void pack_lanes(const float *weights, int64_t O, int64_t K, int64_t N, float *lanes, hipStream_t stream) {
  const long long pieces = lane_weight_floats(O, K, N) / 4;
  if (pieces == 0) return;
  pack_lanes_kernel<<<grid_for(pieces, 256, 4096), 256, 0, stream>>>(
      weights, static_cast<int>(K), static_cast<int>(N), static_cast<int>(div_ceil(N, int64_t{16})),
      static_cast<int>(div_ceil(K, int64_t{16})), pieces, reinterpret_cast<uint4 *>(lanes));
  check_launch("pack_lanes_kernel");
}

// `weights`: [O][K][N] or, with `lanes`, as pack_lanes leaves them.
void compact_forward(const float *sources, const float *weights, bool lanes, const int *kernel_map, int64_t S,
                     int64_t Tn, int64_t O, int64_t K, int64_t N, const Epilogue &ep, float *out, hipStream_t stream) {
  CompactShape s;
  s.num_targets = Tn;
  s.num_offsets = static_cast<int>(O);
  s.K = static_cast<int>(K);
  s.N = static_cast<int>(N);
  s.chunks = static_cast<int>(div_ceil(K, 64));
  const int ki = static_cast<int>(div_ceil(K, 16 * s.chunks));
  const bool whole = K == 16 * ki * s.chunks;
  // Targets, channel blocks and wavefronts of a workgroup by how many workgroups
  // of 64 targets and 16 channels there are to a compute unit (`full`): small
  // clouds need small workgroups to reach the whole chip, beyond that two blocks
  // share the source rows (from 1.95 to 3 workgroups over 32 targets each: over 64
  // those two blocks are one to one and a half workgroups a compute unit).  With
  // one step of 16 input channels a workgroup is its
  // map and its sums, and 32 targets are enough at any size; not for many targets
  // and weights as [O][K][N], of which four blocks read whole lines.  Those have
  // one block up to 4.75 workgroups, since a second doubles the loads of their
  // weights (in lanes it does not).  `split` is the same for both forms of the
  // weights, whose sums are then the same bit for bit; a unit of less than two
  // steps (K < 32) is short, and eight wavefronts pay a little longer.
  //
  // Weights in lanes, over 1 057 layers of three kinds of scene (3x3x3 and strided
  // 2x2x2, 130 to 580 000 targets, 4 to 256 channels): the form before there were
  // two, and its lines, took 1.14 times as long (the best of 14 shapes for each
  // layer 0.96).  [O][K][N], which is what layers have, against that form: 1.00
  // over 285 of them, 0.99 over 130 of 3 to 4.75 workgroups, 1.01 over 204 of 20 to
  // 28 channels.  us, that form and here, lanes: 256 -> 256 channels over 130 targets
  // 19.7 / 12.8, 128 -> 128 over 2 980 46 / 33, 8 -> 128 over 40 000 27.6 / 26.5;
  // [O][K][N], objects: 128 -> 128 over 700 14.0 / 10.6, 32 -> 32 over 20 000 14.0 /
  // 13.4, 64 -> 64 over 12 000 21.5 / 20.1, 28 -> 128 over 4 000 under 5x5x5 29.4 / 29.1;
  // slower: 128 -> 128 over 3 000 25.8 / 27.7, 80 -> 64 over 9 000 of 2x2x2 10.6 / 12.1,
  // 64 -> 16 onto 13 700 5.8 / 6.7.  What two blocks cost is layers with few hits,
  // whose blocks of rows are nearly empty, which the host cannot know: in lanes 96 ->
  // 256 over 2 000 of a LiDAR scan 13.7 / 16.5 and, with one block, 13.7; where a
  // target has 13 hits 35 / 26 and 32.
  const int64_t cus = compute_units(), cols = div_ceil(N, int64_t{16});
  const double full = static_cast<double>(div_ceil(Tn, int64_t{64}) * cols) / static_cast<double>(cus);
  int c = 1, targets = 64, split = full < (K < 32 ? 2.26 : 1.95) ? 8 : 4;
  if (N % 32 != 0) {
    targets = full < 0.3 ? 16 : full < 0.9 ? 32 : 64;
    split = full < 2.25 ? 8 : 4;
  } else if (K <= 16 && full >= 0.93 && (lanes || full < 4.75)) {
    c = 2;
    targets = 32;
    split = full < 3.0 ? 8 : 4;
  } else if (!lanes && K > 16 && full < 4.75) {
    targets = full < 0.26 ? 16 : full < 0.6 ? 32 : 64;
  } else if (full < 0.6) {
    c = full >= 0.26 && full < 0.42 ? 2 : 1;
    targets = full < 0.42 ? 16 : 32;
  } else if (full < 1.37) {
    c = full < 0.93 ? 2 : 1;
    targets = full < 0.93 ? 32 : 64;
  } else {
    c = full >= 4.75 && N % 64 == 0 ? 4 : 2;
    targets = full >= 1.95 && full < 3.0 ? 32 : 64;
  }
  // Layers that three kernels would take otherwise (hits_rows_limit has the lines):
  // there a target's sum takes products that have been added up offset by offset,
  // and so it does here.  Where sums go in as accumulators (64 to 128 channels by
  // 3x3x3 over 100 000 voxels) they are off by 1.1 to 1.3 times as much, added
  // afterwards as much as there; it takes 2 to 8 % longer.  (Added while the next
  // 16 rows are multiplied: 232 registers instead of 160, 10 % longer.)
  const bool after = !lanes && K <= 48 && K * N > 1024 && O >= 27 && S * K * N > 2100000000 / O;
  if (after) {
    targets = 64;
    split = 4;
  }
  s.steps = static_cast<int>(div_ceil(K, int64_t{16}));
  // Columns side by side, so that the workgroups of a die share few of them and
  // its L2 holds their weights, up to the threads a grid may have along x.
  const int64_t rows = div_ceil(Tn, int64_t{targets}), columns = div_ceil(cols, int64_t{c});
  const bool beside = rows * columns * 64 * split < (int64_t{1} << 32);
  s.columns = beside ? static_cast<int>(columns) : 1;
  const dim3 grid(static_cast<unsigned>(beside ? rows * columns : rows), static_cast<unsigned>(beside ? 1 : columns));
  const unsigned weight_bytes = static_cast<unsigned>((lanes ? lane_weight_floats(O, K, N) : O * K * N) * 4);
#define MNT_COMPACT_W(C, KI, SPLIT, TARGETS, WHOLE, LANES, AFTER)                                              \
  compact_forward_kernel<C, KI, SPLIT, TARGETS, WHOLE, LANES, AFTER><<<grid, 64 * SPLIT, 0, stream>>>(                \
      sources, static_cast<unsigned>(S * K * 4), weights, weight_bytes, kernel_map, s,                         \
      reinterpret_cast<unsigned char *>(out), ep)
#define MNT_COMPACT(C, KI, SPLIT, TARGETS)               \
  if (lanes && whole) {                                  \
    MNT_COMPACT_W(C, KI, SPLIT, TARGETS, true, true, false);    \
  } else if (lanes) {                                    \
    MNT_COMPACT_W(C, KI, SPLIT, TARGETS, false, true, false);   \
  } else if (whole) {                                    \
    MNT_COMPACT_W(C, KI, SPLIT, TARGETS, true, false, false);   \
  } else {                                               \
    MNT_COMPACT_W(C, KI, SPLIT, TARGETS, false, false, false);  \
  }
#define MNT_COMPACT_K(C, SPLIT, TARGETS)               \
  switch (ki) {                                        \
    case 1: MNT_COMPACT(C, 1, SPLIT, TARGETS) break;   \
    case 2: MNT_COMPACT(C, 2, SPLIT, TARGETS) break;   \
    case 3: MNT_COMPACT(C, 3, SPLIT, TARGETS) break;   \
    default: MNT_COMPACT(C, 4, SPLIT, TARGETS) break;  \
  }
#define MNT_COMPACT_AFTER(C, KI)                           \
  if (whole) {                                             \
    MNT_COMPACT_W(C, KI, 4, 64, true, false, true);        \
  } else {                                                 \
    MNT_COMPACT_W(C, KI, 4, 64, false, false, true);       \
  }
#define MNT_COMPACT_AFTER_K(C)                       \
  switch (ki) {                                      \
    case 1: MNT_COMPACT_AFTER(C, 1) break;           \
    case 2: MNT_COMPACT_AFTER(C, 2) break;           \
    default: MNT_COMPACT_AFTER(C, 3) break;          \
  }
  if (after) {
    if (c == 4) {
      MNT_COMPACT_AFTER_K(4)
    } else if (c == 2) {
      MNT_COMPACT_AFTER_K(2)
    } else {
      MNT_COMPACT_AFTER_K(1)
    }
  } else if (c == 4) {
    MNT_COMPACT_K(4, 4, 64)
  } else if (c == 2) {
    if (targets == 16) {
      MNT_COMPACT_K(2, 8, 16)
    } else if (targets == 32) {
      if (split == 8) {
        MNT_COMPACT_K(2, 8, 32)
      } else {
        MNT_COMPACT_K(2, 4, 32)
      }
    } else if (split == 8) {
      MNT_COMPACT_K(2, 8, 64)
    } else {
      MNT_COMPACT_K(2, 4, 64)
    }
  } else if (targets == 16) {
    MNT_COMPACT_K(1, 8, 16)
  } else if (targets == 32) {
    MNT_COMPACT_K(1, 8, 32)
  } else if (split == 8) {
    MNT_COMPACT_K(1, 8, 64)
  } else {
    MNT_COMPACT_K(1, 4, 64)
  }
#undef MNT_COMPACT_AFTER_K
#undef MNT_COMPACT_AFTER
#undef MNT_COMPACT_K
#undef MNT_COMPACT
#undef MNT_COMPACT_W
  check_launch("compact_forward_kernel");
}

}  // namespace mnt

using namespace mnt;

extern "C" int mnt_pack_weights_in_lanes(const float *weights, int64_t O, int64_t K, int64_t N, float *packed_out,
                                         void *stream_) {
  return guarded([&] {
    MNT_CHECK(O >= 0 && O <= 65535 && K >= 1 && N >= 1 && K <= 65536 && N <= 65536,
              "bad shape O=%lld Cin=%lld Cout=%lld", (long long)O, (long long)K, (long long)N);
    if (O == 0) return;
    MNT_CHECK(weights != nullptr && packed_out != nullptr, "null operand");
    MNT_CHECK(reinterpret_cast<uintptr_t>(packed_out) % 16 == 0, "packed weights are not 16-byte aligned");
    pack_lanes(weights, O, K, N, packed_out, static_cast<hipStream_t>(stream_));
  });
}
