// Pieces the output-stationary forward kernels share: the output pass and the
// host-side entry points of the kernels.
#pragma once

#include "conv_device.h"
#include "device_utils.h"

namespace mnt {

// One output row's worth of epilogue and store: four consecutive channels of
// target t held by this lane.
template <typename T>
__device__ __forceinline__ void finish_four(float (&v)[4], const Epilogue &ep, long long t, int ch, int N,
                                            unsigned char *__restrict__ out) {
  typedef typename VecOf<4 * sizeof(T)>::type V;
  if (ep.scale != nullptr) {
#pragma unroll
    for (int x = 0; x < 4; ++x) v[x] *= ep.scale[ch + x];
  }
  if (ep.shift != nullptr) {
#pragma unroll
    for (int x = 0; x < 4; ++x) v[x] += ep.shift[ch + x];
  }
  if (ep.residual != nullptr) {
    const V raw = *reinterpret_cast<const V *>(static_cast<const unsigned char *>(ep.residual) +
                                               (t * N + ch) * static_cast<long long>(sizeof(T)));
    const T *e = reinterpret_cast<const T *>(&raw);
#pragma unroll
    for (int x = 0; x < 4; ++x) v[x] += to_float(e[x]);
  }
  if (ep.activation == MNT_ACT_RELU) {
#pragma unroll
    for (int x = 0; x < 4; ++x) v[x] = fmaxf(v[x], 0.0f);
  } else if (ep.activation == MNT_ACT_LEAKY_RELU) {
#pragma unroll
    for (int x = 0; x < 4; ++x) v[x] = v[x] > 0.0f ? v[x] : v[x] * ep.slope;
  } else if (ep.activation == MNT_ACT_RELU6) {
#pragma unroll
    for (int x = 0; x < 4; ++x) v[x] = fminf(fmaxf(v[x], 0.0f), 6.0f);
  }
  V raw;
  T *e = reinterpret_cast<T *>(&raw);
#pragma unroll
  for (int x = 0; x < 4; ++x) e[x] = static_cast<T>(v[x]);
  *reinterpret_cast<V *>(out + (t * N + ch) * static_cast<long long>(sizeof(T))) = raw;
}

// The same for one 16-byte piece of an output row (E = 16 / sizeof(T)
// consecutive channels from `ch` on), its sums given in fp32.
template <typename T, int E>
__device__ __forceinline__ void finish_piece(float (&v)[E], const Epilogue &ep, long long t, int ch, int N,
                                             unsigned char *__restrict__ out) {
  if (ep.scale != nullptr) {
#pragma unroll
    for (int x = 0; x < E; ++x) v[x] *= ep.scale[ch + x];
  }
  if (ep.shift != nullptr) {
#pragma unroll
    for (int x = 0; x < E; ++x) v[x] += ep.shift[ch + x];
  }
  if (ep.residual != nullptr) {
    const uint4 raw = *reinterpret_cast<const uint4 *>(static_cast<const unsigned char *>(ep.residual) +
                                                       (t * N + ch) * static_cast<long long>(sizeof(T)));
    const T *e = reinterpret_cast<const T *>(&raw);
#pragma unroll
    for (int x = 0; x < E; ++x) v[x] += to_float(e[x]);
  }
  if (ep.activation == MNT_ACT_RELU) {
#pragma unroll
    for (int x = 0; x < E; ++x) v[x] = fmaxf(v[x], 0.0f);
  } else if (ep.activation == MNT_ACT_LEAKY_RELU) {
#pragma unroll
    for (int x = 0; x < E; ++x) v[x] = v[x] > 0.0f ? v[x] : v[x] * ep.slope;
  } else if (ep.activation == MNT_ACT_RELU6) {
#pragma unroll
    for (int x = 0; x < E; ++x) v[x] = fminf(fmaxf(v[x], 0.0f), 6.0f);
  }
  uint4 raw;
  T *e = reinterpret_cast<T *>(&raw);
#pragma unroll
  for (int x = 0; x < E; ++x) e[x] = static_cast<T>(v[x]);
  *reinterpret_cast<uint4 *>(out + (t * N + ch) * static_cast<long long>(sizeof(T))) = raw;
}

// Where wavefronts multiply whole blocks, a target without a source takes part with
// zeros, which an infinite or undefined weight turns into sums that are undefined.
// A wavefront that has sums which are not finite (`seen`: the largest that a lane
// has) therefore works those out again from the operands in memory, one by one,
// over the offsets that the target has a source under, and stores them in place of
// what it has stored.  That takes trips to memory for every offset and sum; all
// others pay half an instruction a sum, us a layer without and so: 32 -> 256 channels
// over 300 000 voxels of a LiDAR scan in tiles 92.9 / 94.4, 16 -> 256 90.2 / 92.9, of a
// room 8 -> 512 143 / 149, over 3 000 8.4 / 8.4.
// entry(i), offset_of(i): the source row (-1: none) of this lane's target under the
// i-th of `slots` offsets, and the number of that offset.  target_of(): -1 for none.
// Blocks b of which b % GROUPS is not `group` are another wavefront's.
template <int COUNT, typename V>
__device__ __forceinline__ float largest_of(const V &v, float seen) {
#pragma unroll
  for (int j = 0; j < COUNT; j += 2) {         // (maximum: undefined where one of them is)
    seen = __builtin_elementwise_maximum(__builtin_elementwise_maximum(fabsf(v[j]), fabsf(v[j + 1])), seen);
  }
  return seen;
}

template <typename T, int NB, int GROUPS, typename Entry, typename OffsetOf, typename TargetOf>
__device__ __forceinline__ void keep_to_sources(const floatx16 (&acc)[NB], float seen, const T *__restrict__ sources,
                                                int K, const T *__restrict__ wt, int packed_row, int packed_rows,
                                                int first_channel, int N, int h, int group, int slots,
                                                const Entry &entry, const OffsetOf &offset_of,
                                                const TargetOf &target_of, const Epilogue &ep,
                                                unsigned char *__restrict__ out) {
  if (__ballot(!(seen < INFINITY)) == 0ull) return;
  const long long target = target_of();
  __threadfence();                             // (what is stored here comes after what other lanes have stored)
  constexpr int E = 16 / static_cast<int>(sizeof(T));
  unsigned long long wrong = 0;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if (GROUPS > 1 && b % GROUPS != group) continue;
#pragma unroll
    for (int j = 0; j < 16; ++j) wrong |= fabsf(acc[b][j]) < INFINITY ? 0ull : 1ull << (b * 16 + j);
  }
  while (wrong != 0) {
    const int at = __builtin_ctzll(wrong);
    wrong &= wrong - 1;
    const int channel = first_channel + at / 16 * 32 + at % 16 / 4 * 8 + h * 4 + at % 4;
    if (target < 0 || channel >= N) continue;
    float sum = 0.0f;
    for (int i = 0; i < slots; ++i) {
      const int index = entry(i);
      if (index < 0) continue;
      const T *const row = sources + static_cast<long long>(index) * K;
      const T *const weights = wt + (static_cast<long long>(offset_of(i)) * packed_rows + channel) * packed_row;
#pragma unroll 1
      for (int k = 0; k < K; k += E) {         // (K % E == 0)
        const uint4 raw = *reinterpret_cast<const uint4 *>(row + k);
        const uint4 raw_w = *reinterpret_cast<const uint4 *>(weights + k);
        const T *const x = reinterpret_cast<const T *>(&raw), *const w = reinterpret_cast<const T *>(&raw_w);
#pragma unroll
        for (int e = 0; e < E; ++e) sum = fmaf(to_float(x[e]), to_float(w[e]), sum);
      }
    }
    if (ep.scale != nullptr) sum *= ep.scale[channel];
    if (ep.shift != nullptr) sum += ep.shift[channel];
    if (ep.residual != nullptr) sum += to_float(static_cast<const T *>(ep.residual)[target * N + channel]);
    if (ep.activation == MNT_ACT_RELU) sum = fmaxf(sum, 0.0f);
    if (ep.activation == MNT_ACT_LEAKY_RELU) sum = sum > 0.0f ? sum : sum * ep.slope;
    if (ep.activation == MNT_ACT_RELU6) sum = fminf(fmaxf(sum, 0.0f), 6.0f);
    reinterpret_cast<T *>(out)[target * N + channel] = static_cast<T>(sum);
  }
}

// Epilogue and store of one 32 x 32 block of fp32 sums as the matrix
// instructions leave it (lane (r, h) holds channels q * 8 + h * 4 .. + 3 of
// target block_t0 + r in acc[q * 4 .. + 3]), for output rows that are whole
// 16-byte pieces: the wavefront turns the block around in its own `turn` area
// of LDS (kTurnBytes), so that one store instruction covers rows in contiguous
// pieces of 64 bytes (128 in fp32), and the residual is read the same way.
constexpr int kTurnRow = 32 * 4 + 16;
constexpr int kTurnBytes = 32 * kTurnRow;

template <typename T>
__device__ __forceinline__ void store_turned_block(const floatx16 &acc, unsigned char *turn, int lane, int r,
                                                   int h, long long block_t0, long long num_targets, int ch0,
                                                   int N, const Epilogue &ep, unsigned char *__restrict__ out) {
  constexpr int EPV = 16 / static_cast<int>(sizeof(T));
  constexpr int kOutPieces = 32 / EPV;                          // 16-byte pieces of a block's output row
  constexpr int kPieces = 32 * kOutPieces / 64;                 // per lane
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    *reinterpret_cast<float4 *>(turn + r * kTurnRow + (q * 8 + h * 4) * 4) =
        make_float4(acc[q * 4], acc[q * 4 + 1], acc[q * 4 + 2], acc[q * 4 + 3]);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int i = 0; i < kPieces; ++i) {
    const int piece = lane + i * 64;
    const int pr = piece / kOutPieces, part = piece % kOutPieces;
    const int ch = ch0 + part * EPV;
    float v[EPV];
#pragma unroll
    for (int x = 0; x < EPV; x += 4) {
      const float4 f = *reinterpret_cast<const float4 *>(turn + pr * kTurnRow + (part * EPV + x) * 4);
      v[x] = f.x;
      v[x + 1] = f.y;
      v[x + 2] = f.z;
      v[x + 3] = f.w;
    }
    if (block_t0 + pr < num_targets && ch < N) {                // N % EPV == 0: a piece is all in or all out
      finish_piece<T, EPV>(v, ep, block_t0 + pr, ch, N, out);
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename T>
__device__ __forceinline__ void store_turned_rows(const floatx16 &acc, unsigned char *turn, int lane, int r,
                                                   int h, const int *rows, int ch0, int N, const Epilogue &ep,
                                                  unsigned char *__restrict__ out) {
  constexpr int EPV = 16 / static_cast<int>(sizeof(T));
  constexpr int kOutPieces = 32 / EPV;                          // 16-byte pieces of a block's output row
  constexpr int kPieces = 32 * kOutPieces / 64;                 // per lane
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    *reinterpret_cast<float4 *>(turn + r * kTurnRow + (q * 8 + h * 4) * 4) =
        make_float4(acc[q * 4], acc[q * 4 + 1], acc[q * 4 + 2], acc[q * 4 + 3]);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int i = 0; i < kPieces; ++i) {
    const int piece = lane + i * 64;
    const int pr = piece / kOutPieces, part = piece % kOutPieces;
    const int ch = ch0 + part * EPV;
    float v[EPV];
#pragma unroll
    for (int x = 0; x < EPV; x += 4) {
      const float4 f = *reinterpret_cast<const float4 *>(turn + pr * kTurnRow + (part * EPV + x) * 4);
      v[x] = f.x;
      v[x + 1] = f.y;
      v[x + 2] = f.z;
      v[x + 3] = f.w;
    }
    if (rows[i] >= 0 && ch < N) finish_piece<T, EPV>(v, ep, rows[i], ch, N, out);   // N % EPV == 0
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace mnt
