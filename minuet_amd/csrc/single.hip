// Output-stationary forward of a transposed layer whose kernel is its stride: a
// target has one source.  Gather -> GEMM -> Scatter
// (csrc/minuet/cuda/functions/sparse_convolution.cu:504-661) in one kernel.
#include <algorithm>

#include "streamed_kernel.h"

namespace mnt {

constexpr int kSingleMost = 1024;              // targets of a workgroup
constexpr int kSingleWaves = 8;
constexpr int kSingleOffsets = 8;              // one a wavefront
constexpr int kSingleColumns = 64;
constexpr int kSingleStage = 128;              // bytes of a row

struct SingleShape {
  long long num_targets;
  int targets;                 // of a workgroup, a multiple of 64
  int offsets, row_bytes, chunks, N;
  int packed_row_bytes, packed_rows;
};

// A workgroup takes up to 1024 targets and 64 output channels; a wavefront lists
// those that have their source under its offset, about an eighth, and multiplies
// 64 of them at a time: rows and weights go straight to LDS, 128 bytes of each at
// a time, and the products from there to the targets' rows.  Targets without a
// source are the first wavefront's, which multiplies nothing for them: zeros
// times an infinite or undefined weight are no zeros.  Where a target has two
// sources (the caller says there is none) the wavefronts take 32 targets each
// under all offsets instead.
//
// What bounds it: one workgroup a compute unit, whose wavefronts wait for their
// map, their first rows and every next 128 bytes of them; so as few rounds of
// workgroups as fill the chip (256 targets each over 150 000 25.3 us, 640 19.5).
// Under all offsets for every target, as streamed_forward_kernel runs other
// layers, seven of eight products are zeros: us a layer, there and here, 128 -> 64
// channels over 150 000 targets of a room 39.3 / 19.5, over 56 000 of a LiDAR
// level 16.4 / 11.7, 256 -> 128 over 18 600 21.8 / 12.4, over 15 000 of objects
// 12.4 / 9.6.  Rows of up to 128 bytes cost the other kernels no more (64 -> 64
// over 150 000 16.7 / 16.3, 32 -> 32 over 200 000 11.6 / 16.9).
template <typename T>
__global__ __launch_bounds__(64 * kSingleWaves) void single_forward_kernel(
    const T *__restrict__ sources, unsigned source_bytes, const T *__restrict__ wt,
    const int *__restrict__ kernel_map, SingleShape s, unsigned char *__restrict__ out, Epilogue ep) {
  constexpr int BK = kSingleStage, kRounds = kSingleMost / 64;
  struct Wave {
    unsigned char rows[64 * BK], weights[kSingleColumns * BK];
  };
  __shared__ __align__(16) Wave s_wave[kSingleWaves];
  __shared__ int s_source[kSingleMost];
  __shared__ unsigned short s_target[kSingleWaves][kSingleMost];
  __shared__ int s_hits[kSingleMost];
  __shared__ int s_many;
  static_assert(sizeof(s_wave) + sizeof(s_source) + sizeof(s_target) + sizeof(s_hits) + 16 <= 160 * 1024 &&
                kTurnBytes <= sizeof(s_wave[0].rows), "LDS of a compute unit");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, h = lane >> 5;
  const long long first = static_cast<long long>(blockIdx.x) * s.targets;
  const int here = static_cast<int>(min(static_cast<long long>(s.targets), s.num_targets - first));
  const int first_channel = blockIdx.y * kSingleColumns;
  const unsigned lds0 = static_cast<unsigned>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char *)(s_wave[wv].rows)));
  const int4v source_buffer = buffer_words(sources, source_bytes);
  const unsigned offset_stride = static_cast<unsigned>(s.packed_rows * s.packed_row_bytes);
  const int4v weight_buffer = buffer_words(wt, static_cast<unsigned>(s.offsets) * offset_stride);
  // eight lanes a row; rows lie in LDS with their pieces exchanged so that eight
  // rows' same piece are in eight different places
  const int load_row = lane / 8, piece = lane % 8 ^ load_row;
  const bool past_row = (s.chunks - 1) * BK + piece * 16 >= s.row_bytes;
  unsigned w_from[kSingleColumns / 8];
#pragma unroll
  for (int i = 0; i < kSingleColumns / 8; ++i) {
    w_from[i] = static_cast<unsigned>(min(first_channel + i * 8 + load_row, s.packed_rows - 1) * s.packed_row_bytes + piece * 16);
  }
  auto load_weights = [&](int o, int c) {
    const unsigned from = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(o) * offset_stride + c * BK);
#pragma unroll
    for (int i = 0; i < kSingleColumns / 8; ++i) {
      load_lds16(weight_buffer, w_from[i], from, __builtin_amdgcn_readfirstlane(lds0 + sizeof(s_wave[0].rows) + i * 1024));
    }
  };
  if (wv < s.offsets) load_weights(wv, 0);
  // the map: a lane's targets under the wavefront's offset
  int index[kRounds];
#pragma unroll
  for (int j = 0; j < kRounds; ++j) {
    const int t = j * 64 + lane;
    index[j] = wv < s.offsets && t < here ? kernel_map[wv * s.num_targets + first + t] : -1;
  }
  for (int i = tid; i < kSingleMost; i += 64 * kSingleWaves) {
    s_hits[i] = 0;
    s_source[i] = -1;
  }
  if (tid == 0) s_many = 0;
  __syncthreads();
  int count = 0;
#pragma unroll
  for (int j = 0; j < kRounds; ++j) {
    if (j * 64 >= here) continue;
    const int t = j * 64 + lane;
    const bool hit = index[j] >= 0;
    const unsigned long long votes = __ballot(hit);
    if (hit) {
      s_target[wv][count + __popcll(votes & lanes_below())] = static_cast<unsigned short>(t);
      s_source[t] = index[j];
      atomicAdd(&s_hits[t], 1);
    }
    count += __popcll(votes);
  }
  const int hits = __builtin_amdgcn_readfirstlane(count);      // (behind them: targets without a source)
  __syncthreads();
  for (int t = tid; t < here; t += 64 * kSingleWaves) {
    if (s_hits[t] > 1) s_many = 1;
  }
  if (wv == 0) {
    for (int j = 0; j * 64 < here; ++j) {
      const int t = j * 64 + lane;
      const bool none = t < here && s_hits[t] == 0;
      const unsigned long long votes = __ballot(none);
      if (none) s_target[0][count + __popcll(votes & lanes_below())] = static_cast<unsigned short>(t);
      count += __popcll(votes);
    }
  }
  __syncthreads();
  const bool many = s_many != 0;
  count = __builtin_amdgcn_readfirstlane(count);

  floatx16 acc[2][2];
  auto clear = [&]() {
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[a][b][j] = 0.0f;
      }
    }
  };
  // source(row): that of one of 64 rows; groups of 32 rows, those of the second
  // only where there are any
  bool ready = true;                           // the first stage of the weights is on its way
  auto multiply = [&](int o, int groups, bool more, auto source) {
    unsigned starts[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int at = i < 4 * groups ? source(i * 8 + load_row) : -1;
      starts[i] = at < 0 ? kPastEnd : static_cast<unsigned>(at) * static_cast<unsigned>(s.row_bytes) + piece * 16u;
    }
    auto load = [&](int c) {
      const unsigned from = __builtin_amdgcn_readfirstlane(c * BK);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (i >= 4 * groups) continue;
        load_lds16(source_buffer, c == s.chunks - 1 && past_row ? kPastEnd : starts[i], from,
                   __builtin_amdgcn_readfirstlane(lds0 + i * 1024));
      }
      if (c > 0 || !ready) load_weights(o, c);
    };
    load(0);
    for (int c = 0; c < s.chunks; ++c) {
      wait_loads<0>();
      uint4 x[4][2], w[4][2];
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const int at = ((2 * kk + h) ^ (r & 7)) * 16 + r * BK;
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          w[kk][b] = *reinterpret_cast<const uint4 *>(s_wave[wv].weights + b * 32 * BK + at);
          x[kk][b] = *reinterpret_cast<const uint4 *>(s_wave[wv].rows + b * 32 * BK + at);
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (c + 1 < s.chunks) {
        load(c + 1);
      } else if (more) {
        load_weights(o, 0);
      }
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          acc[0][b] = Mfma<T>::run(w[kk][b], x[kk][0], acc[0][b]);
          if (groups > 1) acc[1][b] = Mfma<T>::run(w[kk][b], x[kk][1], acc[1][b]);
        }
      }
    }
    ready = more;
  };
  // target(row): that of one of 64 rows, -1: none
  auto store = [&](int groups, auto target) {
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      if (a >= groups) break;
      int rows[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int t = target(a * 32 + (lane + i * 64) / 4);
        rows[i] = t < 0 ? -1 : static_cast<int>(first) + t;
      }
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int ch0 = first_channel + b * 32;
        if (ch0 < s.N) store_turned_rows<T>(acc[a][b], s_wave[wv].rows, lane, r, h, rows, ch0, s.N, ep, out);
      }
    }
  };
  if (!many) {
    for (int from = 0; from < hits; from += 64) {
      const int groups = hits - from > 32 ? 2 : 1;
      auto target = [&](int row) -> int { return from + row < hits ? s_target[wv][from + row] : -1; };
      clear();
      multiply(wv, groups, from + 64 < hits, [&](int row) {
        const int t = target(row);
        return t < 0 ? -1 : s_source[t];
      });
      store(groups, target);
    }
    if (hits == 0) wait_loads<0>();            // (none may land after the workgroup has gone)
    clear();
    for (int from = hits; from < count; from += 64) {
      store(count - from > 32 ? 2 : 1, [&](int row) -> int { return from + row < count ? s_target[wv][from + row] : -1; });
    }
    return;
  }
  ready = false;
  for (int from = wv * 32; from < here; from += 32 * kSingleWaves) {
    auto target = [&](int row) -> int { return from + row < here ? from + row : -1; };
    clear();
    for (int o = 0; o < s.offsets; ++o) {
      auto source = [&](int row) {
        const int t = target(row);
        return t < 0 ? -1 : kernel_map[o * s.num_targets + first + t];
      };
      floatx16 before[2] = {acc[0][0], acc[0][1]};
      multiply(o, 1, false, source);
      const bool used = source(r) >= 0;        // (a lane's sums are those of target r)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[0][b][j] = used ? acc[0][b][j] : before[b][j];
      }
    }
    store(1, target);
  }
}

template <typename T>
void single_forward(const T *sources, const T *packed, const int *kernel_map, int64_t S, int64_t Tn, int64_t O,
                    int64_t K, int64_t N, const Epilogue &ep, T *out, hipStream_t stream) {
  SingleShape s;
  s.num_targets = Tn;
  s.offsets = static_cast<int>(O);
  s.row_bytes = static_cast<int>(K * sizeof(T));
  s.chunks = static_cast<int>(div_ceil(s.row_bytes, kSingleStage));
  s.N = static_cast<int>(N);
  s.packed_row_bytes = s.chunks * kSingleStage;
  s.packed_rows = static_cast<int>(div_ceil(N, 32) * 32);
  const int64_t columns = div_ceil(N, int64_t{kSingleColumns});
  // the fewest rounds of workgroups, all of them full: a few workgroups more than
  // the compute units take as long as twice as many (160 -> 144 channels over
  // 60 000 targets, 258 workgroups of 704 36.7 us, 237 of 768 27.0)
  const int64_t cus = compute_units();
  int64_t rounds = std::max<int64_t>(1, div_ceil(Tn * columns, kSingleMost * cus)), targets;
  do {
    const int64_t beside = std::max<int64_t>(1, rounds++ * cus / columns);
    targets = div_ceil(div_ceil(Tn, beside), int64_t{64}) * 64;
  } while (targets > kSingleMost);
  s.targets = static_cast<int>(std::max<int64_t>(128, targets));
  const dim3 grid(static_cast<unsigned>(div_ceil(Tn, static_cast<int64_t>(s.targets))), static_cast<unsigned>(columns));
  single_forward_kernel<T><<<grid, 64 * kSingleWaves, 0, stream>>>(
      sources, static_cast<unsigned>(S * s.row_bytes), packed, kernel_map, s, reinterpret_cast<unsigned char *>(out), ep);
  check_launch("single_forward_kernel");
}

}  // namespace mnt

using namespace mnt;

static bool single_takes(int64_t O, int64_t K, int64_t N) {
  return O == kSingleOffsets && K % 8 == 0 && 2 * K > kSingleStage && 2 * K <= 512 && N % 8 == 0 && N >= 8 && N <= 512;
}

extern "C" int mnt_sparse_convolution_single(int64_t O, int64_t K, int64_t N, int float_dtype) {
  return float_dtype != MNT_FLOAT32 && single_takes(O, K, N) ? 1 : 0;
}

extern "C" int mnt_sparse_convolution_forward_single(
    const void *sources, const void *packed_weights, const int32_t *kernel_map, int64_t S, int64_t T, int64_t O,
    int64_t K, int64_t N, int float_dtype, const float *channel_scale, const float *channel_shift,
    const void *residual, int activation, float negative_slope, void *out, void *stream_) {
  return guarded([&] {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MNT_CHECK(S >= 0 && T >= 0 && S <= INT32_MAX && T <= INT32_MAX && single_takes(O, K, N),
              "bad shape S=%lld T=%lld O=%lld Cin=%lld Cout=%lld", (long long)S, (long long)T, (long long)O,
              (long long)K, (long long)N);
    MNT_CHECK(float_dtype == MNT_FLOAT16 || float_dtype == MNT_BFLOAT16, "this forward takes 16-bit features");
    MNT_CHECK(S * K * 2 < static_cast<int64_t>(kPastEnd),
              "source features of %lld bytes exceed the 4 GiB a buffer resource addresses", (long long)(S * K * 2));
    MNT_CHECK(activation >= MNT_ACT_NONE && activation <= MNT_ACT_RELU6, "unknown activation code %d", activation);
    MNT_CHECK(reinterpret_cast<uintptr_t>(sources) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(residual) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(packed_weights) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(channel_scale) % 4 == 0 &&
                  reinterpret_cast<uintptr_t>(channel_shift) % 4 == 0,
              "operands are not aligned (features, out, residual, weights: 16 bytes, scale / shift: 4 bytes)");
    if (T == 0) return;
    MNT_CHECK(out != nullptr && kernel_map != nullptr && packed_weights != nullptr, "null operand");
    const Epilogue ep = {channel_scale, channel_shift, residual, activation, negative_slope, nullptr};
    profile_mark("enter:implicit", stream);
    if (float_dtype == MNT_FLOAT16) {
      single_forward<half_t>(static_cast<const half_t *>(sources), static_cast<const half_t *>(packed_weights),
                             kernel_map, S, T, O, K, N, ep, static_cast<half_t *>(out), stream);
    } else {
      single_forward<bf16_t>(static_cast<const bf16_t *>(sources), static_cast<const bf16_t *>(packed_weights),
                             kernel_map, S, T, O, K, N, ep, static_cast<bf16_t *>(out), stream);
    }
    profile_mark("implicit", stream);
  });
}
