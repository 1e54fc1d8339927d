// Column sums of partial sums: the last step of a bias gradient, in a launch of its own (elementwise_inst.hip) or
// in workgroups of the launch that rounds the weight gradient.  (The lists of live tiles that a weight gradient begins
// with ride on the launch of the gate in turn: two launches of 4 - 5 us each less in a backward pass.  Forward and
// backward, us: 300 k frame of two layers 572.0 -> 554.3, 128 channels at 1 M voxels 766.0 -> 756.7, stride 2,
// 128 -> 256 channels at 300 k 823.1 -> 813.7.)
#pragma once
#include "common.h"

namespace cummhip {

struct ColumnFinalParams {
  const float *from;    // [blocks, channels]
  void *dst;            // [channels]
  int32_t blocks, channels;
  int32_t groups;       // workgroups that do this: one per 16 channels (0 = nothing to do)
};

constexpr int kColumnFinalBatch = 16;   // loads that a thread has in flight

// Sum of the blocks [first, end) for the channels 16 group ... in a fixed shape: 64 shares of the blocks, each
// added in block order, then sixteen sums in order, then those four.  256 threads, four channels of one
// share each; the sum of channel 16 group + t comes back in thread t < 16.  A chain of few round trips:
// 1024 blocks are one batch of loads.
__device__ __forceinline__ float column_final_sum(const float *from, int channels, int first, int end, int group) {
  typedef float v4f_any __attribute__((ext_vector_type(4), aligned(4)));      // (a workspace is aligned to floats)
  __shared__ float part[64][17];
  const int quad = threadIdx.x & 3, j = threadIdx.x >> 2;
  const int c = group * 16 + quad * 4;
  const int share = (end - first + 63) >> 6;
  const int b0 = first + j * share, b1 = b0 + share < end ? b0 + share : end;
  v4f s = v4f{0, 0, 0, 0};
  if (c < channels) {
    for (int b = b0; b < b1; b += kColumnFinalBatch) {
      v4f v[kColumnFinalBatch];
#pragma unroll
      for (int u = 0; u < kColumnFinalBatch; ++u)     // (a repeat past the share, not added)
        v[u] = *reinterpret_cast<const v4f_any *>(from + (int64_t)(b + u < b1 ? b + u : b) * channels + c);
#pragma unroll
      for (int u = 0; u < kColumnFinalBatch; ++u)
        if (b + u < b1) s += v[u];
    }
  }
#pragma unroll
  for (int x = 0; x < 4; ++x) part[j][quad * 4 + x] = s[x];
  __syncthreads();
  const int cl = threadIdx.x & 15, k0 = threadIdx.x >> 4;
  float sum = 0.0f;
  if (threadIdx.x < 64) {
    sum = part[k0 * 16][cl];
#pragma unroll
    for (int k = 1; k < 16; ++k) sum += part[k0 * 16 + k][cl];
  }
  __syncthreads();
  if (threadIdx.x < 64) part[k0][cl] = sum;
  __syncthreads();
  sum = ((part[0][cl] + part[1][cl]) + part[2][cl]) + part[3][cl];
  __syncthreads();      // (the next group's turn)
  return sum;
}

// the sums of one group of channels, rounded
template <class T>
__device__ __forceinline__ void column_final(const ColumnFinalParams &p, int group) {
  const float total = column_final_sum(p.from, p.channels, 0, p.blocks, group);
  const int c = group * 16 + (int)threadIdx.x;
  if (threadIdx.x < 16 && c < p.channels) reinterpret_cast<uint16_t *>(p.dst)[c] = Elem<T>::from_float(total);
}

}  // namespace cummhip
