// Row-wise helper kernels around the GEMM / sparse-convolution kernels: HBM-bound elementwise and
// reduction work that a caller of the convolution needs between launches.
//
//   finish_rows      out[r, c] = cvt(act(alpha * acc[r, c] + beta * bias[c])) from an fp32 image of
//                    the result (the per-offset "native" convolution accumulates in fp32 and
//                    rounds once, here)
//   relu_backward    dst = grad where the forward output was positive, else 0; with sums also the
//                    column sums of dst, which then cost no pass of their own
//   column_sum       dst[c] = cvt(sum over rows of src[r, c]) in fp32, in a fixed order (the
//                    gradient of a bias): per-block partial sums, then a sum over blocks in
//                    block order, so the result is the same from run to run
//
// All three move 16-byte pieces (8 two-byte elements), consecutive lanes on consecutive pieces.  The gate
// and the sums are bound by HBM and run as many short workgroups in memory order: a resident grid
// whose workgroups walk the tensor with a stride drifts apart and loses open pages (gate of 652 k rows of
// 256 channels, 1.0 GB: 203 us with 4096 workgroups walking, 169 us with one per 256 pieces).  Operands
// of more than kStreamBytes are loaded non-temporally (1 M rows of 128: 130 -> 110 us; 161 us for the
// 1.0 GB; 64 MB with the gradient fresh from its producer 36 -> 33 us, all of it in memory 59 -> 37;
// only where the last-level cache holds all three tensors, from a call just before, up to 90 MB each,
// it costs: 300 k rows of 128 again and again 34 -> 37 us).
#include "launch.h"

namespace cummhip {

namespace {

template <class T>
__device__ __forceinline__ void unpack8(const v4i &v, float (&f)[8]) {
  const uint16_t *h = reinterpret_cast<const uint16_t *>(&v);
#pragma unroll
  for (int x = 0; x < 8; ++x) f[x] = Elem<T>::to_float(h[x]);
}
template <class T>
__device__ __forceinline__ v4i pack8(const float (&f)[8]) {
  v4i v;
  uint16_t *h = reinterpret_cast<uint16_t *>(&v);
#pragma unroll
  for (int x = 0; x < 8; ++x) h[x] = Elem<T>::from_float(f[x]);
  return v;
}

// one thread per 8 consecutive channels of one row
template <class T>
__global__ __launch_bounds__(256) void finish_rows_kernel(const FinishRowsParams p) {
  const int64_t vecs_per_row = p.channels / 8;
  const int64_t total = p.rows * vecs_per_row;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / vecs_per_row;
    const int c = (int)(i - r * vecs_per_row) * 8;
    const v4f *ap = reinterpret_cast<const v4f *>(p.acc + r * p.channels + c);
    const v4f a0 = ap[0], a1 = ap[1];
    float b[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (p.bias != nullptr && p.beta != 0.0f)
      unpack8<T>(*reinterpret_cast<const v4i *>(reinterpret_cast<const uint16_t *>(p.bias) + c), b);
    float t[8];
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      const float a = x < 4 ? a0[x & 3] : a1[x & 3];
      // the fused form of the GEMM kernels' epilogue
      const float v = p.bias != nullptr && p.beta != 0.0f ? __builtin_fmaf(p.alpha, a, p.beta * b[x]) : p.alpha * a;
      t[x] = apply_act(v, p.act, p.act_alpha);
    }
    *reinterpret_cast<v4i *>(reinterpret_cast<uint16_t *>(p.out) + r * p.channels + c) = pack8<T>(t);
  }
}

constexpr int kBatch = 4;   // pieces per operand that a row lane of the sums has on their way

template <class T>
__device__ __forceinline__ v4i gate8(const v4i &g, const v4i &o) {
  const uint16_t *gh = reinterpret_cast<const uint16_t *>(&g);
  const uint16_t *oh = reinterpret_cast<const uint16_t *>(&o);
  v4i r;
  uint16_t *rh = reinterpret_cast<uint16_t *>(&r);
#pragma unroll
  for (int x = 0; x < 8; ++x) rh[x] = Elem<T>::to_float(oh[x]) > 0.0f ? gh[x] : (uint16_t)0;
  return r;
}

// the elements of g that eight bits let through
__device__ __forceinline__ v4i gate8_bits(const v4i &g, uint32_t bits) {
  v4i r;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const uint32_t lo = (uint32_t)((int32_t)(bits << (31 - 2 * x)) >> 31), hi = (uint32_t)((int32_t)(bits << (30 - 2 * x)) >> 31);
    r[x] = g[x] & (int)((lo & 0xFFFFu) | (hi & 0xFFFF0000u));
  }
  return r;
}

// thread: eight channels of a position (one that names no row of out is left alone, as by the convolution kernels)
__global__ __launch_bounds__(256) void gate_bits_kernel(uint8_t *gate, const v4i *out, const int32_t *order, int n, int rows, int pieces) {
  const int64_t total = (int64_t)n * pieces;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int pos = (int)(i / pieces), piece = (int)(i - (int64_t)pos * pieces);
    const int row = order ? order[pos] : pos;
    if ((uint32_t)row >= (uint32_t)rows) continue;
    gate[((int64_t)(piece >> 3) * n + pos) * 8 + (piece & 7)] = (uint8_t)positive8(out[(int64_t)row * pieces + piece]);
  }
}

constexpr size_t kStreamBytes = (size_t)64 << 20;
constexpr int kNonTemporal = 2;      // of a buffer load: aux bit 1

template <bool NT>
__device__ __forceinline__ v4i load_piece(const v4i *p) {
  return NT ? __builtin_nontemporal_load(p) : *p;
}

template <class T, bool NT>
__global__ __launch_bounds__(256) void relu_backward_kernel(v4i *dst, const v4i *grad, const v4i *out, size_t vecs) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < vecs) dst[i] = gate8<T>(load_piece<NT>(grad + i), load_piece<NT>(out + i));
}

// partial[b][c] = sum of src[r][c] over the rows of block b - with GATE of the gated rows, which are
// written to gated on the way.  Thread t takes the 8-channel piece t % V of the rows t / V, t / V + R,
// ... of its block (V pieces per row, R = 256 / V rows at a time); the R row lanes of a piece are then
// summed through LDS in lane order.  The first pre_blocks workgroups prepare a weight gradient instead
// (wgrad_prepare: lists and zeros that depend on nothing here; in a launch of its own it is 4 us).
// GATE: 0 = no gate; 1 = the forward output; 2 = its bits, an eighth of the bytes of one of three tensors, the rows
// then in the order of the positions, in which the bits lie (rows of 128 bytes and more in any order move as
// fast): 128 channels at 1 M voxels 117 -> 83 us, 797 k rows of 256 channels 195 -> 147; passes forward and
// backward 716.8 -> 695.1 and 779.1 -> 736.0.  3 = the forward output, the rows in that order too: the sums of 2 for
// whoever has no bits.  2 and 3 by 32-bit offsets into bounded buffers: rows of 64 channels at 120 k positions 9.7 us; with a
// look at each row before its load and store 10.4, unchecked and with 64-bit addresses 9.9.
template <class T, int GATE, bool NT>
__global__ __launch_bounds__(256) void column_partial_kernel(const ColumnSumParams p, const WgradPrepareParams pre, int pre_blocks) {
  __shared__ float lds[256][9];
  if ((int)blockIdx.x < pre_blocks) {
    wgrad_prepare(pre, blockIdx.x, pre_blocks);
    return;
  }
  const int64_t block = blockIdx.x - pre_blocks;
  const int V = p.channels / 8;
  const int R = 256 / V;
  const int t = threadIdx.x;
  const int piece = t % V, lane_row = t / V;
  float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (lane_row < R) {
    const int64_t r0 = block * p.rows_per_block;
    int64_t r1 = r0 + p.rows_per_block;
    if (r1 > p.rows) r1 = p.rows;
    const v4i *src = reinterpret_cast<const v4i *>(p.src) + piece;
    const v4i *out = reinterpret_cast<const v4i *>(p.out) + piece;
    v4i *gated = reinterpret_cast<v4i *>(p.gated) + piece;
    // By position (tensors below 2 GiB: checked on the host): nothing branches, a position past the block and one that
    // names no row lie outside the buffers.
    if constexpr (GATE >= 2) {
      const uint32_t row_bytes = (uint32_t)p.channels * 2u, bytes = (uint32_t)p.rows * row_bytes, rows = (uint32_t)p.rows;
      const __amdgpu_buffer_rsrc_t rs_order = make_rsrc(p.order, rows * 4u), rs_src = make_rsrc(p.src, bytes), rs_to = make_rsrc(p.gated, bytes);
      const __amdgpu_buffer_rsrc_t rs_gate = GATE == 2 ? make_rsrc(p.gate, (uint32_t)((p.channels + 63) >> 6) * rows * 8u) : make_rsrc(p.out, bytes);
      const uint32_t plane = (uint32_t)(piece >> 3) * rows * 8u + (uint32_t)(piece & 7);
      constexpr int kHint = NT ? kNonTemporal : 0;
      for (uint32_t pos = (uint32_t)r0 + (uint32_t)lane_row; pos < (uint32_t)r1; pos += kBatch * R) {
        v4i g[kBatch], o[kBatch];
        uint32_t at[kBatch], b[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          const uint32_t here = pos + (uint32_t)(u * R);
          const bool in = here < (uint32_t)r1;
          at[u] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs_order, here * 4u, 0, 0);
          if constexpr (GATE == 2) b[u] = __builtin_amdgcn_raw_buffer_load_b8(rs_gate, in ? plane + here * 8u : kOob, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          at[u] = at[u] < rows && pos + (uint32_t)(u * R) < (uint32_t)r1 ? at[u] * row_bytes + (uint32_t)piece * 16u : kOob;
          g[u] = __builtin_amdgcn_raw_buffer_load_b128(rs_src, at[u], 0, kHint);
          if constexpr (GATE == 3) o[u] = __builtin_amdgcn_raw_buffer_load_b128(rs_gate, at[u], 0, kHint);
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          if constexpr (GATE == 2) g[u] = gate8_bits(g[u], b[u]);
          else g[u] = gate8<T>(g[u], o[u]);
          __builtin_amdgcn_raw_buffer_store_b128(g[u], rs_to, at[u], 0, 0);
          float f[8];
          unpack8<T>(g[u], f);
#pragma unroll
          for (int x = 0; x < 8; ++x) s[x] += f[x];
        }
      }
    } else {
      for (int64_t r = r0 + lane_row; r < r1; r += kBatch * R) {
        v4i g[kBatch], o[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          const int64_t at = (r + u * R < r1 ? r + u * R : r) * V;
          g[u] = load_piece<NT>(src + at);
          if constexpr (GATE) o[u] = load_piece<NT>(out + at);
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          if (r + u * R >= r1) break;
          if constexpr (GATE) {
            g[u] = gate8<T>(g[u], o[u]);
            gated[(r + u * R) * V] = g[u];
          }
          float f[8];
          unpack8<T>(g[u], f);
#pragma unroll
          for (int x = 0; x < 8; ++x) s[x] += f[x];
        }
      }
    }
  }
#pragma unroll
  for (int x = 0; x < 8; ++x) lds[t][x] = s[x];
  __syncthreads();
  if (lane_row == 0) {
    for (int j = 1; j < R; ++j)
#pragma unroll
      for (int x = 0; x < 8; ++x) s[x] += lds[j * V + piece][x];
    float *dst = p.partial + block * p.channels + piece * 8;
#pragma unroll
    for (int x = 0; x < 8; ++x) dst[x] = s[x];
  }
}

// The blocks of slice blockIdx.y of gridDim.y; the last stage (one slice) converts.
template <class T, bool LAST>
__global__ __launch_bounds__(256) void column_final_kernel(const ColumnFinalParams p, float *to) {
  if constexpr (LAST) {
    column_final<T>(p, blockIdx.x);
  } else {
    const int slice = (p.blocks + gridDim.y - 1) / gridDim.y;
    const int first = (int)blockIdx.y * slice, end = first + slice < p.blocks ? first + slice : p.blocks;
    const float total = column_final_sum(p.from, p.channels, first, end, blockIdx.x);
    const int c = blockIdx.x * 16 + threadIdx.x;
    if (threadIdx.x < 16 && c < p.channels) to[(int64_t)blockIdx.y * p.channels + c] = total;
  }
}

unsigned grid_for(size_t items) {
  size_t blocks = (items + 255) / 256;
  if (blocks > 256 * 16) blocks = 256 * 16;
  return (unsigned)(blocks > 0 ? blocks : 1);
}

}  // namespace

hipError_t launch_finish_rows(const FinishRowsParams &p, bool bf16, hipStream_t s) {
  const size_t items = (size_t)p.rows * (size_t)(p.channels / 8);
  if (items == 0) return hipSuccess;
  if (bf16) hipLaunchKernelGGL(finish_rows_kernel<BF16>, dim3(grid_for(items)), dim3(256), 0, s, p);
  else hipLaunchKernelGGL(finish_rows_kernel<F16>, dim3(grid_for(items)), dim3(256), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_gate_bits(uint8_t *gate, const void *out, const int32_t *order, int n, int rows, int channels, hipStream_t s) {
  if (n <= 0 || channels <= 0) return hipSuccess;
  const int pieces = channels / 8;
  hipLaunchKernelGGL(gate_bits_kernel, dim3(grid_for((size_t)n * pieces)), dim3(256), 0, s, gate, reinterpret_cast<const v4i *>(out), order, n, rows, pieces);
  return hipGetLastError();
}

constexpr size_t kGatePieces = (size_t)1 << 31;      // of one launch, which has fewer than 2^32 threads

template <class T>
static hipError_t relu_backward(void *dst, const void *grad, const void *out, size_t vecs, hipStream_t s) {
  v4i *d = reinterpret_cast<v4i *>(dst);
  const v4i *g = reinterpret_cast<const v4i *>(grad), *o = reinterpret_cast<const v4i *>(out);
  const bool stream = vecs * 16 > kStreamBytes;
  for (size_t at = 0; at < vecs; at += kGatePieces) {
    const size_t n = vecs - at < kGatePieces ? vecs - at : kGatePieces;
    const dim3 grid((unsigned)((n + 255) / 256));
    if (stream) hipLaunchKernelGGL((relu_backward_kernel<T, true>), grid, dim3(256), 0, s, d + at, g + at, o + at, n);
    else hipLaunchKernelGGL((relu_backward_kernel<T, false>), grid, dim3(256), 0, s, d + at, g + at, o + at, n);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_relu_backward(void *dst, const void *grad, const void *out, size_t vecs, bool bf16, hipStream_t s) {
  return bf16 ? relu_backward<BF16>(dst, grad, out, vecs, s) : relu_backward<F16>(dst, grad, out, vecs, s);
}

// Rows per block: two batches per row lane (32 KB of each operand), more below kFewBlocks blocks' worth of
// rows, where one stage of sums is to do (at most 1024 blocks).
constexpr int kFewBlocks = 1024, kSlices = 64;
static int64_t column_rows_per_block(int64_t rows, int channels) {
  const int V = channels / 8;
  const int R = V > 0 && V <= 256 ? 256 / V : 1;
  const int64_t small = (int64_t)R * 2 * kBatch;
  const int64_t blocks = (rows + small - 1) / small;
  if (blocks > 4 * kFewBlocks) return small;
  int64_t few = blocks;
  if (few > kFewBlocks) few = kFewBlocks;
  return few > 0 ? (rows + few - 1) / few : 1;
}
static int column_blocks(int64_t rows, int channels) {
  const int64_t per = column_rows_per_block(rows, channels);
  return rows > 0 ? (int)((rows + per - 1) / per) : 1;
}
// rows of partial sums in the workspace: one per block, and one per slice of the first of two stages
int column_sum_blocks(int64_t rows, int channels) {
  const int blocks = column_blocks(rows, channels);
  return blocks > kFewBlocks ? blocks + kSlices : blocks;
}

template <class T>
static void column_partial(const ColumnSumParams &p, const WgradPrepareParams &pre, int pre_blocks, hipStream_t s) {
  const bool stream = (size_t)p.rows * (size_t)p.channels * 2 > kStreamBytes;
  const dim3 grid((unsigned)(p.blocks + pre_blocks));
  const auto launch = [&](auto gate) {
    constexpr int GATE = decltype(gate)::value;
    if (stream) hipLaunchKernelGGL((column_partial_kernel<T, GATE, true>), grid, dim3(256), 0, s, p, pre, pre_blocks);
    else hipLaunchKernelGGL((column_partial_kernel<T, GATE, false>), grid, dim3(256), 0, s, p, pre, pre_blocks);
  };
  if (p.gated == nullptr) launch(std::integral_constant<int, 0>{});
  else if (p.gate != nullptr) launch(std::integral_constant<int, 2>{});
  else if (p.order != nullptr) launch(std::integral_constant<int, 3>{});
  else launch(std::integral_constant<int, 1>{});
}

hipError_t launch_column_partial(ColumnSumParams p, const WgradPrepareParams *pre, int pre_blocks, bool bf16, hipStream_t s,
                                 ColumnFinalParams *last) {
  p.blocks = column_blocks(p.rows, p.channels);
  p.rows_per_block = column_rows_per_block(p.rows, p.channels);
  const WgradPrepareParams none = {};
  if (bf16) column_partial<BF16>(p, pre ? *pre : none, pre ? pre_blocks : 0, s);
  else column_partial<F16>(p, pre ? *pre : none, pre ? pre_blocks : 0, s);
  hipError_t e = hipGetLastError();
  *last = ColumnFinalParams{p.partial, p.dst, p.blocks, p.channels, (p.channels + 15) / 16};
  if (e == hipSuccess && p.blocks > kFewBlocks) {
    float *to = p.partial + (int64_t)p.blocks * p.channels;
    hipLaunchKernelGGL((column_final_kernel<F16, false>), dim3((unsigned)last->groups, kSlices), dim3(256), 0, s, *last, to);
    e = hipGetLastError();
    last->from = to;
    last->blocks = kSlices;
  }
  return e;
}

hipError_t launch_column_sum(const ColumnSumParams &p, bool bf16, hipStream_t s) {
  ColumnFinalParams last;
  const hipError_t e = launch_column_partial(p, nullptr, 0, bf16, s, &last);
  if (e != hipSuccess) return e;
  if (bf16) hipLaunchKernelGGL((column_final_kernel<BF16, true>), dim3((unsigned)last.groups), dim3(256), 0, s, last, nullptr);
  else hipLaunchKernelGGL((column_final_kernel<F16, true>), dim3((unsigned)last.groups), dim3(256), 0, s, last, nullptr);
  return hipGetLastError();
}

}  // namespace cummhip
