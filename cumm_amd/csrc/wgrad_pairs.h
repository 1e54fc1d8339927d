// Weight gradients over explicit pair lists:
//
//   dW[:, r, :] = act(alpha * sum over pairs i < count[r] of  dOut[pair_out[r][i]]^T (x) In[pair_in[r][i]]
//                     + beta * D[:, r, :])
//
// for one list (the ShuffleAB GEMM: the weight gradient of one kernel offset) or for up to 128 lists
// in one launch (the per-offset convolution).  Output channels are few and pairs are many, so the
// contraction has to be what is split: one workgroup per output tile, as a tiled GEMM cuts it, walks
// all pairs alone (6.05 ms for 150 k pairs of 64 + 64 channels; 16 ms for the 125 launches of a
// 5 x 5 x 5 kernel).
//
// The pairs of all lists are one stream of 32-pair steps (a list starts a new step); workgroup b takes
// the steps [b * per_wg, (b + 1) * per_wg), its four waves take every fourth step of a list each.
// A wave works alone: its own ring of NS stages (32 rows of dOut and of In, 128 bytes each) filled
// by direct-to-LDS loads, its own hand-counted waits, no barrier in the stream, and the whole 64 x 64
// tile in its accumulators (16 MFMAs for 16 transposing fragment reads; four waves on one tile
// would read as much for 4).  Where its share of a list ends the workgroup adds its four tiles up in
// LDS and stores the sum into slot b + r of the workspace; wgrad_pairs_finalize_kernel adds the
// slots of an element in workgroup order, applies the epilogue and rounds once.  No atomics, nothing
// to zero, the same bits from run to run.
//
// Bound by the gathered rows (2 x 128 bytes per pair and 64 x 64 channel block) and, below about
// 100 k pairs, by the chain of row numbers -> rows -> products -> slots -> finalize (two launches,
// 8 us for 256 to 4096 pairs).  Measured: 150 k pairs, 64 x 64 channels, f16: 11.6 + 4.2 us (6.05 ms on
// the tiled kernel; the 40 MB take 8.1 us at the rate of a large copy); 128 x 128 channels 20.2 us
// (6.36 ms); the 125 lists of a 5 x 5 x 5 kernel over 120 k voxels (386 k pairs) 19.2 us + finalize
// (16.1 ms).
#pragma once
#include "column_sum.h"
#include "common.h"
#include "lds_dma.h"

namespace cummhip {

constexpr int kWgradPairsMaxLists = 128;
constexpr int kWgradPairsSlotFloats = 64 * 64;

struct WgradPairsParams {
  const void *dout;            // rows of K channels, ldy elements apart
  const void *inp;             // rows of C channels, ldx elements apart
  const int32_t *pair_out, *pair_in;   // list r begins at r * list_stride
  float *slots;                // [(wgs + lists) * combos][64 x 64]
  int64_t ldy, ldx, list_stride;
  int32_t rows_y, rows_x;      // row numbers outside [0, rows) contribute nothing
  int32_t K, C, lists;
  int32_t kblocks, cblocks;    // 64-channel blocks; one workgroup per (share of the stream, block)
  int32_t wgs, per_wg;         // shares of the stream, steps per share
  int32_t step0[kWgradPairsMaxLists + 1];   // first step of each list; the last one = number of steps
  int32_t count[kWgradPairsMaxLists];
};

struct WgradPairsFinalizeParams {
  const float *slots;
  void *dw;                    // element (k, r, c) at k * ldw + r * ldr + c
  const void *src;             // the same with lds (0 = one row for every k)
  int64_t ldw, ldr, lds;
  int32_t K, C, lists, kblocks, cblocks, per_wg;
  float alpha, beta, act_alpha;
  int32_t act;
  int32_t step0[kWgradPairsMaxLists + 1];
};

// Four waves of one SIMD each: 4 x (4 stages of 8 KB + 4 KB of row numbers) = 144 KB of LDS, one
// workgroup per CU with 96 KB of rows in flight - twice what hides the 2 us that a gathered row takes
// under load at 5 TB/s.
template <class T>
__global__ __launch_bounds__(256) void wgrad_pairs_kernel(const WgradPairsParams p) {
  using E = Elem<T>;
  constexpr int NS = 4, L = NS - 1;     // ring stages, steps the loads run ahead
  constexpr int PART = 4096;            // 32 rows of 128 bytes
  constexpr int STAGE = 2 * PART;       // the dOut rows, then the In rows
  constexpr int CH = 8;                 // steps of a wave whose row numbers are fetched at once
  constexpr int PER_STEP = 8;           // row loads of a wave per step
  constexpr int PITCH = 68;             // floats per row of a tile parked in LDS (16-byte rows, banks spread)
  constexpr uint32_t kOob = 0x80000000u;
  static_assert(64 * PITCH * 4 <= NS * STAGE, "a wave parks its tile in its own ring");
  static_assert((L - 1) * PER_STEP + CH < 64, "loads in flight fit the counter");
  __shared__ __attribute__((aligned(16))) char ring[4][NS * STAGE];
  __shared__ __attribute__((aligned(16))) int numbers[4][2][2][CH * 32];   // [wave][buffer][dOut, In][pair]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, q = lane >> 4;

  // The channel blocks of one share run on one XCD (numbers w, w + 8, ...), one after the other: the
  // second block finds the rows' other halves in that XCD's L2.  Fewer than eight shares (more than 32
  // blocks) would leave XCDs idle: each then takes an eighth of all blocks of all shares in that order
  // (150 k pairs, 1024 x 1024 channels, one share: 5185 -> 736 us, 512 x 512: 258 -> 143 us; from eight
  // shares on the first map is the faster one, 128 x 128 channels 20.0 and 20.8 us).
  const int combos = p.kblocks * p.cblocks;
  const int xcd = blockIdx.x & 7, nth = blockIdx.x >> 3;
  const int unit = p.wgs >= 8 ? nth : xcd * (int)(gridDim.x >> 3) + nth;
  const int combo = unit % combos;
  const int b = p.wgs >= 8 ? (unit / combos) * 8 + xcd : unit / combos;
  if (b >= p.wgs) return;
  const int kb = combo / p.cblocks, cb = combo % p.cblocks;

  const v4i y_rsrc = rsrc_words(p.dout, (uint32_t)(((int64_t)(p.rows_y - 1) * p.ldy + p.K) * 2));
  const v4i x_rsrc = rsrc_words(p.inp, (uint32_t)(((int64_t)(p.rows_x - 1) * p.ldx + p.C) * 2));
  const uint32_t y_pitch = (uint32_t)p.ldy * 2u, x_pitch = (uint32_t)p.ldx * 2u;

  // loader: lane l of load t fetches 16-byte chunk l % 8 of row 8 t + l / 8; chunks are permuted by
  // 2 * ((row / 2) % 4) against bank conflicts of the transposing reads, on the global side
  auto swz = [](int row) { return 2 * ((row >> 1) & 3); };
  const int lrow = lane >> 3;
  const int gch = ((lane & 7) ^ swz(lrow)) * 8;     // (8 t does not change the permutation)
  const uint32_t y_rows = kb * 64 + gch < p.K ? (uint32_t)p.rows_y : 0u;    // (no rows for a channel past the end)
  const uint32_t x_rows = cb * 64 + gch < p.C ? (uint32_t)p.rows_x : 0u;
  const uint32_t y_ch = (uint32_t)(kb * 64 + gch) * 2u, x_ch = (uint32_t)(cb * 64 + gch) * 2u;
  // reader: lane i of a 16-lane group points at row i / 4 of four, channels 4 (i % 4) ..
  int rd[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int row = q * 8 + h * 4 + (l16 >> 2), col = g * 16 + 4 * (l16 & 3);
      rd[h][g] = row * 128 + (((col >> 3) ^ swz(row)) * 16) + (col & 7) * 2;
    }
  const uint32_t ring_at = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_addr(&ring[wave][0]));
  const uint32_t num_at = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_addr(&numbers[wave][0][0][0]));

  const int first = b * p.per_wg;
  const int last = first + p.per_wg < p.step0[p.lists] ? first + p.per_wg : p.step0[p.lists];
  // (the lists before this share, counted by all lanes at once: a loop would be one dependent load each)
  int r = 0;
  if (p.lists > 1) {
    const int a = lane, c = lane + 64;
    r = __builtin_popcountll(__ballot(a < p.lists && p.step0[a + 1] <= first)) +
        __builtin_popcountll(__ballot(c < p.lists && p.step0[c + 1] <= first));
    r = __builtin_amdgcn_readfirstlane(r);
  }

  for (int at = first; at < last; ++r) {
    const int list_end = p.step0[r + 1];
    if (list_end <= at) continue;                            // an empty list
    const int end = list_end < last ? list_end : last;
    const int s0 = at - p.step0[r];                          // this segment: steps s0 .. s0 + n - 1 of list r
    const int n = end - at;
    const int mine = (n - wave + 3) >> 2;                    // of which this wave takes wave, wave + 4, ...
    const int count = p.count[r];
    const v4i yl = rsrc_words(p.pair_out + (int64_t)r * p.list_stride, (uint32_t)count * 4u);
    const v4i xl = rsrc_words(p.pair_in + (int64_t)r * p.list_stride, (uint32_t)count * 4u);

    auto load_numbers = [&](int c) __attribute__((always_inline)) {
      const uint32_t dst = num_at + (uint32_t)(c & 1) * (2 * CH * 32 * 4);
#pragma unroll
      for (int t = 0; t < CH / 2; ++t) {
        const int j = c * CH + 2 * t + (lane >> 5);
        const int i = (s0 + wave + 4 * j) * 32 + (lane & 31);
        const uint32_t off = j < mine && i < count ? (uint32_t)i * 4u : kOob;
        dma_b32(yl, dst + t * 256, off, 0);
        dma_b32(xl, dst + CH * 32 * 4 + t * 256, off, 0);
      }
    };
    // a step or a pair past the end, a row or a channel out of range: fetched at an offset outside the
    // buffer, zeros arrive, and the number of loads in flight stays the same
    uint32_t yo[4], xo[4];
    auto offsets = [&](int j) __attribute__((always_inline)) {
      const int *nb = &numbers[wave][(j / CH) & 1][0][(j % CH) * 32];
      const int left = j < mine ? count - (s0 + wave + 4 * j) * 32 : 0;
      int o[4], i[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        o[t] = nb[t * 8 + lrow];
        i[t] = nb[CH * 32 + t * 8 + lrow];
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const uint32_t in = t * 8 + lrow < left ? 0u : kOob;
        yo[t] = ((uint32_t)o[t] < y_rows ? (uint32_t)o[t] * y_pitch + y_ch : kOob) | in;
        xo[t] = ((uint32_t)i[t] < x_rows ? (uint32_t)i[t] * x_pitch + x_ch : kOob) | in;
      }
    };
    auto issue = [&](int j) __attribute__((always_inline)) {
      const uint32_t dst = ring_at + (uint32_t)__builtin_amdgcn_readfirstlane((j % NS) * STAGE);
#pragma unroll
      for (int t = 0; t < 4; ++t) dma_b128(y_rsrc, dst + t * 1024, yo[t], 0);
#pragma unroll
      for (int t = 0; t < 4; ++t) dma_b128(x_rsrc, dst + PART + t * 1024, xo[t], 0);
    };

    v4f acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = v4f{0, 0, 0, 0};

    load_numbers(0);
    wait_vmcnt<0>();
    asm volatile("" ::: "memory");
    load_numbers(1);
#pragma unroll
    for (int j = 0; j < L; ++j) {
      offsets(j);
      issue(j);
    }
    offsets(L);
    for (int j = 0; j < mine; ++j) {
      wait_vmcnt<(L - 1) * PER_STEP>();
      asm volatile("" ::: "memory");
      typedef short v4s __attribute__((ext_vector_type(4)));
      typedef __attribute__((address_space(3))) v4s *lds_v4s;
      const char *st = &ring[wave][(j % NS) * STAGE];
      v4i yf[4], xf[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)CUMM_LDS_PTR(st + rd[0][g]));
        const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)CUMM_LDS_PTR(st + rd[1][g]));
        yf[g] = __builtin_bit_cast(v4i, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)CUMM_LDS_PTR(st + PART + rd[0][g]));
        const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)CUMM_LDS_PTR(st + PART + rd[1][g]));
        xf[g] = __builtin_bit_cast(v4i, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
      issue(j + L);
      // The row numbers of chunk c + 1 are requested when the last of chunk c - 1 have been used; they
      // are needed CH steps of row loads later, which is more than are ever in flight.
      if ((j + L + 1) % CH == 0) load_numbers((j + L + 1) / CH + 1);
      offsets(j + L + 1);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) acc[i][jj] = E::mfma(yf[i], xf[jj], acc[i][jj]);
    }
    wait_vmcnt<0>();    // the fetches past the end
    asm volatile("" ::: "memory");

    // ---- the workgroup's sum over its four waves: each parks its tile in its own ring
    float *park = reinterpret_cast<float *>(&ring[wave][0]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int x = 0; x < 4; ++x) park[(i * 16 + 4 * q + x) * PITCH + j * 16 + l16] = acc[i][j][x];
    __syncthreads();
    float *slot = p.slots + (int64_t)((b + r) * combos + combo) * kWgradPairsSlotFloats;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int at4 = (e * 256 + tid) * 4;
      const int off = (at4 >> 6) * PITCH + (at4 & 63);
      v4f sum = *reinterpret_cast<const v4f *>(reinterpret_cast<const float *>(&ring[0][0]) + off);
#pragma unroll
      for (int w = 1; w < 4; ++w) sum += *reinterpret_cast<const v4f *>(reinterpret_cast<const float *>(&ring[w][0]) + off);
      *reinterpret_cast<v4f *>(slot + at4) = sum;
    }
    __syncthreads();
    at = end;
  }
}

// Four consecutive channels of list blockIdx.y per group of G lanes; lane g adds the g-th share of the
// slots first to last, then the G sums are combined pairwise: the order depends on the number of
// slots only.  Latency-bound (loads in batches of eight).  SUMS: with bias sums to finish, whose workgroups come first
// (a kernel of its own: their LDS and branch cost the others 0.2 of 14.8 us, 150 k pairs of 64 x 64 channels).
template <class T, int G, bool WIDE, bool SUMS>
__global__ __launch_bounds__(256) void wgrad_pairs_finalize_kernel(const WgradPairsFinalizeParams p, const ColumnFinalParams sums) {
  using E = Elem<T>;
  const int r = (int)blockIdx.y - (SUMS ? 1 : 0);
  if constexpr (SUMS) {
    if (r < 0) {
      for (int group = blockIdx.x; group < sums.groups; group += gridDim.x) column_final<T>(sums, group);
      return;
    }
  }
  const uint32_t g = threadIdx.x % G;
  const uint32_t group = blockIdx.x * (256 / G) + threadIdx.x / G;
  const uint32_t c4 = (uint32_t)p.C / 4u;
  const bool on = group < (uint32_t)p.K * c4;
  const uint32_t gg = on ? group : 0u;
  const int nn = (int)(gg % c4) * 4, mm = (int)(gg / c4);
  const int combos = p.kblocks * p.cblocks;
  const int s0 = p.step0[r], s1 = p.step0[r + 1];
  const int b0 = s0 / p.per_wg;
  const int count = on && s1 > s0 ? (s1 - 1) / p.per_wg - b0 + 1 : 0;
  const float *first = p.slots + (int64_t)((b0 + r) * combos + (mm >> 6) * p.cblocks + (nn >> 6)) * kWgradPairsSlotFloats +
                       (mm & 63) * 64 + (nn & 63);
  const int64_t next = (int64_t)combos * kWgradPairsSlotFloats;
  const int share = (count + G - 1) / G;
  const int lo = (int)g * share, hi = lo + share < count ? lo + share : count;
  v4f sum = v4f{0, 0, 0, 0};
  for (int t0 = lo; t0 < hi; t0 += 8) {
    v4f part[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int t = t0 + u < hi ? t0 + u : hi - 1;     // (a repeat past the share, not added)
      part[u] = *reinterpret_cast<const v4f *>(first + t * next);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (t0 + u < hi) sum += part[u];
  }
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    float v = sum[x];
#pragma unroll
    for (int d = 1; d < G; d *= 2) v += __shfl_xor(v, d, 64);
    sum[x] = v;
  }
  if (!on || g != 0) return;
  const int64_t at = (int64_t)mm * p.ldw + (int64_t)r * p.ldr + nn;
  const int64_t from = (int64_t)mm * p.lds + (p.lds ? (int64_t)r * p.ldr : 0) + nn;
  if constexpr (WIDE) {
    v4f out, src = v4f{0, 0, 0, 0};
    if (p.beta != 0.0f) src = *reinterpret_cast<const v4f *>(reinterpret_cast<const float *>(p.src) + from);
#pragma unroll
    for (int x = 0; x < 4; ++x)
      out[x] = apply_act(p.beta != 0.0f ? __builtin_fmaf(p.alpha, sum[x], p.beta * src[x]) : p.alpha * sum[x], p.act, p.act_alpha);
    *reinterpret_cast<v4f *>(reinterpret_cast<float *>(p.dw) + at) = out;
  } else {
    typedef uint16_t v4h __attribute__((ext_vector_type(4)));
    v4h out, src = v4h{0, 0, 0, 0};
    if (p.beta != 0.0f) src = *reinterpret_cast<const v4h *>(reinterpret_cast<const uint16_t *>(p.src) + from);
#pragma unroll
    for (int x = 0; x < 4; ++x)
      out[x] = E::from_float(apply_act(p.beta != 0.0f ? __builtin_fmaf(p.alpha, sum[x], p.beta * E::to_float(src[x])) : p.alpha * sum[x],
                                       p.act, p.act_alpha));
    *reinterpret_cast<v4h *>(reinterpret_cast<uint16_t *>(p.dw) + at) = out;
  }
}

}  // namespace cummhip
