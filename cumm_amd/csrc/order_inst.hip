// From finished pair tables to what the mask-based kernels read: the masks, an order of the positions
// in which a tile's masks share their bits, the masks and the table in that order, and the launch
// hints - for one table or for the two of a strided layer in the same launches.  (The reference's
// callers take masks and sort from spconv, cumm/conv/main_real_spconv.py:91-145; its iterator forms
// the table's index per access, cumm/conv/sparse_iters.py:280-357.)
//
// Any order is a valid input of the convolution kernels; it decides only how many kernel offsets a tile
// of 64 or 128 positions has in the OR of its masks, which is what a tile costs.  This one needs two
// radix passes of nine bits, because its key has 18 bits:
//   * one mask word: ascending number of offsets, then ascending value as a rank among the words with
//     that many bits (combinatorial number system), exact up to five offsets (101 584 words of 27
//     bits), the rank scaled into an equal share of what is left of the 18 bits above that.  The
//     tiles' offsets add up to what the full 32-bit sort by count and value gives (45 114 against
//     45 113 at 1 M voxels), which needs four passes.
//   * several words: two bits of weight (more than 2, 4, 8 offsets), a Gray code of the twelve outer planes of
//     the kernel (is there a neighbour with the lowest, second, second last, last index along z, y, x),
//     then four bits of hash.  With hundreds of offsets hardly two masks are equal; what neighbours in the
//     order share is the side on which their neighbours lie.  The weight puts the heaviest tiles at the
//     end, from which the convolution kernels start: a launch ends with its longest tile otherwise.
//     5 x 5 x 5 on 120 k voxels: 47 k (tile, offset) steps against 87 k in the order by count and hash, 46 k
//     without the weight, but forward 74.8 -> 66.1 us, backward-input 74.8 -> 65.8.
// Where the caller does not ask for more (coarse), one word and up to 2^20 positions have a key of 11 bits and
// one pass: exact up to two offsets, the bins above that dealt out by number of offsets, without the middle
// offset in a submanifold layer's table, which has it everywhere.  The chain is then masks, sums, pass, position:
// of a frame's tables (120 k and 447 k positions) the second pass was 12 + 16 us of 98, frame of 120 k voxels
// 239 -> 214.6 us, of 300 k forward and backward 616 -> 580.  (Tile, offset) steps against the key of 18 bits:
// 1.000 - 1.005 up to 324 k positions, 1.016 at 792 k of a stride-2 table, whose layer (128 -> 256 channels, forward
// and backward) is none the slower, 851 -> 847 us: rows of one bin stay in their order, neighbours near
// each other.  At 1 M positions of a submanifold layer it is 1.05 (at 300 k 1.001), and its passes take 791 us for
// 767: those have two radix passes above 2^19 positions.  The lines, us with one pass / two, bf16, geometry and then forward
// of a layer of 64 channels: submanifold, 400 k positions 121 / 137 and 30.4 / 30.3, 500 k 149 / 167 and 36.6 / 36.7, but 600 k
// 185 / 204 and 47.2 / 45.9, 900 k 258 / 277 and 71.3 / 69.6 (128 channels 185 / 182); stride 2, 541 k sites 113 / 135 and 35.5 /
// 35.4, 798 k 143 / 165 and 49.5 / 49.4, 922 k 161 / 187 and 56.1 / 56.8; the sums of more than 2^20 positions do not fit a
// trip of the scan.
// Chain of kernels: masks, keys and the digits' counts per block of 512 positions - sums of the counts over
// the blocks - two passes - position.  The first pass knows every chunk's place from the sums, the second
// looks back (ticket, flagged words); both rank by ballot and are stable.  (Instead of a kernel that clears,
// counts by device-wide atomics and look-backs in both passes.  The first pass can then be cut as finely as
// the device is wide: 1024 positions per workgroup, over 447 k positions of two tables 21.2 -> 7.1 us, over
// 120 k 13.2 -> 4.8; the second 21.2 -> 15.2, 13.2 -> 11.4; the sums 5 us for 3 - 4 of clearing.  Each pass
// adding up the counts by itself instead took 6 us back.)  The mask kernel reads the tables at 4.4 TB/s (1024
// positions per workgroup 35.7 for 27.2 us at 1.1 M).  The position kernel writes them again; what it fetches by
// row is little more than a word pair per position (51.5 -> 39.1 us at 1.1 M positions against a fetch of mask
// and entries).
// Measured (kernel times): the tables of a frame of 120 k voxels - submanifold and stride 2, 326 k output
// sites - 98 us in ten launches, in eight with one pass 71; with masks by atomics, a sort each and a
// gather of every entry it was 305 us in 27.
#include <algorithm>
#include <cstring>

#include "launch.h"
#include "lds_dma.h"

namespace cummhip {

namespace {

constexpr int kDigit = 9, kDigitBins = 1 << kDigit;      // 512
constexpr int kKeyBits = 2 * kDigit;
constexpr int kPassThreads = 1024, kPassWaves = kPassThreads / 64;
constexpr int kMaskBatch = 16;                            // table rows whose loads are in flight together
constexpr int kBlock = 512;                               // positions per workgroup of the masks kernel
constexpr int kLowBlocks = kPassThreads / kBlock;         // blocks per chunk of the first pass
constexpr uint32_t kNowhere = 0xF0000000u;                // past any matrix of counts (up to 2^31 + 2048 bytes: 2^20 rows and the sums)
constexpr int kExact = 5;                                 // offsets up to which a one-word key is exact
constexpr uint32_t kAggregate = 1u << 30, kInclusive = 2u << 30, kCount = (1u << 30) - 1u;
constexpr int kSpins = 1 << 20;                           // (about a second)

// the order of one pass
constexpr int kOnceDigit = 11, kOnceBins = 1 << kOnceDigit;      // 2048
constexpr int kOnceExact = 2;                             // offsets up to which its key is exact
constexpr int kOnceChunk = 1024;                          // positions per workgroup of the pass
constexpr int kOnceMost = 1 << 20;                        // positions up to which it is taken,
constexpr int kOnceMostReversed = 1 << 19;                // ... of a submanifold layer's table

struct Side {
  const int32_t *indices;      // [kv, n]
  int32_t n, chunks;
  uint32_t *raw;               // [n, words] masks by row; one word: [n, 2] mask and lead
  uint32_t *keys;              // [n]; one pass: [n] of 16 bits
  int32_t *tmp_rows;           // [n] after the first pass
  uint16_t *tmp_high;          // [n]
  uint32_t *counts[2];         // per pass [rows + 1][kDigitBins]: keys per digit and block of positions, then
                               // the same of the blocks before it, and at the end of all
  int32_t rows;                // blocks
  uint16_t *once_counts;       // one pass: [rows][kOnceBins] keys per bin and block of positions
  uint32_t *once_before;       // [chunks + 1][kOnceBins] keys of the chunks before; at the end of all
  uint32_t *state;             // [chunks][kDigitBins] look-back words of the second pass
  uint32_t *ticket;
  uint32_t *sorted;            // [n, words]
  int32_t *order;              // [n]
  int32_t *by_pos, *by_pos_rev;   // [kv, n]; the second, with its offsets reversed, may be NULL
  int32_t *hint_slot;          // or NULL
};

struct OrderParams {
  Side side[2];
  int32_t sides, kv, words;
  int32_t rows_per_chunk;
  int32_t sparse;              // tables by position: only runs of 128 positions with a pair
  int32_t *give_ups;
  uint32_t base[kExact + 2];   // first key of the words with c offsets; [kExact + 1]: of those with more
  uint32_t share;              // keys per number of offsets above kExact
  float per_word[33];          // share / number of words with c offsets, c > kExact
  // one pass: is the middle offset left out of the key (a submanifold layer's masks all have it), the first
  // key of the words with c (other) offsets, and for c > kOnceExact how many keys they have in all and per word
  int32_t once_drop;
  uint32_t once_base[34];
  float once_per_word[33];
  // planes[i]: the offsets of outer plane i (several words)
  uint32_t planes[12][4];
  uint32_t filter;
};

// rank of a word among those with as many bits, ascending value: sum of C(position of the i-th bit, i).  Up to
// kExact bits
__device__ __forceinline__ uint32_t word_rank(uint32_t rest) {
  uint32_t rank = 0;
#pragma unroll
  for (int i = 1; i <= kExact; ++i) {
    if (rest == 0u) break;
    const uint32_t b = (uint32_t)__builtin_ctz(rest);
    rest &= rest - 1u;
    uint32_t v = b;                                    // C(b, i)
    if (i >= 2) v = v * (b - 1u) / 2u;
    if (i >= 3) v = v * (b - 2u) / 3u;
    if (i >= 4) v = v * (b - 3u) / 4u;
    if (i >= 5) v = v * (b - 4u) / 5u;
    rank += b >= (uint32_t)i ? v : 0u;
  }
  return rank;
}
// any number of bits: in floating point (its leading digits are all that is kept)
__device__ __forceinline__ float word_rank_f32(uint32_t m) {
  float rank = 0.0f;
  uint32_t rest = m;
  int i = 1;
  while (rest != 0u) {
    const float b = (float)__builtin_ctz(rest);
    rest &= rest - 1u;
    float v = b >= (float)i ? 1.0f : 0.0f;
    for (int t = 0; t < i; ++t) v *= (b - (float)t) / (float)(t + 1);
    rank += v;
    ++i;
  }
  return rank;
}

__device__ __forceinline__ uint32_t word_key(const OrderParams &p, uint32_t m) {
  const int c = __builtin_popcount(m);
  if (c <= kExact) return p.base[c] + word_rank(m);
  const uint32_t at = (uint32_t)(word_rank_f32(m) * p.per_word[c]);
  return p.base[kExact + 1] + (uint32_t)(c - kExact - 1) * p.share + (at < p.share ? at : p.share - 1u);
}

// the key of the one pass
__device__ __forceinline__ uint32_t once_key(const OrderParams &p, uint32_t m) {
  const int middle = p.kv / 2;
  if (p.once_drop) m = (m & ((1u << middle) - 1u)) | ((m >> middle >> 1) << middle);
  const int c = __builtin_popcount(m);
  if (c <= kOnceExact) return p.once_base[c] + word_rank(m);
  const float rank = c <= kExact ? (float)word_rank(m) : word_rank_f32(m);
  const uint32_t at = p.once_base[c] + (uint32_t)(rank * p.once_per_word[c]), last = p.once_base[c + 1] - 1u;
  return at < last ? at : last;
}

__device__ __forceinline__ uint32_t words_key(const OrderParams &p, const uint32_t *w) {
  uint32_t planes = 0u, h = 0u;
#pragma unroll
  for (int i = 0; i < 12; ++i) {
    const uint32_t any = (w[0] & p.planes[i][0]) | (w[1] & p.planes[i][1]) | (w[2] & p.planes[i][2]) | (w[3] & p.planes[i][3]);
    planes |= any ? 1u << i : 0u;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) h = (h ^ w[i]) * 0x9E3779B1u;
  // the place of `planes` in the Gray code
  planes ^= planes >> 1;
  planes ^= planes >> 2;
  planes ^= planes >> 4;
  planes ^= planes >> 8;
  const int c = __builtin_popcount(w[0]) + __builtin_popcount(w[1]) + __builtin_popcount(w[2]) + __builtin_popcount(w[3]);
  const uint32_t weight = (c > 2 ? 1u : 0u) + (c > 4 ? 1u : 0u) + (c > 8 ? 1u : 0u);
  return (weight << (kKeyBits - 2)) | (planes << (kKeyBits - 14)) | (h >> (32 - (kKeyBits - 14)));
}

// What lies beside a one-word mask: is the row's entry for the middle offset the row itself (as
// everywhere in a submanifold table), and the entry of its lowest other offset.
constexpr uint32_t kSelf = 0x80000000u, kLeadEntry = 0x7FFFFFFFu;

// side and index inside it of a workgroup, when side 0 has `first` workgroups
__device__ __forceinline__ int side_of(int first, int *block) {
  const int s = *block >= first ? 1 : 0;
  *block -= s ? first : 0;
  return s;
}

// One position per lane: its mask out of the table (every row read coalesced, kv independent loads), its
// key, the entry of its lowest offset, and how many of the block's keys have which digit, for both
// passes.  A block's counts are a row of its own, so that nothing has to be zero before.  (Eight positions
// per lane, one after the other: fewer rows, but 55 us for 27 at 1.1 M positions.)
template <int WORDS, bool ONCE = false>
__global__ __launch_bounds__(kBlock) void order_masks_kernel(const OrderParams p) {
  constexpr int kCounts = ONCE ? kOnceBins : 2 * kDigitBins;
  __shared__ uint32_t hist[kCounts];
  const int t = threadIdx.x, lane = t & 63;
  int block = blockIdx.x;
  const Side &d = p.side[side_of(p.side[0].rows, &block)];
  static_assert(kBlock == kDigitBins && kOnceBins == 4 * kBlock, "a thread per digit, or per four");
#pragma unroll
  for (int i = 0; i < kCounts / kBlock; ++i) hist[i * kBlock + t] = 0u;
  if (!ONCE && block % p.rows_per_chunk == 0) d.state[(size_t)(block / p.rows_per_chunk) * kDigitBins + t] = 0u;
  if (block == 0) {
    if (!ONCE && t == 0) *d.ticket = 0u;
    if (t < 8 && d.hint_slot != nullptr)   // names no array yet; the two counts start at "everything" / "nothing"
      d.hint_slot[t] = t == 4 ? (d.n / 128) * 128 : (t == 5 ? ((d.n + 63) / 64) * 64 : 0);
  }
  __syncthreads();
  // (kv * n entries are below 2^31 bytes: the row of the table is a scalar offset)
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t *>(d.indices), 0,
                                                                      (int)((uint32_t)p.kv * (uint32_t)d.n * 4u), 0x00020000);
  const int o = block * kBlock + t;
  const bool on = o < d.n;
  uint32_t w[4] = {0u, 0u, 0u, 0u};
  uint32_t lead = 0u;
  bool self = false;
  const uint32_t at = (uint32_t)(on ? o : 0) * 4u;
#pragma unroll
  for (int q = 0; q < WORDS; ++q) {
    const int hi = p.kv - 32 * q < 32 ? p.kv - 32 * q : 32;
    for (int b0 = ((hi - 1) / kMaskBatch) * kMaskBatch; b0 >= 0; b0 -= kMaskBatch) {      // (the lowest offset last)
      int v[kMaskBatch];
#pragma unroll
      for (int u = 0; u < kMaskBatch; ++u) v[u] = __builtin_amdgcn_raw_buffer_load_b32(rs, at, (32 * q + (b0 + u < hi ? b0 + u : 0)) * d.n * 4, 0);
#pragma unroll
      for (int u = kMaskBatch - 1; u >= 0; --u) {
        const bool has = b0 + u < hi && v[u] >= 0;
        w[q] |= has ? 1u << (b0 + u) : 0u;
        if constexpr (WORDS == 1) {
          if (b0 + u == p.kv / 2) self = v[u] == o;
          else lead = has ? (uint32_t)v[u] : lead;
        }
      }
    }
  }
  const uint32_t key = ONCE ? once_key(p, w[0]) : (WORDS == 1 ? word_key(p, w[0]) : words_key(p, w));
  if (on) {
    if constexpr (WORDS == 1) {
      reinterpret_cast<uint2 *>(d.raw)[o] = uint2{w[0], self ? lead | kSelf : lead};
    } else {
#pragma unroll
      for (int q = 0; q < WORDS; ++q) d.raw[(int64_t)o * WORDS + q] = w[q];
    }
    if constexpr (ONCE) reinterpret_cast<uint16_t *>(d.keys)[o] = (uint16_t)key;
    else d.keys[o] = key;
  }
  // most waves of a sparse cloud hold one key: one add for all lanes
  const unsigned long long live = __ballot(on);
  if (live != 0ull) {
    const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)key);
    if (__ballot(on && key == first) == live) {
      if constexpr (ONCE) {
        if (lane == 0) atomicAdd(&hist[first], (uint32_t)__popcll(live));
      } else if (lane < 2) {
        atomicAdd(&hist[lane * kDigitBins + ((first >> (lane * kDigit)) & (kDigitBins - 1))], (uint32_t)__popcll(live));
      }
    } else if (on) {
      if constexpr (ONCE) {
        atomicAdd(&hist[key], 1u);
      } else {
        atomicAdd(&hist[key & (kDigitBins - 1)], 1u);
        atomicAdd(&hist[kDigitBins + (key >> kDigit)], 1u);
      }
    }
  }
  __syncthreads();
  if constexpr (ONCE) {
    const v4i c = reinterpret_cast<const v4i *>(hist)[t];
    reinterpret_cast<uint2 *>(d.once_counts + (size_t)block * kOnceBins)[t] = uint2{(uint32_t)(c.x | c.y << 16), (uint32_t)(c.z | c.w << 16)};
  } else {
    d.counts[0][(size_t)block * kDigitBins + t] = hist[t];
    d.counts[1][(size_t)block * kDigitBins + t] = hist[kDigitBins + t];
  }
}

// blocks per run of the scan: whole chunks of the first pass
__host__ __device__ constexpr int scan_run(int rows) { return (rows + 64 * kLowBlocks - 1) / (64 * kLowBlocks) * kLowBlocks; }

// Counts -> totals behind the last block and, for the first pass, the sums over the blocks before every chunk
// (the second pass wants the totals alone).  A workgroup takes 16 digits of one pass and table in 64 runs of
// blocks, ROWS blocks of each at a time.  (Rows past a run's end are fetched outside the matrix: as conditional
// loads each waited for the one before, 18 us for 5.  They cost their issue all the same: ROWS is the least of
// three that takes a run in one trip, 48 where none does, and of the sums only those that are read are written:
// with 48 and all of them 120 k positions 7.0 us for 4.7, 447 k of two tables 8.6 for 5.3, 1.4 M 12.7 for 8.6.)
template <int ROWS>
__global__ __launch_bounds__(1024) void order_scan_kernel(const OrderParams p) {
  __shared__ uint32_t run_sum[64][16];
  static_assert(ROWS % kLowBlocks == 0, "a chunk of the first pass begins at the same row of every trip");
  const int digit = threadIdx.x & 15, run = threadIdx.x >> 4;
  const bool low = (blockIdx.y & 1) == 0;
  const Side &d = p.side[blockIdx.y >> 1];
  const __amdgpu_buffer_rsrc_t rs =
      __builtin_amdgcn_make_buffer_rsrc(low ? d.counts[0] : d.counts[1], 0, (int)((uint32_t)(d.rows + 1) * (kDigitBins * 4u)), 0x00020000);
  const uint32_t col = (uint32_t)(blockIdx.x * 16 + digit) * 4u;
  const int per = scan_run(d.rows), r0 = run * per, r1 = r0 + per < d.rows ? r0 + per : d.rows;
  const auto at = [&](int t) -> uint32_t { return t < per && r0 + t < r1 ? (uint32_t)(r0 + t) * (kDigitBins * 4u) + col : kNowhere; };
  uint32_t v[ROWS], sum = 0;
  for (int t0 = 0; t0 < per; t0 += ROWS) {
#pragma unroll
    for (int u = 0; u < ROWS; ++u) v[u] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, at(t0 + u), 0, 0);
#pragma unroll
    for (int u = 0; u < ROWS; ++u) sum += v[u];
  }
  run_sum[run][digit] = sum;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll 16
  for (int i = 0; i < 64; ++i) {
    const uint32_t x = run_sum[i][digit];
    before += i < run ? x : 0u;
    all += x;
  }
  if (run == 0) __builtin_amdgcn_raw_buffer_store_b32((int)all, rs, (uint32_t)d.rows * (kDigitBins * 4u) + col, 0, 0);
  if (!low) return;
  for (int t0 = 0; t0 < per; t0 += ROWS) {
    if (per > ROWS) {
#pragma unroll
      for (int u = 0; u < ROWS; ++u) v[u] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, at(t0 + u), 0, 0);
    }
#pragma unroll
    for (int u = 0; u < ROWS; ++u) {
      if (u % kLowBlocks == 0) __builtin_amdgcn_raw_buffer_store_b32((int)before, rs, at(t0 + u), 0, 0);
      before += v[u];
    }
  }
}

// The same for the one pass: 32 bins of a table per workgroup, two per thread (16-bit counts of blocks), the
// sums before every chunk and the totals as 32 bits.  ROWS takes a run in one trip.  The sums over the 64 runs are
// a wave's prefix sum per pair of bins (every thread adding up all 64 by itself read 512 KB of LDS per workgroup:
// 7.5 -> 4.8 us for the tables of 447 k positions, 9.6 -> 8.0 for 1.1 M).
template <int ROWS>
__global__ __launch_bounds__(1024) void order_once_scan_kernel(const OrderParams p) {
  __shared__ uint2 run_sum[64][17];
  static_assert(ROWS % kLowBlocks == 0 && kLowBlocks * kBlock == kOnceChunk, "two blocks of a run are a chunk");
  const int pair = threadIdx.x & 15, run = threadIdx.x >> 4;
  const Side &d = p.side[blockIdx.y];
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(d.once_counts, 0, (int)((uint32_t)d.rows * (kOnceBins * 2u)), 0x00020000);
  const uint32_t col = (uint32_t)(blockIdx.x * 16 + pair);
  const int per = scan_run(d.rows), r0 = run * per, r1 = r0 + per < d.rows ? r0 + per : d.rows;
  uint32_t v[ROWS];
  uint2 sum = {0u, 0u};
#pragma unroll
  for (int u = 0; u < ROWS; ++u)      // (past the run's end: outside the matrix)
    v[u] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, u < per && r0 + u < r1 ? (uint32_t)(r0 + u) * (kOnceBins * 2u) + col * 4u : kNowhere, 0, 0);
#pragma unroll
  for (int u = 0; u < ROWS; ++u) {
    sum.x += v[u] & 0xFFFFu;
    sum.y += v[u] >> 16;
  }
  run_sum[run][pair] = sum;
  __syncthreads();
  uint2 *to = reinterpret_cast<uint2 *>(d.once_before) + blockIdx.x * 16;
  {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;      // (a run per lane, a pair of bins per wave)
    const uint2 x = run_sum[lane][wave];
    const uint2 upto = {(uint32_t)wave_prefix_sum_dpp((int)x.x), (uint32_t)wave_prefix_sum_dpp((int)x.y)};
    if (lane == 63) to[(size_t)d.chunks * (kOnceBins / 2) + wave] = upto;
    run_sum[lane][wave] = uint2{upto.x - x.x, upto.y - x.y};
  }
  __syncthreads();
  uint2 before = run_sum[run][pair];
  to += pair;
#pragma unroll
  for (int u = 0; u < ROWS; ++u) {
    if (u % kLowBlocks == 0 && u < per && r0 + u < r1) to[(size_t)((r0 + u) / kLowBlocks) * (kOnceBins / 2)] = before;
    before.x += v[u] & 0xFFFFu;
    before.y += v[u] >> 16;
  }
}

// The one pass: a position per lane, its place = keys below its own + equal ones in the chunks before + in the
// waves before + in the lanes before.  A wave's lanes of one key are found by ballot; their number, one byte,
// goes to the key's 16 bytes, one for each wave, of which a lane adds up those before its own in four
// instructions (a histogram of words per wave, added up bin by bin, would be 128 KB and 32 reads per thread).
__global__ __launch_bounds__(kOnceChunk) void order_once_pass_kernel(const OrderParams p) {
  constexpr int kWaves = kOnceChunk / 64;
  static_assert(kWaves == 16 && kOnceBins == 2 * kOnceChunk, "sixteen bytes per bin, two bins per thread");
  __shared__ v4i wave_counts[kOnceBins];
  __shared__ uint32_t first[kOnceBins];
  __shared__ uint32_t wave_sum[kWaves];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  int chunk = blockIdx.x;
  const Side &d = p.side[side_of(p.side[0].chunks, &chunk)];
  const int pos = chunk * kOnceChunk + t;
  const bool on = pos < d.n;
  const uint32_t key = reinterpret_cast<const uint16_t *>(d.keys)[on ? pos : d.n - 1];
  const uint2 total = reinterpret_cast<const uint2 *>(d.once_before + (size_t)d.chunks * kOnceBins)[t];
  wave_counts[t] = wave_counts[t + kOnceChunk] = v4i{0, 0, 0, 0};
  const uint32_t before_chunk = d.once_before[(size_t)chunk * kOnceBins + key];
  // first place of each bin: exclusive prefix over the totals
  uint32_t incl = total.x + total.y;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t up = (uint32_t)__shfl_up((int)incl, off, 64);
    if (lane >= off) incl += up;
  }
  if (lane == 63) wave_sum[wave] = incl;
  unsigned long long peers = __ballot(on);
#pragma unroll
  for (int b = 0; b < kOnceDigit; ++b) {
    const unsigned long long has = __ballot((key >> b) & 1u);
    peers &= ((key >> b) & 1u) ? has : ~has;
  }
  const uint32_t rank = (uint32_t)__popcll(peers & ((1ull << lane) - 1ull));
  __syncthreads();
  if (on && rank == 0u) reinterpret_cast<uint8_t *>(&wave_counts[key])[wave] = (uint8_t)__popcll(peers);
  uint32_t base = incl - total.x - total.y;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) base += w < wave ? wave_sum[w] : 0u;
  reinterpret_cast<uint2 *>(first)[t] = uint2{base, base + total.x};
  __syncthreads();
  if (!on) return;
  uint32_t dst = first[key] + before_chunk + rank;
  const v4i c = wave_counts[key];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int bytes = wave - 4 * i;      // waves of these four before this one
    const uint32_t those = bytes >= 4 ? ~0u : (bytes > 0 ? (1u << (8 * bytes)) - 1u : 0u);
    dst = __builtin_amdgcn_sad_u8((uint32_t)c[i] & those, 0u, dst);
  }
  d.order[dst] = pos;
}

// One pass over one digit (LOW: the low one, rows in ascending order to tmp; else the high one, tmp to
// order).  A workgroup ranks the keys of a chunk per digit in position order and scatters them.  Where a
// chunk's keys of a digit begin: in the first pass the blocks' counts say it; in the second, whose chunks are
// made by the first, a workgroup takes the next chunk by ticket (its predecessors have then started),
// publishes its counts and adds up those of the chunks before it.  Words carry flag and value: relaxed
// device-scope accesses do.
template <int ITEMS, bool LOW>
__global__ __launch_bounds__(kPassThreads) void order_pass_kernel(const OrderParams p) {
  constexpr int kChunk = kPassThreads * ITEMS;
  __shared__ uint32_t wave_hist[kPassWaves][kDigitBins];
  __shared__ uint32_t bin_base[kDigitBins];
  __shared__ uint32_t wave_sum[8];
  __shared__ int chunk_of_block;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  int block = blockIdx.x;
  const auto chunks_of = [](const Side &side) { return LOW ? (side.n + kChunk - 1) / kChunk : side.chunks; };
  const Side &d = p.side[side_of(chunks_of(p.side[0]), &block)];
  int chunk = block;
  if (!LOW && t == 0) chunk_of_block = (int)atomicAdd(d.ticket, 1u);
  for (int i = t; i < kPassWaves * kDigitBins; i += kPassThreads) (&wave_hist[0][0])[i] = 0u;
  // keys per bin of the whole input and (first pass) of the chunks before this one
  uint32_t total = 0, earlier = 0;
  if (t < kDigitBins) {
    const uint32_t *c = d.counts[LOW ? 0 : 1] + t;
    total = c[(size_t)d.rows * kDigitBins];
    if constexpr (LOW) earlier = c[(size_t)(block * kLowBlocks) * kDigitBins];
  }
  __syncthreads();
  if constexpr (!LOW) chunk = chunk_of_block;
  if (chunk >= chunks_of(d)) return;      // (never: one workgroup per chunk)
  // wave w owns positions [base, base + 64 ITEMS), item u of lane l is position base + 64 u + l
  const int64_t base = (int64_t)chunk * kChunk + (int64_t)wave * (64 * ITEMS);
  uint32_t digit[ITEMS], high[ITEMS];
  int32_t row[ITEMS];
  uint32_t rank[ITEMS];
#pragma unroll
  for (int u = 0; u < ITEMS; ++u) {
    const int64_t pos = base + u * 64 + lane;
    const int64_t at = pos < d.n ? pos : d.n - 1;
    if constexpr (LOW) {
      const uint32_t key = d.keys[at];
      digit[u] = key & (kDigitBins - 1);
      high[u] = key >> kDigit;
      row[u] = (int32_t)pos;
    } else {
      digit[u] = d.tmp_high[at];
      row[u] = d.tmp_rows[at];
    }
  }
  // first place of each bin: exclusive prefix over the bins
  uint32_t incl = total;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t up = (uint32_t)__shfl_up((int)incl, off, 64);
    if (lane >= off) incl += up;
  }
  if (t < kDigitBins && lane == 63) wave_sum[wave] = incl;
#pragma unroll
  for (int u = 0; u < ITEMS; ++u) {
    const bool valid = base + u * 64 + lane < d.n;
    unsigned long long peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < kDigit; ++b) {
      const unsigned long long has = __ballot((digit[u] >> b) & 1u);
      peers &= ((digit[u] >> b) & 1u) ? has : ~has;
    }
    const uint32_t before = (uint32_t)__popcll(peers & ((1ull << lane) - 1ull));
    uint32_t prev = 0;
    if (valid) prev = wave_hist[wave][digit[u]];
    __builtin_amdgcn_wave_barrier();
    if (valid && before == 0) wave_hist[wave][digit[u]] = prev + (uint32_t)__popcll(peers);
    __builtin_amdgcn_wave_barrier();
    rank[u] = prev + before;
  }
  __syncthreads();
  if (t < kDigitBins) {
    uint32_t first = incl - total;
#pragma unroll
    for (int w = 0; w < 8; ++w) first += w < wave ? wave_sum[w] : 0u;
    uint32_t count = 0;
#pragma unroll
    for (int w = 0; w < kPassWaves; ++w) {
      const uint32_t c = wave_hist[w][t];
      wave_hist[w][t] = count;
      count += c;
    }
    uint32_t before = LOW ? earlier : 0u;
    uint32_t *state = d.state;
    if (!LOW)
      __hip_atomic_store(&state[(size_t)chunk * kDigitBins + t], (chunk == 0 ? kInclusive : kAggregate) | count, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    if (!LOW && chunk > 0) {
      constexpr int kLook = 32;      // words per round trip
      bool done = false, gave_up = false;
      int j = chunk - 1, spins = 0;
      while (!done && !gave_up) {
        uint32_t sw[kLook];
#pragma unroll
        for (int i = 0; i < kLook; ++i)
          sw[i] = j - i >= 0 ? __hip_atomic_load(&state[(size_t)(j - i) * kDigitBins + t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                             : kInclusive;
        int taken = 0;
#pragma unroll
        for (int i = 0; i < kLook; ++i) {
          if (!done && taken == i) {
            const uint32_t flag = sw[i] >> 30;
            if (flag != 0u) {
              before += sw[i] & kCount;
              ++taken;
              done = flag == 2u;
            }
          }
        }
        j -= taken;
        if (!done && taken == 0) {
          if (++spins > kSpins) gave_up = true;
          __builtin_amdgcn_s_sleep(1);
        }
      }
      if (gave_up && p.give_ups != nullptr) atomicAdd(p.give_ups, 1);
      __hip_atomic_store(&state[(size_t)chunk * kDigitBins + t], kInclusive | (before + count), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    }
    bin_base[t] = first + before;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < ITEMS; ++u) {
    if (base + u * 64 + lane < d.n) {
      const uint32_t dst = bin_base[digit[u]] + wave_hist[wave][digit[u]] + rank[u];
      if (dst < (uint32_t)d.n) {      // (always, unless a look-back gave up)
        if constexpr (LOW) {
          d.tmp_rows[dst] = row[u];
          d.tmp_high[dst] = (uint16_t)high[u];
        } else {
          d.order[dst] = row[u];
        }
      }
    }
  }
}

// 256 positions and the offsets of one mask word per workgroup: masks, table(s) by position, and (one
// word) the counts of the launch hints - as sort_finish_kernel, whose remarks on give-ups hold here too:
// the identity order replaces one that cannot be trusted.  A fetch by row costs a sector for four
// bytes: of one-word masks the lowest offset's entry comes with the mask, the middle one's is mostly
// the row itself, and of the others those are fetched that some lane of the wave has (the positions are
// sorted by their masks: few).  (Mask and entry carried through both passes instead: 14 us less here
// at 1.1 M positions, 20 us more there.)
// sparse: of the 27 entries of a position one or two are pairs, and the kernels look at a table only where a tile of
// 64 or 128 positions has the offset; the rest of it - 86 MB for 798 k positions - is not written: 38.4 -> 25.0 us at
// 1.1 M positions, 17.4 -> 12.2 at 447 k, and the layers after it find more in the caches (stride 2, 32 -> 64 channels
// forward 57 -> 50 us).
constexpr int kLight = 3, kHeavy = 10;
template <int WORDS>
__global__ __launch_bounds__(256) void order_position_kernel(const OrderParams p) {
  __shared__ uint32_t half_or[4];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  int block = blockIdx.x;
  const Side &d = p.side[side_of((p.side[0].n + 255) / 256, &block)];
  const int pos = block * 256 + t;
  const bool on = pos < d.n;
  const bool broken = p.give_ups != nullptr && __hip_atomic_load(p.give_ups, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
  const int row = on ? (broken ? pos : d.order[pos]) : -1;
  const int word = blockIdx.y, k0 = 32 * word;
  uint32_t mine = 0u, lead = 0u;
  if (row >= 0 && row < d.n) {
    if constexpr (WORDS == 1) {
      const uint2 both = reinterpret_cast<const uint2 *>(d.raw)[row];
      mine = both.x;
      lead = both.y;
    } else {
      mine = d.raw[(int64_t)row * WORDS + word];
    }
  }
  const int middle = p.kv / 2;
  const bool self = (lead & kSelf) != 0u;
  const int lead_at = WORDS == 1 ? __ffs((int)(mine & ~(1u << middle))) - 1 : -1;
  uint32_t fetch = mine;
  if (lead_at >= 0) fetch &= ~(1u << lead_at);
  if (self) fetch &= ~(1u << middle);
  const uint32_t fetch_or = wave_or_dpp(fetch);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t *>(d.indices), 0,
                                                                      (int)((uint32_t)p.kv * (uint32_t)d.n * 4u), 0x00020000);
  int v[32];
#pragma unroll
  for (int u = 0; u < 32; ++u) {
    v[u] = u == lead_at ? (int)(lead & kLeadEntry) : (self && u == middle ? row : -1);
    if ((fetch_or >> u) & 1u) {      // (a clear bit is fetched outside the table: no memory is touched)
      const int e = __builtin_amdgcn_raw_buffer_load_b32(
          rs, (fetch >> u) & 1u ? (uint32_t)((k0 + u) * d.n + row) * 4u : 0x80000000u, 0, 0);
      v[u] = (fetch >> u) & 1u ? e : v[u];
    }
  }
  const uint32_t o = wave_or_dpp(mine);
  if (lane == 0) half_or[wave] = o;
  __syncthreads();
  const uint32_t write = p.sparse ? (uint32_t)__builtin_amdgcn_readfirstlane((int)(half_or[wave & ~1] | half_or[wave | 1])) : ~0u;
  const int bytes = (int)((uint32_t)p.kv * (uint32_t)d.n * 4u);
  const __amdgpu_buffer_rsrc_t to = __builtin_amdgcn_make_buffer_rsrc(d.by_pos, 0, bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rev = __builtin_amdgcn_make_buffer_rsrc(d.by_pos_rev, 0, d.by_pos_rev ? bytes : 0, 0x00020000);
  if (on) {
#pragma unroll
    for (int u = 0; u < 32; ++u) {
      if (k0 + u >= p.kv) break;
      if (!((write >> u) & 1u)) continue;
      __builtin_amdgcn_raw_buffer_store_b32(v[u], to, (uint32_t)pos * 4u, (k0 + u) * d.n * 4, 0);
      if (d.by_pos_rev != nullptr) __builtin_amdgcn_raw_buffer_store_b32(v[u], rev, (uint32_t)pos * 4u, (p.kv - 1 - k0 - u) * d.n * 4, 0);
    }
    d.sorted[(int64_t)pos * WORDS + word] = mine;
    if (broken && word == 0) d.order[pos] = pos;
  }
  if (WORDS > 1 || blockIdx.y != 0 || d.hint_slot == nullptr) return;
  if (broken) {
    if (block == 0 && t < 8) d.hint_slot[t] = 0;
    return;
  }
  if (t < 2) {
    const int run = block * 2 + t;
    const int c0 = __builtin_popcount(half_or[2 * t]), c1 = __builtin_popcount(half_or[2 * t + 1]);
    if (run < d.n / 128 && (c0 > kLight || c1 > kLight)) atomicMin(&d.hint_slot[4], run * 128);
    if (c0 >= kHeavy || c1 >= kHeavy) atomicMin(&d.hint_slot[5], run * 128 + (c0 >= kHeavy ? 0 : 64));
  }
  if (block == 0 && t == 0) {
    const uint64_t a = (uint64_t)d.sorted;
    d.hint_slot[0] = (int32_t)(uint32_t)a;
    d.hint_slot[1] = (int32_t)(uint32_t)(a >> 32);
    d.hint_slot[2] = d.n;
    d.hint_slot[3] = (int32_t)p.filter;
    d.hint_slot[6] = 1;
  }
}

size_t up256(size_t x) { return (x + 255) & ~(size_t)255; }
// chunks of the second pass: 4096 positions up to 2^18 (few chunks: it is as long as one chunk's chain), 8192
// above (120 k positions: 11.4 us, with 1024 12.7, 8192 14.2; 1.1 M: 19.5 us, with 4096 22.8, 1024 43.1)
int pass_items(int n) { return n <= (1 << 18) ? 4 : 8; }
int mask_rows(int n) { return (int)(((int64_t)n + kBlock - 1) / kBlock); }

}  // namespace

size_t order_pairs_workspace_bytes(int n, int words, bool coarse) {
  const size_t nn = (size_t)(n > 0 ? n : 1);
  if (coarse && words == 1 && n <= kOnceMost) {
    const size_t rows = (size_t)mask_rows((int)nn), chunks = (nn + kOnceChunk - 1) / kOnceChunk;
    const size_t once = up256(8 * nn) + up256(2 * nn) + up256(2 * rows * kOnceBins) + up256(4 * (chunks + 1) * kOnceBins);
    return std::max(once, order_pairs_workspace_bytes(n, words, false));      // (the other table may be larger)
  }
  const size_t chunks = (nn + 4095) / 4096;
  return up256(4 * nn * (words == 1 ? 2 : words)) + 2 * up256(4 * nn) + up256(2 * nn) + 2 * up256(4 * ((size_t)mask_rows((int)nn) + 1) * kDigitBins) +
         up256(4 * chunks * kDigitBins) + 256;
}

// Keys of the one pass: exact up to kOnceExact offsets, and what is left of the bins dealt out to the larger
// numbers of offsets, 0.6 of the rest to each (a cloud's masks thin out at about that rate, and at least one).
static void once_keys(OrderParams &p) {
  const int bits = p.kv - p.once_drop;
  double choose = 1.0;
  uint32_t next = 0;
  for (int c = 0; c <= bits; ++c) {
    p.once_base[c] = next;
    uint32_t keys = (uint32_t)choose;
    if (c > kOnceExact) {
      const uint32_t left = (uint32_t)kOnceBins - next, others = (uint32_t)(bits - c);
      keys = c == bits ? 1u : (uint32_t)std::min({choose, 0.6 * left, (double)(left - others)});
      if (keys == 0u) keys = 1u;
      p.once_per_word[c] = (float)((double)keys / choose);
    }
    next += keys;
    choose = choose * (bits - c) / (c + 1);
  }
  p.once_base[bits + 1] = next;
}

static hipError_t launch_order_once(OrderParams &p, hipStream_t s) {
  int rows = 0, chunks = 0, blocks = 0, run = 0;
  for (int i = 0; i < p.sides; ++i) {
    rows += p.side[i].rows;
    chunks += p.side[i].chunks;
    blocks += (p.side[i].n + 255) / 256;
    run = std::max(run, scan_run(p.side[i].rows));
  }
  hipLaunchKernelGGL((order_masks_kernel<1, true>), dim3(rows), dim3(kBlock), 0, s, p);
  const dim3 scan_grid(kOnceBins / 32, p.sides);
  static_assert(kOnceMost / kBlock <= 64 * 32, "a run fits the largest trip");
  if (run <= 8) hipLaunchKernelGGL(order_once_scan_kernel<8>, scan_grid, dim3(1024), 0, s, p);
  else if (run <= 16) hipLaunchKernelGGL(order_once_scan_kernel<16>, scan_grid, dim3(1024), 0, s, p);
  else hipLaunchKernelGGL(order_once_scan_kernel<32>, scan_grid, dim3(1024), 0, s, p);
  hipLaunchKernelGGL(order_once_pass_kernel, dim3(chunks), dim3(kOnceChunk), 0, s, p);
  hipLaunchKernelGGL(order_position_kernel<1>, dim3(blocks), dim3(256), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_order_pairs(const OrderPairsSide *sides, int n_sides, int kv, const int32_t *ksize, void *workspace,
                              int32_t *give_ups, bool coarse, hipStream_t s) {
  OrderParams p;
  std::memset(&p, 0, sizeof(p));
  p.kv = kv; p.words = (kv + 31) / 32; p.give_ups = give_ups; p.sparse = coarse;
  p.filter = kv < 32 ? (1u << kv) - 1u : 0xFFFFFFFFu;
  char *at = reinterpret_cast<char *>(workspace);
  auto take = [&](size_t bytes) { char *q = at; at += up256(bytes); return q; };
  int most = 0;
  for (int i = 0; i < n_sides; ++i)
    if (sides[i].n > 0 && sides[i].n > most) most = sides[i].n;
  bool once = coarse && p.words == 1;
  for (int i = 0; i < n_sides; ++i) once = once && sides[i].n <= (sides[i].by_pos_rev != nullptr ? kOnceMostReversed : kOnceMost);
  const int items = pass_items(most), chunk = once ? kOnceChunk : kPassThreads * items;
  p.rows_per_chunk = chunk / kBlock;
  for (int i = 0; i < n_sides; ++i) {
    if (sides[i].n <= 0) continue;
    Side &d = p.side[p.sides++];
    const size_t n = (size_t)sides[i].n;
    d.indices = sides[i].indices; d.n = sides[i].n; d.chunks = (int)((n + chunk - 1) / chunk);
    d.sorted = sides[i].sorted; d.order = sides[i].order; d.by_pos = sides[i].by_pos; d.by_pos_rev = sides[i].by_pos_rev;
    d.hint_slot = p.words == 1 ? sides[i].hint_slot : nullptr;
    char *const begin = at;
    d.raw = reinterpret_cast<uint32_t *>(take(4 * n * (p.words == 1 ? 2 : p.words)));
    d.rows = mask_rows(d.n);
    if (once) {
      d.keys = reinterpret_cast<uint32_t *>(take(2 * n));
      d.once_counts = reinterpret_cast<uint16_t *>(take(2 * (size_t)d.rows * kOnceBins));
      d.once_before = reinterpret_cast<uint32_t *>(take(4 * ((size_t)d.chunks + 1) * kOnceBins));
      if (d.by_pos_rev != nullptr) p.once_drop = 1;      // (the table of a submanifold layer)
      at = begin + order_pairs_workspace_bytes(d.n, p.words, coarse);
      continue;
    }
    d.keys = reinterpret_cast<uint32_t *>(take(4 * n));
    d.tmp_rows = reinterpret_cast<int32_t *>(take(4 * n));
    d.tmp_high = reinterpret_cast<uint16_t *>(take(2 * n));
    for (uint32_t *&c : d.counts) c = reinterpret_cast<uint32_t *>(take(4 * ((size_t)d.rows + 1) * kDigitBins));
    d.state = reinterpret_cast<uint32_t *>(take(4 * (size_t)d.chunks * kDigitBins));
    d.ticket = reinterpret_cast<uint32_t *>(take(256));
    at = begin + order_pairs_workspace_bytes(d.n, p.words, coarse);
  }
  if (p.sides == 0) return hipSuccess;
  if (once) {
    p.give_ups = nullptr;      // (nothing looks back)
    p.once_drop = p.sides == 1 ? p.once_drop : 0;
    once_keys(p);
    return launch_order_once(p, s);
  }
  if (p.words == 1) {
    // words of kv bits with c offsets: C(kv, c)
    double choose = 1.0;
    uint32_t next = 0;
    for (int c = 0; c <= kv; ++c) {
      if (c <= kExact) {
        p.base[c] = next;
        next += (uint32_t)choose;
      }
      if (c == (kExact < kv ? kExact : kv)) {
        for (int e = c + 1; e <= kExact + 1; ++e) p.base[e] = next;
        p.share = kv > kExact ? ((1u << kKeyBits) - next) / (uint32_t)(kv - kExact) : 1u;
      }
      if (c > kExact) p.per_word[c] = (float)((double)p.share / choose);
      choose = choose * (kv - c) / (c + 1);
    }
  } else {
    for (int k = 0; k < kv; ++k) {
      const int i[3] = {k / (ksize[1] * ksize[2]), (k / ksize[2]) % ksize[1], k % ksize[2]};
      for (int a = 0; a < 3; ++a) {
        // the two lowest and the two highest planes of an axis (an axis of three has its outer ones only)
        const int last = ksize[a] - 1, mid = last / 2;
        const int plane = last == 0 || i[a] == mid ? -1 : (i[a] < mid ? (i[a] == 0 ? 0 : 1) : (i[a] == last ? 3 : 2));
        if (plane >= 0) p.planes[a * 4 + plane][k / 32] |= 1u << (k % 32);
      }
    }
  }
  int blocks = 0, chunks = 0;
  for (int i = 0; i < p.sides; ++i) {
    blocks += (p.side[i].n + 255) / 256;
    chunks += p.side[i].chunks;
  }
  int rows = 0;
  for (int i = 0; i < p.sides; ++i) rows += p.side[i].rows;
  switch (p.words) {
  case 1: hipLaunchKernelGGL(order_masks_kernel<1>, dim3(rows), dim3(kBlock), 0, s, p); break;
  case 2: hipLaunchKernelGGL(order_masks_kernel<2>, dim3(rows), dim3(kBlock), 0, s, p); break;
  case 3: hipLaunchKernelGGL(order_masks_kernel<3>, dim3(rows), dim3(kBlock), 0, s, p); break;
  default: hipLaunchKernelGGL(order_masks_kernel<4>, dim3(rows), dim3(kBlock), 0, s, p); break;
  }
  int run = 0;
  for (int i = 0; i < p.sides; ++i) run = scan_run(p.side[i].rows) > run ? scan_run(p.side[i].rows) : run;
  const dim3 scan_grid(kDigitBins / 16, 2 * p.sides);
  if (run <= 8) hipLaunchKernelGGL(order_scan_kernel<8>, scan_grid, dim3(1024), 0, s, p);
  else if (run <= 24) hipLaunchKernelGGL(order_scan_kernel<24>, scan_grid, dim3(1024), 0, s, p);
  else hipLaunchKernelGGL(order_scan_kernel<48>, scan_grid, dim3(1024), 0, s, p);
  int chunks_low = 0;
  for (int i = 0; i < p.sides; ++i) chunks_low += (p.side[i].n + kPassThreads - 1) / kPassThreads;
  hipLaunchKernelGGL((order_pass_kernel<1, true>), dim3(chunks_low), dim3(kPassThreads), 0, s, p);
  if (items == 4) hipLaunchKernelGGL((order_pass_kernel<4, false>), dim3(chunks), dim3(kPassThreads), 0, s, p);
  else hipLaunchKernelGGL((order_pass_kernel<8, false>), dim3(chunks), dim3(kPassThreads), 0, s, p);
  const dim3 grid(blocks, p.words);
  switch (p.words) {
  case 1: hipLaunchKernelGGL(order_position_kernel<1>, grid, dim3(256), 0, s, p); break;
  case 2: hipLaunchKernelGGL(order_position_kernel<2>, grid, dim3(256), 0, s, p); break;
  case 3: hipLaunchKernelGGL(order_position_kernel<3>, grid, dim3(256), 0, s, p); break;
  default: hipLaunchKernelGGL(order_position_kernel<4>, grid, dim3(256), 0, s, p); break;
  }
  return hipGetLastError();
}

}  // namespace cummhip
