// Dense GEMM,  D[m][n] = epilogue( sum_k Y[m][k] * X[n][k] ),  two-byte elements, every layout of the
// operands, any m, n and k (pieces of 8 elements along each operand's contiguous dimension), streamed
// through an LDS ring with direct-to-LDS buffer loads (see lds_dma.h and rowgemm_lds.h for the
// mechanism: hidden loads, hand-counted waits, fence-less barrier, XOR-permuted 16-byte chunks applied
// on the global side).
//
// What differs from tilegemm.h, and why:
//   * the wave tile (RBW x NBW blocks of 16 x 16), the step depth and the number of wave groups that share
//     a tile's steps are template parameters;
//     per k-step of 32 a wave reads (RBW + NBW) KB of fragments for RBW*NBW MFMAs, so larger wave
//     tiles need fewer LDS bytes per MFMA (the chip lowers its clock under MFMA load, what
//     counts is work per MFMA, not only cycles);
//   * nothing passes through registers on the way in, no LDS stores, one barrier per step, the
//     loads of step s + NS - 1 are in flight while step s computes;
//   * an operand that is contiguous along the contraction sits in LDS as [row][BK] and is read 16
//     bytes a lane; one that is contiguous along its rows (XT, YT: B of A B, A of A^T B) sits there
//     as [BK][row] and is read with transposing reads (lane s of a 16-lane group points at step row
//     s / 4, rows 4 (s % 4) ..; lane i receives 4 consecutive k of row i).  tilegemm.h transposes
//     such an operand with two-byte LDS stores: 27.0 us against 11.0 us for 2000 x 776 x 1160 bf16;
//   * X rows of the first kind sit in LDS in the order that gives a lane 8 consecutive output columns of
//     every two blocks (row i of block nb holds column (nb/2)*32 + (i/4)*8 + (nb%2)*4 + i%4): 16-byte stores,
//     64 consecutive bytes per row.  With XT that order would read half of every chunk, two passes per
//     transposing read: there the lanes exchange pieces before they store;
//   * the end of k is made of zeros: a chunk past it is fetched at an offset outside the buffer, and
//     so are rows past m and n - no branch, the same number of loads in flight on every path;
//   * workgroup numbers are mapped to tiles so that the workgroups that share an XCD (numbers
//     w, w + 8, ...) work on neighbouring tiles: 8 tile rows x all tile columns at a time, each
//     operand panel is fetched into that XCD's L2 once per group.
#pragma once
#include "lds_dma.h"
#include "tilegemm.h"

namespace cummhip {

// One operand of a step: ROWS rows, BK elements each.  TR: stored [k][row] in memory and in LDS.
template <int ROWS, int KS, int WAVES, bool TR, int SLAB_BLOCKS, bool WIDE_ORDER>
struct DenseOperand {
  static constexpr int LPR = 4 * KS;                 // 16-byte chunks per row of [row][BK]
  static constexpr int CPR = ROWS / 8;               // and per step row of [BK][row]
  static constexpr int BK = 32 * KS;
  static constexpr int VECS = ROWS * LPR;            // of a stage
  static constexpr int IP = VECS / (WAVES * 64);     // loads per wave and step
  static_assert(IP >= 1 && VECS % (WAVES * 64) == 0, "tile too small for the workgroup");
  static constexpr uint32_t kOob = 0x80000000u;

  // chunk permutation of step row e of [BK][row]: the 4 step rows of a 16-lane group, and with the next
  // group the 8, sit in different banks
  static __device__ __forceinline__ int swap_tr(int e) {
    return CPR >= 16 ? 2 * ((e & 3) + 4 * ((e >> 3) & 1)) : 2 * ((e & 3) ^ ((e >> 3) & 1));
  }
  static __device__ __forceinline__ int swap_kc(int row) {
    return KS == 1 ? (row >> 1) & 3 : ((row * KS) >> 2) & (LPR - 1);
  }

  uint32_t voff[IP];      // byte offset of this lane's chunk at step 0
  int kpos[IP];           // its first k inside a step; a chunk whose k is past the end is not fetched
  uint32_t step_bytes;

  __device__ __forceinline__ void init(int wave, int lane, int first, int count, int64_t ld) {
#pragma unroll
    for (int t = 0; t < IP; ++t) {
      const int slot = (wave * IP + t) * 64 + lane;
      if constexpr (TR) {
        const int e = slot / CPR, c = (slot % CPR) ^ swap_tr(e);
        const int row = first + c * 8;
        kpos[t] = e;
        voff[t] = row < count ? (uint32_t)(((int64_t)e * ld + row) * 2) : kOob;
      } else {
        const int rho = slot / LPR, c = (slot % LPR) ^ swap_kc(rho);
        const int i = rho & 15, nb = (rho >> 4) % SLAB_BLOCKS, slab = rho / (16 * SLAB_BLOCKS);
        const int row = first + (WIDE_ORDER ? slab * (16 * SLAB_BLOCKS) + (nb >> 1) * 32 + (i >> 2) * 8 + (nb & 1) * 4 + (i & 3) : rho);
        kpos[t] = c * 8;
        voff[t] = row < count ? (uint32_t)((int64_t)row * ld * 2) + (uint32_t)c * 16u : kOob;
      }
    }
    step_bytes = (uint32_t)(TR ? (int64_t)BK * ld * 2 : BK * 2);
  }

  __device__ __forceinline__ void issue(const v4i &rsrc, uint32_t lds, int wave, int s, int k) const {
    const uint32_t soff = (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)s * step_bytes));
    const int left = k - s * BK;      // elements of k from this step on
    if (left >= BK) {
#pragma unroll
      for (int t = 0; t < IP; ++t) dma_b128(rsrc, lds + (wave * IP + t) * 1024, voff[t], soff);
    } else {
#pragma unroll
      for (int t = 0; t < IP; ++t) dma_b128(rsrc, lds + (wave * IP + t) * 1024, kpos[t] < left ? voff[t] : kOob, soff);
    }
  }

  // fragments of the SLAB_BLOCKS blocks of slab `slab`, step slice ks (counted from slice `first`, which a
  // transposed operand gets with the base address)
  template <int N>
  __device__ __forceinline__ void offsets(int lane, int slab, int (&rd)[N], int first = 0) const {
    const int l16 = lane & 15, q = lane >> 4;
    if constexpr (TR) {
      static_assert(N == SLAB_BLOCKS, "a read offset per block");
      const int e = q * 8 + (l16 >> 2);
#pragma unroll
      for (int b = 0; b < N; ++b) {
        const int col = (slab * SLAB_BLOCKS + b) * 16 + 4 * (l16 & 3);
        rd[b] = e * (ROWS * 2) + (((col >> 3) ^ swap_tr(e)) * 16) + (col & 7) * 2;
      }
    } else {
      static_assert(N <= KS, "a read offset per step slice");
#pragma unroll
      for (int s = 0; s < N; ++s)
        rd[s] = (slab * (SLAB_BLOCKS * 16) * LPR + l16 * LPR + (((first + s) * 4 + q) ^ swap_kc(l16))) * 16;
    }
  }
  template <int N>
  static __device__ __forceinline__ v4i fragment(const char *base, const int (&rd)[N], int ks, int b) {
    if constexpr (TR) {
      typedef short v4s __attribute__((ext_vector_type(4)));
      typedef __attribute__((address_space(3))) v4s *lds_v4s;
      const char *at = base + rd[b] + ks * 32 * (ROWS * 2);
      const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)CUMM_LDS_PTR(at));
      const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)CUMM_LDS_PTR(at + 4 * (ROWS * 2)));
      return __builtin_bit_cast(v4i, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    } else {
      return *reinterpret_cast<const v4i *>(base + rd[ks] + b * 16 * LPR * 16);
    }
  }
};

// Tile of a workgroup: the workgroups that share an XCD take neighbouring tiles, eight tile rows times all
// tile columns at a time.
__device__ __forceinline__ void dense_tile(int tiles_m, int tiles_n, int *tile_m, int *tile_n) {
  int logical = blockIdx.x;
  const int nwg = gridDim.x;
  if (nwg % 8 == 0) logical = (blockIdx.x % 8) * (nwg / 8) + blockIdx.x / 8;
  constexpr int GROUP = 8;
  const int per_group = GROUP * tiles_n;
  const int g = logical / per_group, r = logical % per_group;
  const int rows_here = tiles_m - g * GROUP < GROUP ? tiles_m - g * GROUP : GROUP;
  *tile_m = g * GROUP + r % rows_here;
  *tile_n = r / rows_here;
}

// Lane (q, m) of a wave holds four columns of each of its blocks of 16, of row m.  Two blocks make one store
// of 16 bytes: with the wide order of X the lane's two pieces are neighbours already, with XT the lanes of an
// even and the next odd q exchange one.  A store covers 64 consecutive bytes of each of 16 rows: 4096^2 x 64
// 22.8 -> 20.4 us with XT.  NT: the output goes past the caches - it is larger than the L2s where the
// large tile is chosen: 4096^3 124.5 -> 120 us, 4096^2 x 1024 43.6 -> 41.3.
template <class E, int RBW, int NBW, bool XT, bool NT>
__device__ __forceinline__ void dense_epilogue(const TileGemmParams &p, const typename E::AccV (&acc)[RBW][NBW], int m_wave, int n_wave,
                                               int lane) {
  static_assert(NBW % 2 == 0, "blocks are stored in pairs");
  const int m = lane & 15, q = lane >> 4;
  const bool read_src = p.beta != 0.0f;
  uint16_t *cbase = reinterpret_cast<uint16_t *>(p.C);
  const uint16_t *dbase = reinterpret_cast<const uint16_t *>(p.D);
  typedef uint16_t v4h __attribute__((ext_vector_type(4)));
  typedef uint32_t v2u __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int rb = 0; rb < RBW; ++rb) {
    const int mm = m_wave + rb * 16 + m;
    const bool row_ok = mm < p.m;
#pragma unroll
    for (int pair = 0; pair < NBW / 2; ++pair) {
      v2u piece[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int col = n_wave + pair * 32 + (XT ? b * 16 + q * 4 : q * 8 + b * 4);
        v4h sv = {0, 0, 0, 0}, ov;
        if (read_src && row_ok && col < p.n) sv = *reinterpret_cast<const v4h *>(dbase + (int64_t)mm * p.ldd + col);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float a = acc[rb][pair * 2 + b][e];
          const float t = read_src ? __builtin_fmaf(p.alpha, a, p.beta * E::to_float(sv[e])) : p.alpha * a;
          ov[e] = E::from_float(apply_act(t, p.act, p.act_alpha));
        }
        piece[b] = __builtin_bit_cast(v2u, ov);
      }
      if constexpr (XT) {      // (odd q of the first block against even q of the second)
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          const auto r = __builtin_amdgcn_permlane16_swap(piece[0][w], piece[1][w], false, false);
          piece[0][w] = r[0];
          piece[1][w] = r[1];
        }
      }
      const int nn = n_wave + pair * 32 + (XT ? (q & 1) * 16 + (q >> 1) * 8 : q * 8);
      const v4i out = {(int)piece[0][0], (int)piece[0][1], (int)piece[1][0], (int)piece[1][1]};
      v4i *at = reinterpret_cast<v4i *>(cbase + (int64_t)mm * p.ldc + nn);
      if (row_ok && nn < p.n) {
        if constexpr (NT) __builtin_nontemporal_store(out, at);
        else *at = out;
      }
    }
  }
}

// The waves of a workgroup are WM x WN wave tiles, times WK groups that share them: group g takes the slices
// g KS / WK .. of a step's KS slices of 32 k, and the groups' sums are added up in LDS at the end.  Eight
// waves per workgroup throughout: with four, one per SIMD where a CU has a single workgroup, a step is the
// chain barrier - fragment reads - products of one wave (more stages do not shorten it: 2000 x 776 x 1160
// bf16 14.5 us with three, 15.5 with six); a second wave per SIMD reads while the first multiplies.  Over
// 290 random products of 64 .. 4096 the time is 0.92 of that with four waves: 1024^3 nt 8.8 -> 7.5 us,
// 2000 x 776 x 1160 nn 14.5 -> 11.9, 2048^3 tn 28.4 -> 23.6, 1344 x 3328 x 880 tn 22.1 -> 18.0.
template <class T, int WM, int WN, int WK, int RBW, int NBW, int KS, int NS, bool XT, bool YT>
__global__ __launch_bounds__(WM *WN *WK * 64) void densegemm_lds_kernel(const TileGemmParams p, int tiles_m, int tiles_n) {
  using E = Elem<T>;
  using AccV = typename E::AccV;
  constexpr int TM = WM * RBW * 16;
  constexpr int TN = WN * NBW * 16;
  using OpY = DenseOperand<TM, KS, WM * WN * WK, YT, RBW, false>;
  using OpX = DenseOperand<TN, KS, WM * WN * WK, XT, NBW, !XT>;
  constexpr int STAGE = (OpY::VECS + OpX::VECS) * 16;
  constexpr int L = NS - 1;                // steps the loads run ahead
  constexpr int WAIT_STEP = (L - 1) * (OpY::IP + OpX::IP);   // loads issued after those of step s when it starts
  static_assert(WAIT_STEP < 64, "too many loads in flight for the counter");
  constexpr int BK = OpY::BK;              // contraction elements per step
  static_assert(E::kBytes == 2, "two-byte elements");

  __shared__ __attribute__((aligned(16))) char ring[NS * STAGE];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave / (WM * WN), wm = wave / WN % WM, wn = wave % WN;
  constexpr int KW = KS / WK;
  int tile_m, tile_n;
  dense_tile(tiles_m, tiles_n, &tile_m, &tile_n);
  const int m0 = tile_m * TM, n0 = tile_n * TN;

  OpY y;
  OpX x;
  y.init(wave, lane, m0, p.m, p.ldy);
  x.init(wave, lane, n0, p.n, p.ldx);
  const uint32_t y_bytes = (uint32_t)(((int64_t)((YT ? p.k : p.m) - 1) * p.ldy + (YT ? p.m : p.k)) * 2);
  const uint32_t x_bytes = (uint32_t)(((int64_t)((XT ? p.k : p.n) - 1) * p.ldx + (XT ? p.n : p.k)) * 2);
  const int steps = (p.k + BK - 1) / BK;
  int y_rd[YT ? RBW : KW], x_rd[XT ? NBW : KW];
  y.offsets(lane, wm, y_rd, wk * KW);
  x.offsets(lane, wn, x_rd, wk * KW);

  AccV acc[RBW][NBW];
#pragma unroll
  for (int rb = 0; rb < RBW; ++rb)
#pragma unroll
    for (int nb = 0; nb < NBW; ++nb) acc[rb][nb] = AccV{0, 0, 0, 0};

  const uint32_t ring_at = lds_addr(ring);
  auto issue = [&](int s, int stage) __attribute__((always_inline)) {
    // a step past the end is fetched through descriptors without records: zeros, no traffic,
    // the same number of loads in flight
    const bool live = s < steps;
    const v4i rs_y = rsrc_words(p.Y, live ? y_bytes : 0u);
    const v4i rs_x = rsrc_words(p.X, live ? x_bytes : 0u);
    const uint32_t st = ring_at + (uint32_t)__builtin_amdgcn_readfirstlane(stage * STAGE);
    y.issue(rs_y, st, wave, s, p.k);
    x.issue(rs_x, st + OpY::VECS * 16, wave, s, p.k);
  };

  for (int s = 0; s < L; ++s) issue(s, s);
  int cs = 0, ls = L;   // stage computed, stage loaded (the one the previous step computed)
  for (int s = 0; s < steps; ++s) {
    wait_vmcnt<WAIT_STEP>();
    lds_barrier();
    const char *st = ring + cs * STAGE;
    v4i yf[RBW][KW], xf[NBW][KW];
#pragma unroll
    for (int nb = 0; nb < NBW; ++nb)
#pragma unroll
      for (int k = 0; k < KW; ++k) xf[nb][k] = OpX::fragment(st + OpY::VECS * 16 + (XT ? wk * KW * 32 * TN * 2 : 0), x_rd, k, nb);
#pragma unroll
    for (int rb = 0; rb < RBW; ++rb)
#pragma unroll
      for (int k = 0; k < KW; ++k) yf[rb][k] = OpY::fragment(st + (YT ? wk * KW * 32 * TM * 2 : 0), y_rd, k, rb);
    issue(s + L, ls);
    cs = cs + 1 == NS ? 0 : cs + 1;
    ls = ls + 1 == NS ? 0 : ls + 1;
#pragma unroll
    for (int k = 0; k < KW; ++k)
#pragma unroll
      for (int rb = 0; rb < RBW; ++rb)
#pragma unroll
        for (int nb = 0; nb < NBW; ++nb) acc[rb][nb] = E::mfma(xf[nb][k], yf[rb][k], acc[rb][nb]);
  }
  wait_vmcnt<0>();

  if constexpr (WK == 1) {
    dense_epilogue<E, RBW, NBW, XT, false>(p, acc, m0 + wm * (RBW * 16), n0 + wn * (NBW * 16), lane);
  } else {
    // each group finishes its share of the row blocks: it adds up all groups' sums of them, in group order
    constexpr int RO = RBW / WK;
    static_assert(RBW % WK == 0 && NS * STAGE >= WM * WN * WK * RBW * NBW * 1024, "the ring holds every group's sums");
    AccV own[RO][NBW];
    __builtin_amdgcn_s_waitcnt(0xC07F);     // lgkmcnt(0): this wave has read its last stage,
    lds_barrier();                          // and so has every other
    v4f *park = reinterpret_cast<v4f *>(ring);   // [group][wave of the group][rb][nb][lane]
    const int wg = wave % (WM * WN);
#pragma unroll
    for (int rb = 0; rb < RBW; ++rb)
#pragma unroll
      for (int nb = 0; nb < NBW; ++nb) park[(((wk * (WM * WN) + wg) * RBW + rb) * NBW + nb) * 64 + lane] = acc[rb][nb];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RO; ++r)
#pragma unroll
      for (int nb = 0; nb < NBW; ++nb) {
        AccV t = park[((wg * RBW + wk * RO + r) * NBW + nb) * 64 + lane];
#pragma unroll
        for (int g = 1; g < WK; ++g) t += park[(((g * (WM * WN) + wg) * RBW + wk * RO + r) * NBW + nb) * 64 + lane];
        own[r][nb] = t;
      }
    dense_epilogue<E, RO, NBW, XT, false>(p, own, m0 + wm * (RBW * 16) + wk * RO * 16, n0 + wn * (NBW * 16), lane);
  }
}

// The large tile, pipelined through registers: while the MFMAs of step s run on one set of fragments, the
// fragments of step s + 1 are read into the other, so that a step is not a chain of barrier, reads and
// products (with two waves per SIMD, both at the same point, nothing else fills the matrix cores).  A
// stage is free as soon as its fragments are in registers: the loads run NS steps ahead.  4096^3 f16 (one
// tile per CU) 129 -> 124 us, 8192^3 974 -> 885 us (1240 TFLOP/s, two thirds of the MFMA rate at the
// clock that the chip holds under this load, 1.86 GHz).  Slower: MFMAs of 32 x 32 x 16 (8192^3 965 us),
// half of the products in front of the barrier, raised priority around the products.
template <class T, int WM, int WN, int RBW, int NBW, int NS, bool XT, bool YT>
__global__ __launch_bounds__(WM *WN * 64) void densegemm_pipe_kernel(const TileGemmParams p, int tiles_m, int tiles_n) {
  using E = Elem<T>;
  constexpr int TM = WM * RBW * 16;
  constexpr int TN = WN * NBW * 16;
  using OpY = DenseOperand<TM, 1, WM * WN, YT, RBW, false>;
  using OpX = DenseOperand<TN, 1, WM * WN, XT, NBW, !XT>;
  constexpr int STAGE = (OpY::VECS + OpX::VECS) * 16;
  constexpr int PER = OpY::IP + OpX::IP;
  constexpr int BK = 32;
  __shared__ __attribute__((aligned(16))) char ring[NS * STAGE];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  int tile_m, tile_n;
  dense_tile(tiles_m, tiles_n, &tile_m, &tile_n);
  const int m0 = tile_m * TM, n0 = tile_n * TN;
  OpY y;
  OpX x;
  y.init(wave, lane, m0, p.m, p.ldy);
  x.init(wave, lane, n0, p.n, p.ldx);
  const uint32_t y_bytes = (uint32_t)(((int64_t)((YT ? p.k : p.m) - 1) * p.ldy + (YT ? p.m : p.k)) * 2);
  const uint32_t x_bytes = (uint32_t)(((int64_t)((XT ? p.k : p.n) - 1) * p.ldx + (XT ? p.n : p.k)) * 2);
  const int steps = (p.k + BK - 1) / BK;
  int y_rd[YT ? RBW : 1], x_rd[XT ? NBW : 1];
  y.offsets(lane, wm, y_rd);
  x.offsets(lane, wn, x_rd);
  v4f acc[RBW][NBW];
#pragma unroll
  for (int rb = 0; rb < RBW; ++rb)
#pragma unroll
    for (int nb = 0; nb < NBW; ++nb) acc[rb][nb] = v4f{0, 0, 0, 0};
  const uint32_t ring_at = lds_addr(ring);
  auto issue = [&](int s, int stage) __attribute__((always_inline)) {
    const bool live = s < steps;
    const v4i rs_y = rsrc_words(p.Y, live ? y_bytes : 0u);
    const v4i rs_x = rsrc_words(p.X, live ? x_bytes : 0u);
    const uint32_t st = ring_at + (uint32_t)__builtin_amdgcn_readfirstlane(stage * STAGE);
    y.issue(rs_y, st, wave, s, p.k);
    x.issue(rs_x, st + OpY::VECS * 16, wave, s, p.k);
  };
  v4i ya[RBW], xa[NBW], yb[RBW], xb[NBW];   // the fragments of two steps
  auto read = [&](int stage, v4i (&yf)[RBW], v4i (&xf)[NBW]) __attribute__((always_inline)) {
    const char *st = ring + stage * STAGE;
#pragma unroll
    for (int nb = 0; nb < NBW; ++nb) xf[nb] = OpX::fragment(st + OpY::VECS * 16, x_rd, 0, nb);
#pragma unroll
    for (int rb = 0; rb < RBW; ++rb) yf[rb] = OpY::fragment(st, y_rd, 0, rb);
  };
  for (int s = 0; s < NS; ++s) issue(s, s);
  wait_vmcnt<(NS - 1) * PER>();
  lds_barrier();
  read(0, ya, xa);
  int cs = 0;
  auto phase = [&](int s, v4i (&yc)[RBW], v4i (&xc)[NBW], v4i (&yn)[RBW], v4i (&xn)[NBW]) __attribute__((always_inline)) {
    wait_vmcnt<(NS - 2) * PER>();
    __builtin_amdgcn_s_waitcnt(0xC07F);     // lgkmcnt(0): the fragments of step s are in registers
    lds_barrier();
    issue(s + NS, cs);
    cs = cs + 1 == NS ? 0 : cs + 1;
    read(cs, yn, xn);
#pragma unroll
    for (int rb = 0; rb < RBW; ++rb)
#pragma unroll
      for (int nb = 0; nb < NBW; ++nb) acc[rb][nb] = E::mfma(xc[nb], yc[rb], acc[rb][nb]);
    // (reads and products interleaved: the scheduler would put all reads first)
    constexpr int READS = RBW * (YT ? 2 : 1) + NBW * (XT ? 2 : 1);
    constexpr int MF = RBW * NBW;
#pragma unroll
    for (int i = 0; i < READS; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, MF / READS > 0 ? MF / READS : 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, MF, 0);
  };
  int s = 0;
  for (; s + 1 < steps; s += 2) {
    phase(s, ya, xa, yb, xb);
    phase(s + 1, yb, xb, ya, xa);
  }
  if (s < steps) phase(s, ya, xa, yb, xb);
  wait_vmcnt<0>();
  dense_epilogue<E, RBW, NBW, XT, true>(p, acc, m0 + wm * (RBW * 16), n0 + wn * (NBW * 16), lane);
}

// The same product with the contraction split over the waves of a workgroup: 64 x 64 per workgroup, wave w
// takes the steps w, w + W, ... of 32 KS elements for the whole tile, with a ring of its own, its own waits
// and no barrier; the W tiles are added up in LDS in wave order at the end.  For products with too
// few tiles to fill the device more than about twice a tile's life is its chain of steps (wait - barrier -
// fragment reads - MFMA, 0.24 us each at one or two workgroups per CU): here the chain is a W-th as
// long, and a wave reads 2 KS KB of fragments per 4 KS MFMAs instead of twice that.
template <class T, int W, int KS, int NS, bool XT, bool YT>
__global__ __launch_bounds__(W * 64) void densegemm_wave_kernel(const TileGemmParams p, int tiles_m, int tiles_n) {
  using E = Elem<T>;
  using OpY = DenseOperand<64, KS, 1, YT, 4, false>;
  using OpX = DenseOperand<64, KS, 1, XT, 4, !XT>;
  constexpr int STAGE = (OpY::VECS + OpX::VECS) * 16;
  constexpr int L = NS - 1;
  constexpr int WAIT_STEP = (L - 1) * (OpY::IP + OpX::IP);
  constexpr int BK = OpY::BK;
  static_assert(WAIT_STEP < 64 && NS * STAGE >= 64 * 64 * 4 && E::kBytes == 2, "the ring holds a tile of sums");
  __shared__ __attribute__((aligned(16))) char ring[W][NS * STAGE];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, q = lane >> 4;
  int logical = blockIdx.x;
  const int nwg = gridDim.x;
  if (nwg % 8 == 0) logical = (blockIdx.x % 8) * (nwg / 8) + blockIdx.x / 8;
  const int m0 = (logical % tiles_m) * 64, n0 = (logical / tiles_m) * 64;

  OpY y;
  OpX x;
  y.init(0, lane, m0, p.m, p.ldy);
  x.init(0, lane, n0, p.n, p.ldx);
  const v4i rs_y = rsrc_words(p.Y, (uint32_t)(((int64_t)((YT ? p.k : p.m) - 1) * p.ldy + (YT ? p.m : p.k)) * 2));
  const v4i rs_x = rsrc_words(p.X, (uint32_t)(((int64_t)((XT ? p.k : p.n) - 1) * p.ldx + (XT ? p.n : p.k)) * 2));
  int y_rd[YT ? 4 : KS], x_rd[XT ? 4 : KS];
  y.offsets(lane, 0, y_rd);
  x.offsets(lane, 0, x_rd);
  const int steps = (p.k + BK - 1) / BK;
  const int mine = (steps - wave + W - 1) / W;

  v4f acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = v4f{0, 0, 0, 0};

  const uint32_t ring_at = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_addr(&ring[wave][0]));
  auto issue = [&](int j) __attribute__((always_inline)) {      // (a step past the end has no k left: zeros, no traffic)
    const uint32_t st = ring_at + (uint32_t)__builtin_amdgcn_readfirstlane((j % NS) * STAGE);
    const int s = wave + j * W;
    y.issue(rs_y, st, 0, s, p.k);
    x.issue(rs_x, st + OpY::VECS * 16, 0, s, p.k);
  };
  for (int j = 0; j < L; ++j) issue(j);
  for (int j = 0; j < mine; ++j) {
    wait_vmcnt<WAIT_STEP>();
    asm volatile("" ::: "memory");
    const char *st = &ring[wave][(j % NS) * STAGE];
    v4i yf[4][KS], xf[4][KS];
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int k = 0; k < KS; ++k) xf[b][k] = OpX::fragment(st + OpY::VECS * 16, x_rd, k, b);
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int k = 0; k < KS; ++k) yf[b][k] = OpY::fragment(st, y_rd, k, b);
    issue(j + L);
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[i][b] = E::mfma(xf[b][k], yf[i][k], acc[i][b]);
  }
  wait_vmcnt<0>();
  asm volatile("" ::: "memory");

  // ---- every wave parks its tile in its own ring: row m of 16 units of four columns, permuted by m
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int m = i * 16 + l16, unit = XT ? b * 4 + q : (b >> 1) * 8 + q * 2 + (b & 1);
      reinterpret_cast<v4f *>(&ring[wave][0])[m * 16 + (unit ^ l16)] = acc[i][b];
    }
  __syncthreads();
  // W * 64 threads: thread (m, part) adds up 64 / W consecutive columns of row m
  constexpr int UNITS = 16 / W;            // of four columns
  constexpr int PIECE = UNITS >= 2 ? 8 : 4;
  typedef uint16_t vh __attribute__((ext_vector_type(PIECE)));
  const int m = tid / W, part = tid % W;
  if (m0 + m >= p.m) return;
  const bool read_src = p.beta != 0.0f;
#pragma unroll
  for (int g = 0; g < UNITS * 4 / PIECE; ++g) {
    const int nn = n0 + part * (UNITS * 4) + g * PIECE;
    if (nn >= p.n) return;
    vh sv, ov;
    if (read_src) sv = *reinterpret_cast<const vh *>(reinterpret_cast<const uint16_t *>(p.D) + (int64_t)(m0 + m) * p.ldd + nn);
#pragma unroll
    for (int u = 0; u < PIECE / 4; ++u) {
      const int at = m * 16 + ((part * UNITS + g * (PIECE / 4) + u) ^ (m & 15));
      v4f sum = reinterpret_cast<const v4f *>(&ring[0][0])[at];
#pragma unroll
      for (int w = 1; w < W; ++w) sum += reinterpret_cast<const v4f *>(&ring[w][0])[at];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float t = read_src ? __builtin_fmaf(p.alpha, sum[e], p.beta * E::to_float(sv[u * 4 + e])) : p.alpha * sum[e];
        ov[u * 4 + e] = E::from_float(apply_act(t, p.act, p.act_alpha));
      }
    }
    *reinterpret_cast<vh *>(reinterpret_cast<uint16_t *>(p.C) + (int64_t)(m0 + m) * p.ldc + nn) = ov;
  }
}

}  // namespace cummhip
