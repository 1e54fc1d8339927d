// Instantiations of the LDS-tiled GEMM for one element type (selected with -DCUMM_ELEM=...).
#include <algorithm>

#include "launch.h"
#include "densegemm_lds.h"

namespace cummhip {

#define CUMM_CAT_(a, b) a##b
#define CUMM_CAT(a, b) CUMM_CAT_(a, b)

// -DCUMM_WIDE=1 builds the tiled kernels with four-byte outputs (s32 / f32) under the name
// launch_tilegemm_wide_<type>, in a translation unit of its own (and nothing else)
#ifndef CUMM_WIDE
#define CUMM_WIDE 0
#endif
constexpr bool kWide = CUMM_WIDE != 0;
#if CUMM_WIDE
#define CUMM_LAUNCH_NAME CUMM_CAT(launch_tilegemm_wide_, CUMM_NAME)
#else
#define CUMM_LAUNCH_NAME CUMM_CAT(launch_tilegemm_, CUMM_NAME)
#endif

template <class T, int BM, int BN>
static hipError_t launch_xy(bool xk, bool yk, const TileGemmParams &p, dim3 grid, hipStream_t s) {
  if (grid.x == 0 || grid.y == 0 || grid.z == 0) return hipSuccess;
  if (xk && yk) hipLaunchKernelGGL((tilegemm_kernel<T, true, true, BM, BN, 1, kWide>), grid, dim3(256), 0, s, p);
  else if (xk && !yk) hipLaunchKernelGGL((tilegemm_kernel<T, true, false, BM, BN, 1, kWide>), grid, dim3(256), 0, s, p);
  else if (!xk && yk) hipLaunchKernelGGL((tilegemm_kernel<T, false, true, BM, BN, 1, kWide>), grid, dim3(256), 0, s, p);
  else hipLaunchKernelGGL((tilegemm_kernel<T, false, false, BM, BN, 1, kWide>), grid, dim3(256), 0, s, p);
  return hipGetLastError();
}

// Plain GEMM of two-byte elements in every layout, shapes with 16-byte pieces along each operand's and
// the result's contiguous dimension: the LDS-ring kernels.  (One fp32 sum over k per element whatever
// the tile - in two parts where two groups of waves share it, in eight, added in order, for the kernel that
// splits k over its waves.)
template <class T, int WM, int WN, int WK, int RBW, int NBW, int KS, int NS, bool XT, bool YT>
static hipError_t launch_dense_ring_as(const TileGemmParams &p, hipStream_t s) {
  constexpr int TM = WM * RBW * 16, TN = WN * NBW * 16;
  if (!counted_waits_hold<densegemm_lds_kernel<T, WM, WN, WK, RBW, NBW, KS, NS, XT, YT>>()) return hipErrorNotSupported;
  const int tiles_m = (p.m + TM - 1) / TM, tiles_n = (p.n + TN - 1) / TN;
  hipLaunchKernelGGL((densegemm_lds_kernel<T, WM, WN, WK, RBW, NBW, KS, NS, XT, YT>), dim3((unsigned)(tiles_m * tiles_n)),
                     dim3(WM * WN * WK * 64), 0, s, p, tiles_m, tiles_n);
  return hipGetLastError();
}

// the large tile: fragments double-buffered in registers
template <class T, bool XT, bool YT>
static hipError_t launch_dense_pipe(const TileGemmParams &p, hipStream_t s) {
  if (!counted_waits_hold<densegemm_pipe_kernel<T, 2, 4, 8, 4, 4, XT, YT>>()) return hipErrorNotSupported;
  const int tiles_m = (p.m + 255) / 256, tiles_n = (p.n + 255) / 256;
  hipLaunchKernelGGL((densegemm_pipe_kernel<T, 2, 4, 8, 4, 4, XT, YT>), dim3((unsigned)(tiles_m * tiles_n)), dim3(512), 0, s, p, tiles_m,
                     tiles_n);
  return hipGetLastError();
}

// Which tile: the least estimated time, fitted to 290 random products of 64 .. 4096 in bf16 on the 256 CUs
// that the figures are for (us; n = tiles per CU, rounded up; k in elements; where there are two figures,
// the second is for rows that are no whole number of 128-byte lines, whose fetches touch a line more each).
// What it picks is 1.3 % slower than the fastest of the seven on average.
//   64 x 64 x 64, 2 x 2 x 2 waves, three stages   up to 32 tiles 3.7 + 0.0036 k;  n = 1: 3.7 + 0.0040 /
//                                              0.0046 k;  n = 2: 4.9 + 0.0063 / 0.0076 k;  else 2.4 + n (1.12 + 0.0031 /
//                                              0.0040 k)              (3000 x 1000 x 504 11.3)
//   64 x 64 x 128, four stages                 n = 1 only: up to 32 tiles 4.1 + 0.0026 / 0.0030 k, else 4.2 + 0.0030 /
//                                              0.0038 k               (1024^3 7.5 against 8.0; 424 x 656 x 2992
//                                              15.6 against 18.7; two tiles per CU 1.3 times as long)
//   64 x 64, k split over eight waves          up to 32 tiles 4.2 + 0.0020 k, with broken lines and tiles * k above
//                                              40 k 0.0032 k (128 x 192 x 3008 9.7 against 12.2; 96 x 80 x 3344,
//                                              broken, 10.2 against 12.8; 920 x 96 x 3816, broken, 24.9 against 17.1)
//   64 x 128 x 64, 2 x 4 waves, three stages   n = 1: 4.4 + 0.0053 / 0.0060 k;  n = 2: 5.8 + 0.0085 / 0.0104 k;  else
//                                              3.5 + n (1.6 + 0.0039 / 0.0057 k)
//                                              (2000 x 776 x 1160 11.9 against 13.8; 1504^3 18.5 against 19.7)
//   128 x 128 x 64, 2 x 4 waves, four stages   n = 1 only: 7.0 + 0.0072 / 0.0080 k, at least 9.4
//                                              (2048^3 23.5 against 27; 3488 x 600 x 1072 15.1 against 15.8)
//   the same, two stages (two workgroups       n = 2: 8.2 + 0.0122 k;  else n (3.9 + 0.0077 k) / 4.0 + n (3.4 + 0.0088 k)
//   per CU)                                    (1344 x 3328 x 880 18.0 against 21.1; 3224 x 1392 x 2968 45.7 against
//                                              54.9)
//   256 x 256 x 32, 2 x 4 waves, four stages   2.0 + n (14.8 + 0.0235 k), up to k = 384 with result rows that are
//                                              no whole lines, which it stores past the caches, 20.0;
//                                              8.5 + 0.0255 n k
//                                              (4096^3 120; 3000^3 85 against 104; 4096^2 x 256 21.5 against 27;
//                                              tn 5768 x 2456 x 192 28 against 23)
// The step-by-step cost of the small tiles is the chain of a step; from two workgroups per CU on it is the
// 64 bytes per clock that a CU fetches: a 64 x 64 tile needs 512 bytes per MFMA of 16 x 16 x 32 (four clocks of
// the CU's matrix cores), a 128 x 128 tile 256, a 256 x 256 tile 128.
constexpr int kFigureCus = 256;
inline int tiles_per_cu(const TileGemmParams &p, int tm, int tn) {
  return (int)(((int64_t)((p.m + tm - 1) / tm) * ((p.n + tn - 1) / tn) + kFigureCus - 1) / kFigureCus);
}

template <class T, bool XT, bool YT>
static hipError_t launch_dense_ring_layout(const TileGemmParams &p, hipStream_t s) {
  const auto most = [](double a, double b) { return a > b ? a : b; };
  const double k = p.k;
  const bool lines = p.ldx % 64 == 0 && p.ldy % 64 == 0;
  const auto of = [&](double whole, double broken) { return lines ? whole : broken; };
  const int n64 = tiles_per_cu(p, 64, 64), n128 = tiles_per_cu(p, 64, 128), n128s = tiles_per_cu(p, 128, 128), n256 = tiles_per_cu(p, 256, 256);
  const double tiles = (double)((p.m + 63) / 64) * ((p.n + 63) / 64);
  const bool few = tiles <= 32;
  const double t64 = few        ? 3.7 + 0.0036 * k
                     : n64 == 1 ? 3.7 + of(0.0040, 0.0046) * k
                     : n64 == 2 ? 4.9 + of(0.0063, 0.0076) * k
                                : 2.4 + n64 * (1.12 + of(0.0031, 0.0040) * k);
  const double t64k = few ? 4.1 + of(0.0026, 0.0030) * k : (n64 == 1 ? 4.2 + of(0.0030, 0.0038) * k : 1e30);
  const double tw = few ? 4.2 + (lines || tiles * k <= 40000 ? 0.0020 : 0.0032) * k : 1e30;
  const double t128 = n128 == 1   ? 4.4 + of(0.0053, 0.0060) * k
                      : n128 == 2 ? 5.8 + of(0.0085, 0.0104) * k
                                  : 3.5 + n128 * (1.6 + of(0.0039, 0.0057) * k);
  const double t128s = n128s == 1   ? most(9.4, 7.0 + of(0.0072, 0.0080) * k)
                       : n128s == 2 ? 8.2 + 0.0122 * k
                                    : of(n128s * (3.9 + 0.0077 * k), 4.0 + n128s * (3.4 + 0.0088 * k));
  const double t256 = most(2.0 + n256 * ((p.ldc % 64 == 0 || k > 384 ? 14.8 : 20.0) + 0.0235 * k), 8.5 + 0.0255 * n256 * k);
  const double least = std::min({t64, t64k, tw, t128, t128s, t256});
  if (least == t256) return launch_dense_pipe<T, XT, YT>(p, s);
  if (least == t128s)
    return n128s == 1 ? launch_dense_ring_as<T, 2, 4, 1, 4, 2, 2, 4, XT, YT>(p, s) : launch_dense_ring_as<T, 2, 4, 1, 4, 2, 2, 2, XT, YT>(p, s);
  if (least == t128) return launch_dense_ring_as<T, 2, 4, 1, 2, 2, 2, 3, XT, YT>(p, s);
  if (least == t64k) return launch_dense_ring_as<T, 2, 2, 2, 2, 2, 4, 4, XT, YT>(p, s);
  if (least == tw) {
    if (!counted_waits_hold<densegemm_wave_kernel<T, 8, 1, 2, XT, YT>>()) return hipErrorNotSupported;
    const int tiles_m = (p.m + 63) / 64, tiles_n = (p.n + 63) / 64;
    hipLaunchKernelGGL((densegemm_wave_kernel<T, 8, 1, 2, XT, YT>), dim3((unsigned)(tiles_m * tiles_n)), dim3(512), 0, s, p, tiles_m,
                       tiles_n);
    return hipGetLastError();
  }
  return launch_dense_ring_as<T, 2, 2, 2, 2, 2, 2, 3, XT, YT>(p, s);
}

// Contractions of a step or two have nothing to stream: half a step always, and up to a step and a half with
// several tiles per CU, where what counts is how many workgroups start and store at once, the
// register-staged kernel in 64 x 64 tiles is the faster one (536 x 928 x 16 3.7 us and 4.2; 3000^2 x 8 to 64:
// 8.6 - 11.5 us against 13.0 and more; 1352 x 3720 x 72 8.7 and 9.9; 4096^2 x 64 16.1 - 19.2 and 17.7; with
// k = 128 13.8 and 13.6 at 3000^2).
inline bool dense_ring_streams(const TileGemmParams &p) {
  const int n = tiles_per_cu(p, 64, 64);
  return p.k > (n >= 4 ? 96 : 32);
}

template <class T>
static bool launch_dense_ring(bool xk, bool yk, const TileGemmParams &p, hipStream_t s, hipError_t *err) {
  if constexpr (Elem<T>::kBytes != 2) {
    return false;
  } else {
    const auto al16 = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15u) == 0; };
    const int64_t y_rows = yk ? p.m : p.k, y_cols = yk ? p.k : p.m, x_rows = xk ? p.n : p.k, x_cols = xk ? p.k : p.n;
    const bool ok = p.kv == 1 && p.split_k == 1 && !p.x_gather && !p.y_gather && !p.red_mask &&
                    p.m > 0 && p.n > 0 && p.k > 0 && y_cols % 8 == 0 && x_cols % 8 == 0 && p.n % 8 == 0 &&
                    p.ldx % 8 == 0 && p.ldy % 8 == 0 && p.ldc % 8 == 0 && p.ldd % 8 == 0 &&
                    al16(p.X) && al16(p.Y) && al16(p.C) && al16(p.D) &&
                    ((y_rows - 1) * p.ldy + y_cols) * 2 < ((int64_t)1 << 31) && ((x_rows - 1) * p.ldx + x_cols) * 2 < ((int64_t)1 << 31);
    if (!ok) return false;
    if (!dense_ring_streams(p)) {
      *err = launch_xy<T, 2, 2>(xk, yk, p, dim3((p.m + 63) / 64, (p.n + 63) / 64, 1), s);
      return true;
    }
    if (xk && yk) *err = launch_dense_ring_layout<T, false, false>(p, s);
    else if (yk) *err = launch_dense_ring_layout<T, true, false>(p, s);
    else if (xk) *err = launch_dense_ring_layout<T, false, true>(p, s);
    else *err = launch_dense_ring_layout<T, true, true>(p, s);
    return *err != hipErrorNotSupported;     // (the register-staged kernel takes over)
  }
}

hipError_t CUMM_LAUNCH_NAME(int tm, int tn, bool xk, bool yk, const TileGemmParams &p, dim3 grid, hipStream_t s) {
  using T = CUMM_ELEM;
  if constexpr (!kWide) {
    hipError_t err = hipSuccess;
    if (launch_dense_ring<T>(xk, yk, p, s, &err)) return err;
  }
  if (tm == 64 && tn == 64) return launch_xy<T, 2, 2>(xk, yk, p, grid, s);
  if (tm == 128 && tn == 128) return launch_xy<T, 4, 4>(xk, yk, p, grid, s);
  return hipErrorInvalidValue;
}

#if !defined(CUMM_NO_WGRAD_ATOMIC) && !CUMM_WIDE
// The lists and zeros of a weight gradient: in the launch of the bias sums, if there is one (*last: their last step)
template <class T>
static hipError_t prepare(const WgradPrepareParams &pre, int blocks, const ColumnSumParams *sums, ColumnFinalParams *last, hipStream_t s) {
  if (sums != nullptr) return launch_column_partial(*sums, &pre, blocks, std::is_same_v<T, BF16>, s, last);
  hipLaunchKernelGGL(wgrad_prepare_kernel, dim3((unsigned)blocks), dim3(256), 0, s, pre);
  return hipGetLastError();
}

// The table that the unit-walking kernel reads: 1 = by position, 0 = by row (also where a caller has both and only that
// instantiation holds its counted waits), -1 = neither
constexpr int units_table(bool by_position, bool by_position_holds, bool by_row_holds) {
  return by_position && by_position_holds ? 1 : (by_row_holds ? 0 : -1);
}
static_assert(units_table(true, true, false) == 1 && units_table(true, false, true) == 0 && units_table(true, false, false) == -1 &&
              units_table(false, true, true) == 0 && units_table(false, true, false) == -1, "by position only where asked for");

// The unit-walking kernel, for 128 x 128 channels or 64 x 64
template <class T, bool DET>
static int units_table_of(bool wide, bool by_position) {
  if (wide) return units_table(by_position, counted_waits_hold<wgrad_units_kernel<T, 2, 2, 1, DET, true>>(), counted_waits_hold<wgrad_units_kernel<T, 2, 2, 1, DET>>());
  return units_table(by_position, counted_waits_hold<wgrad_units_kernel<T, 1, 1, 2, DET, true>>(), counted_waits_hold<wgrad_units_kernel<T, 1, 1, 2, DET>>());
}
template <class T, bool DET>
static void launch_units(bool wide, const WgradParams &p, dim3 grid, hipStream_t s) {
  if (p.by_position != nullptr) {
    if (wide) hipLaunchKernelGGL((wgrad_units_kernel<T, 2, 2, 1, DET, true>), grid, dim3(256), 0, s, p);
    else hipLaunchKernelGGL((wgrad_units_kernel<T, 1, 1, 2, DET, true>), grid, dim3(256), 0, s, p);
  } else {
    if (wide) hipLaunchKernelGGL((wgrad_units_kernel<T, 2, 2, 1, DET>), grid, dim3(256), 0, s, p);
    else hipLaunchKernelGGL((wgrad_units_kernel<T, 1, 1, 2, DET>), grid, dim3(256), 0, s, p);
  }
}

hipError_t CUMM_CAT(launch_wgrad_atomic_, CUMM_NAME)(const WgradParams &p, const WgradPrepareParams &pre,
                                                     const WgradFinalizeParams &f, const ColumnSumParams *sums, hipStream_t s) {
  using T = CUMM_ELEM;
  const int groups = (p.num_red + p.tiles_per_wg - 1) / p.tiles_per_wg;
  // both channel counts above 64: units of 128 x 128 channels (one gather of the full rows)
  const bool wide = p.live_list != nullptr && p.K > 64 && p.C > 64;
  const int cpu_ = wide ? 128 : 64;   // channels per unit block
  const int kblocks = (p.K + cpu_ - 1) / cpu_, cblocks = (p.C + cpu_ - 1) / cpu_;
  if (groups == 0 || p.kv == 0) return hipSuccess;
  hipError_t e;
  ColumnFinalParams last = {};
  if (p.live_list != nullptr) {
    // lists + zeroed image, then a resident grid that walks the units
    const int table = units_table_of<T, false>(wide, p.by_position != nullptr);
    if (table < 0) return hipErrorNotSupported;
    static int resident_of[2][2][16] = {};
    int dev = 0;
    e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    int &resident = resident_of[table][wide ? 1 : 0][dev & 15];
    if (resident == 0) {
      int cus = 0, per_cu = 0;
      e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
      if (e == hipSuccess)
        e = table == 1 ? (wide ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, wgrad_units_kernel<T, 2, 2, 1, false, true>, 256, 0)
                               : hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, wgrad_units_kernel<T, 1, 1, 2, false, true>, 256, 0))
                       : (wide ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, wgrad_units_kernel<T, 2, 2, 1>, 256, 0)
                               : hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, wgrad_units_kernel<T, 1, 1, 2>, 256, 0));
      if (e != hipSuccess) return e;
      resident = cus * per_cu > 0 ? cus * per_cu : 1;
    }
    e = prepare<T>(pre, p.kv + kWgradZeroBlocks, sums, &last, s);
    if (e != hipSuccess) return e;
    // With several 64 x 64 channel blocks a unit either takes one of them (more units: small
    // inputs) or walks them all on one set of pair lists (the centre offset alone then gives
    // `groups` units: enough when that fills the device).
    WgradParams q = p;
    if (table == 0) q.by_position = nullptr;
    q.merge_blocks = kblocks * cblocks > 1 && groups >= resident ? 1 : 0;
    // never more workgroups than units can exist
    const long long max_units = ((long long)groups * p.kv + p.kv) * (q.merge_blocks ? 1 : kblocks * cblocks);
    const dim3 units_grid((unsigned)(max_units < resident ? max_units : resident));
    launch_units<T, false>(wide, q, units_grid, s);
  } else {
    if (sums != nullptr && (e = launch_column_partial(*sums, nullptr, 0, std::is_same_v<T, BF16>, s, &last)) != hipSuccess) return e;
    dim3 grid(groups, p.kv * kblocks * cblocks, 1);
    hipLaunchKernelGGL((wgrad_atomic_kernel<T>), grid, dim3(256), 0, s, p);
  }
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (last.groups > 0) hipLaunchKernelGGL((wgrad_finalize_kernel<T, true>), dim3((unsigned)((f.total / 4 + 255) / 256) + last.groups), dim3(256), 0, s, f, last);
  else hipLaunchKernelGGL((wgrad_finalize_kernel<T, false>), dim3((unsigned)((f.total / 4 + 255) / 256) + last.groups), dim3(256), 0, s, f, last);
  return hipGetLastError();
}

// Fixed-order variant: the same units, a contiguous run per workgroup, partial sums stored into
// slots and added up in workgroup order.  `max_wgs` = workgroups the caller's slots allow.  The workgroups of the kernel that
// reads the table by row, whichever table is read: their number decides the order of the sums.
int CUMM_CAT(wgrad_ordered_resident_, CUMM_NAME)(bool wide) {
  using T = CUMM_ELEM;
  static int resident_of[2][16] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  int &resident = resident_of[wide ? 1 : 0][dev & 15];
  if (resident == 0) {
    int cus = 0, per_cu = 0;
    hipError_t e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess)
      e = wide ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, wgrad_units_kernel<T, 2, 2, 1, true>, 256, 0)
               : hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, wgrad_units_kernel<T, 1, 1, 2, true>, 256, 0);
    if (e != hipSuccess) return 0;
    resident = cus * per_cu > 0 ? cus * per_cu : 1;
  }
  return resident;
}

hipError_t CUMM_CAT(launch_wgrad_ordered_, CUMM_NAME)(const WgradParams &p, const WgradPrepareParams &pre,
                                                      const WgradOrderedParams &f, bool wide, int wgs, const ColumnSumParams *sums,
                                                      hipStream_t s) {
  using T = CUMM_ELEM;
  if (p.num_red == 0 || p.kv == 0 || wgs < 1) return hipSuccess;
  const int table = units_table_of<T, true>(wide, p.by_position != nullptr);
  if (table < 0) return hipErrorNotSupported;
  WgradParams q = p;
  if (table == 0) q.by_position = nullptr;
  ColumnFinalParams last = {};
  hipError_t e = prepare<T>(pre, p.kv, sums, &last, s);   // lists only: no image to zero
  if (e != hipSuccess) return e;
  launch_units<T, true>(wide, q, dim3(wgs), s);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (last.groups > 0) hipLaunchKernelGGL((wgrad_finalize_ordered_kernel<T, true>), dim3((unsigned)((f.total / 4 + 31) / 32) + last.groups), dim3(256), 0, s, f, last);
  else hipLaunchKernelGGL((wgrad_finalize_ordered_kernel<T, false>), dim3((unsigned)((f.total / 4 + 31) / 32) + last.groups), dim3(256), 0, s, f, last);
  return hipGetLastError();
}
#endif

}  // namespace cummhip
