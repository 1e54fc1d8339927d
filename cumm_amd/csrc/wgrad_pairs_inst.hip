// Instantiations of the pair-list weight gradient for one element type (selected with -DCUMM_ELEM=...).
#include "launch.h"

namespace cummhip {

#define CUMM_CAT_(a, b) a##b
#define CUMM_CAT(a, b) CUMM_CAT_(a, b)

template <class T, bool WIDE, bool SUMS>
static hipError_t finalize(const WgradPairsFinalizeParams &f, int most_slots, const ColumnFinalParams &sums, hipStream_t s) {
  const uint32_t groups = (uint32_t)f.K * (uint32_t)(f.C / 4);
  const auto grid = [&](uint32_t g) { return dim3((groups * g + 255) / 256, (unsigned)(f.lists + (SUMS ? 1 : 0))); };
  // Lanes per element: enough for one or two batches of eight loads on a lane of the longest list; with
  // many lists, most of which have a few slots, eight lanes at most (125 lists, the longest of 81 slots,
  // 64 x 64 channels: 34.4 us with 32 lanes)
  if (most_slots <= 16) hipLaunchKernelGGL((wgrad_pairs_finalize_kernel<T, 2, WIDE, SUMS>), grid(2), dim3(256), 0, s, f, sums);
  else if (most_slots <= 64 || f.lists > 8) hipLaunchKernelGGL((wgrad_pairs_finalize_kernel<T, 8, WIDE, SUMS>), grid(8), dim3(256), 0, s, f, sums);
  else hipLaunchKernelGGL((wgrad_pairs_finalize_kernel<T, 32, WIDE, SUMS>), grid(32), dim3(256), 0, s, f, sums);
  return hipGetLastError();
}

hipError_t CUMM_CAT(launch_wgrad_pairs_, CUMM_NAME)(const WgradPairsParams &p, const WgradPairsFinalizeParams &f, bool wide,
                                                    int most_slots, const ColumnSumParams *sums, hipStream_t s) {
  using T = CUMM_ELEM;
  if (!counted_waits_hold<wgrad_pairs_kernel<T>>()) return hipErrorNotSupported;
  ColumnFinalParams last = {};
  if (sums != nullptr) {
    const hipError_t e = launch_column_partial(*sums, nullptr, 0, std::is_same_v<T, BF16>, s, &last);
    if (e != hipSuccess) return e;
  }
  const unsigned combos = (unsigned)(p.kblocks * p.cblocks), wgs = (unsigned)p.wgs;
  const unsigned grid = wgs >= 8u ? (wgs + 7u) / 8u * 8u * combos : (wgs * combos + 7u) / 8u * 8u;     // (as the kernel maps them)
  if (grid) {
    hipLaunchKernelGGL(wgrad_pairs_kernel<T>, dim3(grid), dim3(256), 0, s, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (last.groups > 0) return wide ? finalize<T, true, true>(f, most_slots, last, s) : finalize<T, false, true>(f, most_slots, last, s);
  return wide ? finalize<T, true, false>(f, most_slots, last, s) : finalize<T, false, false>(f, most_slots, last, s);
}

}  // namespace cummhip
