// Launch table of the batched persistent stage kernel (per precision x tile).
#pragma once

#include <algorithm>
#include <vector>

#include "batch_kernel.hpp"
#include "stage_dispatch.hpp"

namespace cato {

using BatchLauncher = void (*)(dim3 grid, hipStream_t stream, const BatchStageArgs &args);
BatchLauncher batch_launcher_p0(int tile);
BatchLauncher batch_launcher_p1(int tile);
inline BatchLauncher batch_launcher(int prec, int tile) {
  return prec == CATO_PRECISION_FP32_FLUX ? batch_launcher_p1(tile) : batch_launcher_p0(tile);
}

// Workgroups of 256 threads a CU holds of the batched stage kernel.
template <typename R> inline int batch_wgs_per_cu(int tile) {
  switch (tile) {
    case 0: return batch_waves_per_simd<R, kTiles[0].tx, kTiles[0].ty>();
    case 1: return batch_waves_per_simd<R, kTiles[1].tx, kTiles[1].ty>();
    case 2: return batch_waves_per_simd<R, kTiles[2].tx, kTiles[2].ty>();
    default: return batch_waves_per_simd<R, kTiles[3].tx, kTiles[3].ty>();
  }
}
inline int batch_wgs_per_cu(int prec, int tile) {
  return prec == CATO_PRECISION_FP32_FLUX ? batch_wgs_per_cu<f32x>(tile) : batch_wgs_per_cu<double>(tile);
}

// A solve's share of the work list, and the relative time of one of its tiles
// (us of an FP64 stage of 1024^2 cells, each scheme alone).
struct BatchShare {
  int solve, tiles, variant;
};
inline int variant_cost(int variant) {
  static const int flux[FLUX_COUNT] = {70, 68, 68, 76, 76, 78, 64, 66, 92};
  static const int limiter[LIM_COUNT] = {0, 1, 4, 24, 42};
  return flux[variant / LIM_COUNT] + limiter[variant % LIM_COUNT];
}

// The work list of a stage: kNumXcd slices, one to an XCD, each with its eighth of
// every variant's tiles (neighbouring tiles of a solve in one slice), the dearest
// variants first, so that the XCDs finish together and the last items are the
// cheapest.  A stage of 32 solves of side 64 to 256, four fluxes with minmod or MLP5:
// 104 us with the list cut where it fell, grouped by variant, 86 us so (FP32 flux
// 52 and 46 us); of 128 solves of side 64 to 512 812 and 785 us.
inline void build_work_list(std::vector<BatchShare> shares, std::vector<BatchItem> &items,
                            int (&slices)[kNumXcd + 1]) {
  std::stable_sort(shares.begin(), shares.end(), [](const BatchShare &x, const BatchShare &y) {
    const int cx = variant_cost(x.variant), cy = variant_cost(y.variant);
    return cx != cy ? cx > cy : x.variant < y.variant;
  });
  std::vector<BatchItem> all;
  std::vector<size_t> group{0};  // where each variant's items begin, and the end
  for (size_t k = 0; k < shares.size(); ++k) {
    for (int t = 0; t < shares[k].tiles; ++t) all.push_back({shares[k].solve, t});
    if (k + 1 == shares.size() || shares[k + 1].variant != shares[k].variant) group.push_back(all.size());
  }
  items.clear();
  items.reserve(all.size());
  for (int x = 0; x < kNumXcd; ++x) {
    slices[x] = (int)items.size();
    for (size_t g = 0; g + 1 < group.size(); ++g) {
      const size_t n = group[g + 1] - group[g];
      items.insert(items.end(), all.begin() + group[g] + n * x / kNumXcd, all.begin() + group[g] + n * (x + 1) / kNumXcd);
    }
  }
  slices[kNumXcd] = (int)items.size();
}

}  // namespace cato
