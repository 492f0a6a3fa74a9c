// What the work units of a grouped contraction take, in cycles (host side: the
// tile shapes, the K chunks and the queue's order follow from it).
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

#include "../../include/tenet_hip.h"

namespace tenet {

static const int TILE_EDGE[3] = {64, 32, 16};

// Cycles of a unit outside its K steps (queue, first loads, epilogue), and the
// smallest unit worth cutting off a longer one.  Batches of 40..1024 unlike
// problems time within 2% for 1000..6000 and 8192..32768.
constexpr double UNIT_CYCLES = 3000.0, MIN_UNIT_CYCLES = 16384.0;

// Cycles of a CU's address unit per wave load of 16 rows x 4 contracted
// entries, from the cache lines it touches (rows: the runs of adjacent row
// entries; k: those of the contracted entries; pair: two k steps per load).
inline double gather_cycles(const std::vector<int64_t>& rows, const std::vector<int64_t>& k, bool pair) {
  auto run = [](const std::vector<int64_t>& t) {
    if (t.size() < 2) return 1.0;
    size_t breaks = 0;
    for (size_t i = 1; i < t.size(); ++i) breaks += t[i] != t[i - 1] + 1;
    return (double)t.size() / (double)(breaks + 1);
  };
  const double rr = rows.size() < 2 ? 16.0 : std::min(16.0, run(rows));
  const double kr = k.size() < 2 ? 4.0 : std::min(4.0, run(k));
  const double lines = std::max(4.0, 64.0 / std::max(rr, kr));
  return (16.0 + 2.0 * lines) * (pair && rr < kr ? 0.5 : 1.0);
}

// Modelled cycles of one (tile, 16-wide K step) per tile shape: the larger of
// the MFMA time on each SIMD (64, 16 and 4 blocks x 4 products over the four
// waves) and the operand loads' address time.  The 32 x 32 shape, whose waves
// deal K, measured 0.8 of that (five batches of each type, 4% in the mean).
inline void tile_step_cycles(int dtype, double clx, double cly, double c[3]) {
  const double mf = dtype == TENET_C128 ? 64 : 32;
  c[0] = std::max(64 * mf, 32 * (clx + cly));
  c[1] = 0.8 * std::max(16 * mf, 8 * (clx + cly));
  c[2] = std::max(4 * mf, 4 * (clx + cly));
}

// Modelled cycles of a problem's units: its tiles' K steps, and the rest of
// every unit they are cut into.
inline double tile_cycles(double step, int64_t tiles, int64_t ksteps, int64_t kchunks) {
  return (double)tiles * (step * (double)ksteps + UNIT_CYCLES * (double)kchunks);
}

// What each tile shape takes per modelled cycle, the 64 x 64 shape being 1,
// from the times of one problem in all three and the cycles modelled for it.
inline void tile_efficiency(const double ms[3], const double cycles[3], double eff[3]) {
  const double first = ms[0] / cycles[0];
  for (int v = 0; v < 3; ++v) eff[v] = ms[v] / cycles[v] / first;
}

}  // namespace tenet
