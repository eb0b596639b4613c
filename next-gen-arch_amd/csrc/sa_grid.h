// Launch limits, constexpr for host checks.
#pragma once

namespace sa {

// A grid dimension holds fewer than 2^32 threads.
constexpr bool grid_fits(long long blocks, int threads) { return blocks >= 0 && blocks < (1LL << 32) / threads; }

// Waves that merge one row's P split partials: four from 8 partials on, a
// workgroup per row, where the grid holds that many rows; else one, four rows per
// workgroup.
constexpr int combine_waves(int P, long long rows) { return P >= 8 && grid_fits(rows, 256) ? 4 : 1; }

}  // namespace sa
