// launch_rules.h -- rules of the host's dispatch that are arithmetic alone (host code, no HIP).
#pragma once

#include <algorithm>
#include <cstdint>

namespace pdattn {

// Sources per row that the device-range merge sizes its round trips for. A row has at most ngroups of
// them and ngroups / B + 2 on average, but one long sequence among short ones has nearly all, so never
// fewer than 16 per trip. One sequence of 30000 tokens and 31 of 200 (64 ranges) with 8 / 16 / 32 / 64
// per trip: 37.7 / 35.8 / 35.2 / 35.3 us, and 63 of 200 42.0 / 40.0 / 40.3 / 41.6; 32 ragged sequences of
// 200-6000 73.2 / 72.4 / 72.9 / 73.7.
inline int merge_ranges_sources(int ngroups, int B) { return std::min(ngroups, std::max(ngroups / B + 2, 16)); }

}  // namespace pdattn
