// Host rules of the launch schedule search (prx_batch_autotune).
#pragma once

#include <cstdint>
#include <vector>

namespace prx {

// Wave-wide sweep thresholds (coop_min_contacts) that the search tries.  Islands
// of four or more constraints take the level form whatever the threshold, up to
// the greatest values, which keep every island on a lane (level_island); so
// where the level form takes every island of a batch (allLevel) there are two
// schedules to compare: trials of 8, 16, 64 and 128 would repeat the one of 32.
inline std::vector<std::uint32_t> CoopCandidates(bool allLevel) {
    if (allLevel) return {32u, 0xffffffffu};
    return {8u, 16u, 32u, 64u, 128u, 0xffffffffu};
}

// Whether two thresholds sweep the islands of such a batch alike.
inline bool SameSweeps(std::uint32_t a, std::uint32_t b, bool allLevel) {
    constexpr std::uint32_t kLanes = 0x7fffffffu, kSmallest = 4u;
    auto form = [](std::uint32_t k) { return k >= kLanes ? kLanes : k < kSmallest ? k : kSmallest; };
    return allLevel ? form(a) == form(b) : a == b;
}

}  // namespace prx
