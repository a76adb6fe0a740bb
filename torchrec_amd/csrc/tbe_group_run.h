// How the sixteen-lane kernel takes the bags of a lane group (plain C++: the CPU tests include it too).
#pragma once

#include <cstdint>

namespace tra {

// Ids that a bag of `given` ids pools: as on every route, the low 32 bits of the count, none if that is negative.
constexpr int bag_ids(int64_t given) { return (int32_t)given > 0 ? (int32_t)given : 0; }

// Whether the ids of a bag of len ids end where the next bag's begin.  Only then are a group's bags one run, whose loop
// bound is the distance between their starts.  Lengths that are negative or do not fit 32 bits, and running sums that
// wrap, move the starts by other amounts than the bags' own ids: such bags are walked one by one.
constexpr bool bags_join(int64_t start, int len, int64_t next_start) {
  return (uint64_t)next_start - (uint64_t)start == (uint64_t)len;
}

}  // namespace tra
