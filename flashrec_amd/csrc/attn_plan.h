// The attention plan's layout: one record of fixed size per query group, so
// that where a record stands depends on the group alone, not on how many
// tokens the plan was made for or are attended now (a plan may cover more
// tokens than a call; a captured launch may run more tokens than the batch its
// plan was made for).
#pragma once

#include <cstdint>

namespace fr {

// A record of a group of TOK tokens:
//   [0]            slots shared by all of its tokens, rounded down to 32 (0: none)
//   [1]            plan_tag(group): the record is this group's (a buffer without
//                  it, zeros for instance, is no plan and is not used)
//   [2 + i]        tokens of the segment that starts at token i (0: none starts there)
//   [2 + TOK + i]  leading list positions that hold the same slots for all of them
constexpr int kPlanTag = 1, kPlanCount = 2;
inline constexpr int plan_shared_at(int tok) { return kPlanCount + tok; }
inline constexpr int plan_stride(int tok) { return kPlanCount + 2 * tok; }

inline constexpr int32_t plan_tag(int64_t group) {
  return static_cast<int32_t>(0x46520000u + static_cast<uint32_t>(group));
}

// Tokens of the segment that starts at token `first` of a group of which
// `ntok` tokens are attended, from its record's entry: at least one and no more
// than are left, so that a walk over the segments ends whatever the record
// holds (tokens that the plan did not know have 0 there and go one by one).
inline constexpr int plan_count(int entry, int first, int ntok) {
  return entry < 1 ? 1 : (entry > ntok - first ? ntok - first : entry);
}

}  // namespace fr
