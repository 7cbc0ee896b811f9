// The demand records of ferry_history_count, written by the device and summed by the planner.
#pragma once

#include <cstdint>

namespace ferry {

// tokens of one record (at most 65,535, so that an expert's count fits 16 bits: a token names an
// expert once)
constexpr int64_t kCountTokens = 512;

// int32 words of one record: 0 or 1 + the first token (of the record's) with an ID outside
// [0, E) or a repeated one, then E uint16 counts, padded to whole words
constexpr int64_t count_record_words(int64_t experts) { return 1 + (experts + 1) / 2; }

}  // namespace ferry
