// SPRT walk: the memory plan of a walk launch (k_sprt.hip).
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace gcr {

// Memory plan of a walk launch: 64-bit words of a point row, models per
// window, words of scratch.  max_n / max_slots: the largest pair and the
// longest slot list of the items; budget_words bounds the bit rows of a window
// (a window holds at least 8 models, if the grid does).
struct SprtPlan {
  int words, max_window;
  size_t scratch_words;
};

// Workgroups of a mask launch at most, one per item and model of the window
// (the least is one model per item): a launch of 256-thread workgroups must
// stay below 2^32 threads, which small pairs would pass within the budget
// (points of one word, 32M words: 2^24 workgroups).
constexpr int64_t kSprtMaxBlocks = 1 << 22;

inline SprtPlan sprt_plan(int num_items, int max_n, int max_slots, int64_t budget_words) {
  SprtPlan p;
  const int64_t items = std::max(1, num_items);
  p.words = (max_n + 63) / 64;
  const int64_t per_slot = 2 * (int64_t)p.words * items;
  const int64_t window = std::min(std::max<int64_t>(8, budget_words / std::max<int64_t>(1, per_slot)),
                                  std::max<int64_t>(1, kSprtMaxBlocks / items));
  p.max_window = (int)std::min<int64_t>(max_slots, window);
  // inlier and kept rows of a window, the start and record rows, values, kept
  // and inlier counts
  p.scratch_words = (size_t)(per_slot * p.max_window) + 2 * (size_t)p.words * (size_t)items +
                    2 * (size_t)p.max_window * (size_t)items;
  return p;
}

}  // namespace gcr
