// SPRT walk: the rules that decide without the reference's running product,
// and the memory plan of a walk launch (k_sprt.hip).  Plain functions of
// numbers, for the kernels and for host code.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>

#if defined(__HIP__)
#define GCR_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define GCR_HOST_DEVICE inline
#endif

namespace gcr {

// The ratio's factors, their logarithms and log A with the band around it.
struct Chain {
  double f_in, f_out, A;
  double l_in, l_out, l_A;
  double hi, lo;  // log A and the margin around it
  int unit;       // both factors are 1: the product stays at 1
  int fast;       // the logarithms are finite
};

// The band of a walk over n positions.  Margin of a sum of at most n
// logarithms: the product's n roundings (n 2^-53) and the logarithms' errors,
// each with a factor of fifty and more to spare.
GCR_HOST_DEVICE void chain_band(Chain& c, int n) {
  const double m = 1e-14 * (16.0 + (double)n) + 1e-13 * (double)n * fmax(fabs(c.l_in), fabs(c.l_out));
  c.hi = c.l_A + m;
  c.lo = c.l_A - m;
  c.unit = c.f_in == 1.0 && c.f_out == 1.0;
  c.fast = fabs(c.l_in) < 1e300 && fabs(c.l_out) < 1e300 && fabs(c.l_A) < 1e300;
}

// The logarithm of the ratio after a inliers and b outliers; above A for
// certain, below A for certain, or neither; a product below e^-690 is near the
// subnormal range.
GCR_HOST_DEVICE double chain_log(const Chain& c, int a, int b) { return (double)a * c.l_in + (double)b * c.l_out; }
GCR_HOST_DEVICE bool chain_above(const Chain& c, double l) { return l > c.hi; }
GCR_HOST_DEVICE bool chain_below(const Chain& c, double l) { return l < c.lo; }
GCR_HOST_DEVICE bool chain_low(double l) { return l < -690.0; }

// A product below e^-690 cannot exceed A within `left` more factors: it has at
// least 690 + log A to climb, and no less if it passes through the subnormal
// range (the climb from 2^-1022 on is in the normal range).
GCR_HOST_DEVICE bool chain_no_return(const Chain& c, int left) {
  const double up = fmax(fmax(c.l_in, c.l_out), 0.0);
  return (double)left * up * (1.0 + 1e-9) < 680.0 + c.l_A;
}

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
