// SPRT walk of one model on inlier bits, 64 positions at a time: what one
// wavefront does (k_sprt.hip has the reasons).  Values that decide the control
// flow are the same on every lane.  The wave operations (lane_id, ballot64,
// readlane_i64, uni, wave_sum_i32) are those of dev_common.hpp, included before;
// a host check brings its own.
#pragma once

#include "sprt_rules.hpp"

namespace gcr {

namespace {

// The positions of a word against the threshold (lane l: position l with a
// inliers and b outliers up to it), as lane masks.
struct Sides {
  uint64_t above, open, low;  // above A for certain; undecided; below A with a product near the subnormal range
};
__device__ __forceinline__ Sides chain_sides(const Chain& c, int a, int b) {
  const double L = chain_log(c, a, b);
  Sides s;
  s.above = ballot64(chain_above(c, L));
  const uint64_t below = ballot64(chain_below(c, L));
  s.open = ~(s.above | below);
  s.low = below & ballot64(chain_low(L));
  return s;
}

__device__ __forceinline__ bool no_return(const Chain& c, int left) { return uni(chain_no_return(c, left)) != 0; }

// A model's rows: lane l holds words l of the first 64 words (4,096
// positions); later words come from memory.
struct Rows {
  uint64_t inl, keep, start;  // this lane's words
  const uint64_t *g_inl, *g_keep, *g_start;
  __device__ __forceinline__ uint64_t inl_word(int w) const {
    return w < 64 ? (uint64_t)readlane_i64((int64_t)inl, w) : g_inl[w];
  }
};

struct WalkResult {
  int count, tested;
  bool rejected;
};

// The reference's product over the low cnt positions of m (inlier bits); top:
// the largest product on the way (at least the first).
__device__ __forceinline__ double chain_word(const Chain& c, double lambda, uint64_t m, int cnt, double& top) {
  double x = lambda;
  top = lambda;
  if (cnt == 64) {
#pragma unroll
    for (int l = 0; l < 64; ++l) {
      x = x * (((m >> l) & 1ull) ? c.f_in : c.f_out);
      top = fmax(x, top);
    }
  } else {
    for (int l = 0; l < cnt; ++l) {
      x = x * (((m >> l) & 1ull) ? c.f_in : c.f_out);
      top = fmax(x, top);
    }
  }
  return x;
}

// One model from pool position start (k_sprt.hip); total: its
// inliers among all n points.
__device__ WalkResult walk_pool(const Rows& R, const Chain& c, int start, int n, int total) {
  const int lane = lane_id();
  const uint64_t le = lane == 63 ? ~0ull : ((2ull << lane) - 1ull);
  const int nw = (n + 63) >> 6;
  // 64 bits of the row from position p on (zeros beyond the row)
  auto window = [&](int p) -> uint64_t {
    const int w = p >> 6, s = p & 63;
    uint64_t v = R.inl_word(w) >> s;
    if (s && w + 1 < nw) v |= R.inl_word(w + 1) << (64 - s);
    return v;
  };
  // inlier bits of the test's positions b .. b + 63
  auto word = [&](int b) -> uint64_t {
    int64_t p64 = (int64_t)start + b;
    if (p64 >= n) p64 -= n;
    const int p = (int)p64;
    uint64_t v = window(p);
    if (n - p < 64) v |= window(0) << (n - p);
    return n - b < 64 ? v & ((1ull << (n - b)) - 1ull) : v;
  };
  if (c.unit) {
    // the product stays at 1: above A at the first point, or never
    if (1.0 > c.A) return WalkResult{(int)(word(0) & 1ull), 1, true};
    return WalkResult{total, n, false};
  }
  const WalkResult all{total, n, false};
  bool exact = !c.fast;
  int count = 0;
  for (int b = 0; !exact && b < n; b += 64) {
    const int t = b + lane;
    const uint64_t m = word(b);
    const int a = count + __popcll(m & le);
    Sides s = chain_sides(c, a, t + 1 - a);
    const uint64_t live = n - b < 64 ? (1ull << (n - b)) - 1ull : ~0ull;
    const uint64_t above = s.above & live;
    const uint64_t upto = above ? ((above & -above) << 1) - 1ull : live;  // through the first stop
    if ((s.open | s.low) & upto) {
      if (!(s.open & upto) && no_return(c, n - b)) return all;
      exact = true;
      break;
    }
    if (above) return WalkResult{count + (int)__popcll(m & upto), b + (int)__ffsll((unsigned long long)above), true};
    count += __popcll(m);
  }
  if (!exact) return all;
  // the reference's chain; a word whose largest product is not above A has no
  // stop in it, and a product of zero stays there
  count = 0;
  double lambda = 1.0;
  for (int b = 0; b < n && lambda != 0.0; b += 64) {
    const uint64_t m = word(b);
    const int cnt = n - b < 64 ? n - b : 64;
    double top;
    const double x = chain_word(c, lambda, m, cnt, top);
    if (top > c.A) {
      double y = lambda;
      for (int l = 0; l < cnt; ++l) {
        y = y * (((m >> l) & 1ull) ? c.f_in : c.f_out);
        if (y > c.A) return WalkResult{count + (int)__popcll(m & ((2ull << l) - 1ull)), b + l + 1, true};
      }
    }
    lambda = x;
    count += __popcll(m);
  }
  return all;
}

// One model over its kept cells (preemption_sprt.h:241-258): a rejection
// leaves only the current cell, and the following cells are tested from the
// last accepted ratio.  RECORD: the tested inliers' bits go to rec.
//
// When a point's factor exceeds A it is not kept, so the ratio stays where a
// factor of the same kind exceeds A again while one of the other kind (on the
// other side of 1) does not.  Every following cell that begins with a point of
// that kind is therefore left at its first point, and the walk goes straight
// to the next kept cell that begins with a point of the other kind.
template <bool RECORD>
__device__ WalkResult walk_cells(const Rows& R, const Chain& c, int n, int total, uint64_t* rec) {
  const int lane = lane_id();
  const uint64_t le = lane == 63 ? ~0ull : ((2ull << lane) - 1ull);
  const int nw = (n + 63) >> 6;
  int count = 0, rejected = 0;
  int exact = !c.fast || c.unit;
  if (c.unit && !uni(1.0 > c.A)) {
    if constexpr (RECORD)
      for (int w = lane; w < nw; w += 64) rec[w] = w < 64 ? R.inl : R.g_inl[w];
    return WalkResult{total, n, false};
  }
  int A0 = 0, B0 = 0;  // the accepted factors
  int sunk = 0;        // the ratio cannot climb back to A: only the count is left
  int left = 0;        // the last cell was left by an outlier (1) or an inlier (2)
  for (int w0 = 0; w0 < nw && !exact; w0 += 64) {
    // this block's words, one per lane
    uint64_t kw = 0, iw = 0, sw = 0, hitw = 0;
    if (w0 == 0) {
      kw = R.keep;
      iw = R.inl;
      sw = R.start;
    } else if (w0 + lane < nw) {
      kw = R.g_keep[w0 + lane];
      iw = R.g_inl[w0 + lane];
      sw = R.g_start[w0 + lane];
    }
    const uint64_t first = kw & sw;  // the kept cells' first positions
    const int we = nw - w0 < 64 ? nw - w0 : 64;
    int w = 0, bit = 0;  // the next position of the block
    while (w < we) {
      if (left) {
        // to the next kept cell that begins with a point of the other kind;
        // the inliers that the cells before it are left at count
        const uint64_t from = lane < w ? 0ull : (lane == w ? ~0ull << bit : ~0ull);
        const uint64_t ev = first & (left == 2 ? ~iw : iw) & from;
        const uint64_t has = ballot64(ev != 0);
        const int l = has ? __ffsll((unsigned long long)has) - 1 : 64;
        const uint64_t evw = has ? uni((uint64_t)readlane_i64((int64_t)ev, l)) : 0ull;
        if (left == 2) {
          const uint64_t upto = lane < l ? ~0ull : (lane == l ? (evw & -evw) - 1ull : 0ull);
          hitw |= first & iw & from & upto;
        }
        if (!has) break;
        left = 0;
        w = l;
        bit = __ffsll((unsigned long long)evw) - 1;
      }
      const uint64_t k = uni((uint64_t)readlane_i64((int64_t)kw, w)) & (~0ull << bit);
      const uint64_t in = uni((uint64_t)readlane_i64((int64_t)iw, w)) & k;
      uint64_t above = 0, upto = k;
      if (!sunk) {
        Sides s = chain_sides(c, A0 + __popcll(in & le), B0 + __popcll(k & ~in & le));
        above = s.above & k;
        if (above) upto = k & (((above & -above) << 1) - 1ull);
        if ((s.open | s.low) & upto) {
          if ((s.open & upto) || !no_return(c, n - 64 * (w0 + w))) {
            exact = 1;
            break;
          }
          sunk = 1;
          above = 0;
          upto = k;
        }
      }
      if (lane == w) hitw |= in & upto;
      if (above) {
        const uint64_t at = above & -above, before = at - 1ull;  // the factor that exceeded A is not kept
        rejected = 1;
        left = (in & at) ? 2 : 1;
        A0 += __popcll(in & before);
        B0 += __popcll(k & ~in & before);
        bit = __ffsll((unsigned long long)above);
        w += bit >> 6;
        bit &= 63;
      } else {
        A0 += __popcll(in);
        B0 += __popcll(k & ~in);
        bit = 0;
        ++w;
      }
    }
    if (exact) break;
    count += wave_sum_i32(__popcll(hitw));
    if constexpr (RECORD)
      if (w0 + lane < nw) rec[w0 + lane] = hitw;
  }
  if (!exact) return WalkResult{uni(count), n, rejected != 0};
  // the reference's chain
  WalkResult r{0, n, false};
  double lambda = 1.0;
  bool broken = false;  // the current cell was left
  for (int w0 = 0; w0 < nw; w0 += 64) {
    uint64_t kw = 0, iw = 0, sw = 0, hitw = 0;
    if (w0 == 0) {
      kw = R.keep;
      iw = R.inl;
      sw = R.start;
    } else if (w0 + lane < nw) {
      kw = R.g_keep[w0 + lane];
      iw = R.g_inl[w0 + lane];
      sw = R.g_start[w0 + lane];
    }
    const int we = nw - w0 < 64 ? nw - w0 : 64;
    for (int w = 0; w < we; ++w) {
      const uint64_t k = (uint64_t)readlane_i64((int64_t)kw, w), in = (uint64_t)readlane_i64((int64_t)iw, w) & k;
      const uint64_t st = (uint64_t)readlane_i64((int64_t)sw, w);
      uint64_t hit = 0, todo = k;
      if (broken) {
        // the rest of the cell that was left
        if (st == 0) continue;
        todo &= ~((st & -st) - 1ull);
        broken = false;
      }
      if (lambda == 0.0) {
        hit = in & todo;  // no stop any more
        todo = 0;
      }
      while (todo) {
        const uint64_t at = todo & -todo;
        todo &= todo - 1ull;
        const bool inlier = (in & at) != 0;
        const double next = lambda * (inlier ? c.f_in : c.f_out);
        if (inlier) hit |= at;
        if (next > c.A) {
          r.rejected = true;
          const uint64_t later = st & ~(at | (at - 1ull));  // the cells that begin after this point
          if (later) {
            todo &= ~((later & -later) - 1ull);
          } else {
            todo = 0;
            broken = true;
          }
        } else {
          lambda = next;
        }
      }
      r.count += __popcll(hit);
      if (lane == w) hitw = hit;
    }
    if constexpr (RECORD)
      if (w0 + lane < nw) rec[w0 + lane] = hitw;
  }
  return r;
}

}  // namespace

}  // namespace gcr
