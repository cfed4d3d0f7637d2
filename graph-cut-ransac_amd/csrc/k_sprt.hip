// SPRT preemptive verification (preemption_sprt.h:218-296) of a pair's
// candidate models, in the order the main loop meets them.
//
// The test is sequential twice over: each model walks the pair's points in
// the order of a random pool, starting where the previous model stopped,
// and multiplies a likelihood ratio point by point until it exceeds the
// decision threshold A; and the test's parameters (delta, A) change after a
// rejection that moves the estimated delta by more than 5 %.  What does not
// depend on that order are the inlier decisions themselves, so the walk is
// split in two kernels:
//   k_sprt_masks  every listed model against every point of its pair, four
//                 waves per model: one inlier bit per position of the test
//                 order (the pool, or the space partitioning cells' order);
//   k_sprt_walk   one wavefront per pair steps through the models on those
//                 bits, 64 positions at a time.
// The models of a walk are taken in windows (a mask and a walk launch each),
// so a walk that stops early leaves the later models' masks unmade and the
// mask memory is bounded.
//
// A after a delta change comes from a table the host fills for the current
// epsilon (A for delta = k / N, k = 0..N), so every logarithm that enters a
// result is the host C library's.  The walk stops at the first accepted model
// whose score beats the best value given: the host then makes the
// reference's epsilon update, the validity check and the best-model update,
// and continues the walk.
//
// The ratio's chain on 64 positions at once.  After a inliers and b outliers
// the reference's running product is f_in^a f_out^b up to a relative error of
// (a + b) 2^-53, so "the product exceeds A" is a log f_in + b log f_out >
// log A unless the two sides are within a margin of that rounding and of the
// logarithms'.  Each lane forms the sum for its own position from a popcount
// of the bits before it; the first lane above log A is where the reference
// stops.  A model with a position inside the margin before its stop, or with a
// non-finite logarithm, is walked again by the reference's chain, one
// multiplication per position, so every decision is the reference's.  So is a
// model whose product comes near the subnormal range (a model with many
// inliers under a small delta: the usual good model), unless the positions
// left are too few for the ratio to climb back; there the chain ends as soon
// as the product is zero, from which it never returns.
//
// Value of an accepted model: the mask kernel sums every model's terms in
// parallel, so only a model that can beat the best value (within the two
// sums' rounding) is summed in the reference's order.
//
// What bounds it: the walk is a serial chain of models, one wavefront per
// pair, so it is bound by the latency of a few dozen dependent scalar and
// vector instructions per 64 positions (or per cell the walk stops in), plus
// the divisions and logarithms of a delta change; the masks take 12 us per
// window.  Measured on MI355X, one call with the API's defaults: the walk
// that evaluated residuals and stepped position by position took 148.7 ms of
// a findHomography call's 151.0 ms of kernels (2,000 points, 50 % inliers) and
// 50.4 of 52.6 ms for a fundamental matrix (3,001 points); this one 7.4 ms
// and 2.7 ms.
#include "dev_common.hpp"
#include "dev_sp.hpp"
#include "dev_sprt.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace gcr {

namespace {

constexpr int kMaskThreads = 256;

// The ratio's factors and their logarithms (lanes 0, 1, 2 take one logarithm
// each).
__device__ Chain make_chain(double eps, double delta, double A, int n) {
  Chain c;
  c.f_in = delta / eps;
  c.f_out = (1 - delta) / (1 - eps);
  c.A = A;
  const int lane = lane_id();
  const double l = log(lane == 0 ? c.f_in : (lane == 1 ? c.f_out : A));
  c.l_in = readlane_f64(l, 0);
  c.l_out = readlane_f64(l, 1);
  c.l_A = readlane_f64(l, 2);
  chain_band(c, n);
  c.unit = uni(c.unit);
  c.fast = uni(c.fast);
  return c;
}

}  // namespace

// One workgroup per (item, slot of the window; live of them used).  Position e of item i's test
// order is point order[e]; bit e of row (item win + j) is set when that point is
// an inlier of the window's slot j; inl_count and approx: the number of set bits
// and the sum of their terms in any order.  Space partitioning items also get the
// row of kept positions, the kept point count and (once per item) the row of
// the cells' first positions.
__global__ void __launch_bounds__(kMaskThreads)
    k_sprt_masks(const SprtItem* __restrict__ items, int win_base, int win, int live, const double* __restrict__ pts,
                 const int64_t* __restrict__ pair_pt_off, const int32_t* __restrict__ pair_n,
                 const double* __restrict__ pair_sq_thr, const int32_t* __restrict__ pools,
                 const SpPair* __restrict__ sp_pairs, const SpCell* __restrict__ sp_cells,
                 const int32_t* __restrict__ sp_perm, const int32_t* __restrict__ sp_cell_of, int words,
                 uint64_t* __restrict__ inl_bits, uint64_t* __restrict__ keep_bits, uint64_t* __restrict__ start_bits,
                 int32_t* __restrict__ kept_count, int32_t* __restrict__ inl_count,
                 double* __restrict__ approx) {
  // a bit per cell: the 48 bytes beside it leave room for every cell count that
  // the selector's other kernels hold in LDS, a byte each
  extern __shared__ uint64_t keep[];
  __shared__ int32_t part[kMaskThreads / 64];
  __shared__ double vpart[kMaskThreads / 64];
  const int item = (int)(blockIdx.x / (unsigned)live), j = (int)(blockIdx.x % (unsigned)live);
  const SprtItem& it = items[item];
  const int s = win_base + j;
  if (it.stop >= 0 || s >= it.num_slots) return;
  const int pair = it.pair;
  const int64_t base = pair_pt_off[pair];
  const int n = pair_n[pair];
  const double sq = pair_sq_thr[pair];
  const double* __restrict__ P = pts + 4 * base;
  const double* __restrict__ mp = it.models + 9 * (int64_t)it.slots[s];
  double M[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) M[k] = mp[k];
  const int lane = lane_id(), wave = threadIdx.x >> 6;
  const int64_t row = ((int64_t)item * win + j) * words;
  const int nw = (n + 63) >> 6;
  double value = 0.0;
  int32_t inliers = 0;
  if (it.sp) {
    const SpPair sp = sp_pairs[pair];
    const SpCell* __restrict__ cells = sp_cells + sp.cell_off;
    const int32_t* __restrict__ cell_of = sp_cell_of + base;
    const bool any = !(fabs(sp_det3(M)) < 1e-3);
    int32_t cnt = 0;
    for (int c0 = 64 * wave; c0 < sp.ncells; c0 += kMaskThreads) {
      const int c = c0 + lane;
      bool k = false;
      if (c < sp.ncells) {
        const SpCell cell = cells[c];
        k = any && sp_keep(M, cell, sp);
        if (k) cnt += cell.len;
      }
      const uint64_t b = ballot64(k);
      if (lane == 0) keep[c0 >> 6] = b;
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) cnt += __shfl_xor(cnt, d, 64);
    if (lane == 0) part[wave] = cnt;
    __syncthreads();
    const int32_t kept = part[0] + part[1] + part[2] + part[3];
    if (threadIdx.x == 0) kept_count[(int64_t)item * win + j] = kept;
    const bool starts = j == 0;
    const bool tested = kept >= it.best_count;  // else the walk skips the model
    if (!tested && !starts) return;
    for (int w = wave; w < nw; w += kMaskThreads / 64) {
      const int e = 64 * w + lane;
      bool kp = false, inl = false, first = false;
      if (e < n) {
        const int c = cell_of[e];
        kp = (keep[c >> 6] >> (c & 63)) & 1ull;
        if (starts) first = e == 0 || cell_of[e - 1] != c;
        if (kp && tested) {
          const double r2 = h_sq_residual(P + 4 * (int64_t)sp_perm[base + e], M);
          inl = r2 < sq;
          if (inl) value += 1.0 - r2 / sq;
        }
      }
      const uint64_t bk = ballot64(kp), bi = ballot64(inl), bs = ballot64(first);
      inliers += __popcll(bi);
      if (lane == 0) {
        keep_bits[row + w] = bk;
        inl_bits[row + w] = bi;
        if (starts) start_bits[(int64_t)item * words + w] = bs;
      }
    }
  } else {
    const int32_t* __restrict__ order = pools + base;
    for (int w = wave; w < nw; w += kMaskThreads / 64) {
      const int e = 64 * w + lane;
      bool inl = false;
      if (e < n) {
        const double* p = P + 4 * (int64_t)order[e];
        const double r2 = it.kind == 0 ? h_sq_residual(p, M) : f_sq_sampson(p, M);
        inl = r2 < sq;
        if (inl) value += 1.0 - r2 / sq;
      }
      const uint64_t b = ballot64(inl);
      inliers += __popcll(b);
      if (lane == 0) inl_bits[row + w] = b;
    }
  }
  value = wave_tree64(value);
  __syncthreads();  // part's readers above
  if (lane == 0) {
    vpart[wave] = value;
    part[wave] = inliers;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    approx[(int64_t)item * win + j] = (vpart[0] + vpart[1]) + (vpart[2] + vpart[3]);
    inl_count[(int64_t)item * win + j] = part[0] + part[1] + part[2] + part[3];
  }
}

namespace {

// Sum of 1 - r^2 / tau^2 over the set bits of an accepted model in test
// order from position start; four words' points in flight at a time.
template <class H, class R>
__device__ double ordered_value(int n, int64_t start, H has, R residual, double sq) {
  const int lane = lane_id();
  double value = 0.0;
  for (int b = 0; b < n; b += 256) {
    double term[4];
    uint64_t m[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = b + 64 * u + lane;
      bool in = false;
      term[u] = 0.0;
      if (t < n) {
        int64_t pos = start + t;
        if (pos >= n) pos -= n;
        in = has((int)pos);
        const double r2 = residual((int)pos);
        if (in) term[u] = 1.0 - r2 / sq;
      }
      m[u] = ballot64(in);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (m[u]) value = wave_chain(value, term[u], 1.0, 64 - __builtin_clzll(m[u]));
  }
  return readlane_f64(value, 0);
}

}  // namespace

// One wavefront per item: the window's models in order.  A model's words are
// fetched while the model before it is walked, the models' counts and values
// 64 models at a time.
__global__ void __launch_bounds__(64)
    k_sprt_walk(SprtItem* items, int win_base, int win, const double* __restrict__ pts,
                const int64_t* __restrict__ pair_pt_off, const int32_t* __restrict__ pair_n,
                const double* __restrict__ pair_sq_thr, const int32_t* __restrict__ pools,
                const int32_t* __restrict__ sp_perm, int words, const uint64_t* __restrict__ inl_bits,
                const uint64_t* __restrict__ keep_bits, const uint64_t* __restrict__ start_bits,
                const int32_t* __restrict__ kept_count, const int32_t* __restrict__ inl_count,
                const double* __restrict__ approx, uint64_t* rec_bits, int32_t* __restrict__ sp_list) {
  SprtItem it = items[blockIdx.x];
  if (it.stop >= 0 || win_base >= it.num_slots) return;
  const int lane = threadIdx.x;
  const int64_t base = pair_pt_off[it.pair];
  const int n = uni(pair_n[it.pair]);
  const int is_sp = uni(it.sp);
  const double sq = pair_sq_thr[it.pair];
  const double* __restrict__ P = pts + 4 * base;
  const int32_t* __restrict__ order = is_sp ? sp_perm + base : pools + base;
  const int nw = (n + 63) >> 6;
  const int left_slots = uni(it.num_slots) - win_base;
  const int end = left_slots < win ? left_slots : win;
  const int64_t row0 = (int64_t)blockIdx.x * win * words, slot0 = (int64_t)blockIdx.x * win;
  Rows R;
  R.g_start = start_bits + (int64_t)blockIdx.x * words;
  R.start = is_sp && lane < nw ? R.g_start[lane] : 0ull;
  Chain c = make_chain(it.eps, it.delta, it.A, n);
  Chain c_last = c;  // the chain the last tested model was walked with
  int last = -1;
  uint64_t p_inl = 0, p_keep = 0;
  auto fetch = [&](int j) {
    p_inl = p_keep = 0;
    if (j < end && lane < nw) {
      p_inl = inl_bits[row0 + (int64_t)j * words + lane];
      if (is_sp) p_keep = keep_bits[row0 + (int64_t)j * words + lane];
    }
  };
  auto take = [&](int j) {
    R.inl = p_inl;
    R.keep = p_keep;
    R.g_inl = inl_bits + row0 + (int64_t)j * words;
    R.g_keep = keep_bits + row0 + (int64_t)j * words;
  };
  // the next model at or after j that is tested
  int32_t g_count = 0;
  double g_value = 0.0;
  uint64_t g_tested = 0;
  int g0 = -64;
  auto next_tested = [&](int j) -> int {
    for (; j < end; j = g0 + 64) {
      if (j >= g0 + 64) {
        g0 = j & ~63;
        const bool live = g0 + lane < end;
        const int64_t s = slot0 + g0 + lane;
        const bool tested = live && (!is_sp || kept_count[s] >= it.best_count);
        g_count = tested ? inl_count[s] : 0;
        g_value = tested ? approx[s] : 0.0;
        g_tested = ballot64(tested);
      }
      const uint64_t m = g_tested & (~0ull << (j - g0));
      if (m) return g0 + __ffsll((unsigned long long)m) - 1;
    }
    return end;
  };
  int j = next_tested(0);
  fetch(j);
  while (j < end) {
    take(j);
    const int total = __builtin_amdgcn_readlane(g_count, j - g0);
    const double v = readlane_f64(g_value, j - g0);  // the value, to the rounding of two sums of n terms
    const int jn = next_tested(j + 1);
    fetch(jn);
    const int64_t start = it.pool_idx;
    const WalkResult r = is_sp ? walk_cells<false>(R, c, n, total, nullptr) : walk_pool(R, c, uni((int)start), n, total);
    last = j;
    c_last = c;
    it.last = win_base + j;
    if (!is_sp) it.pool_idx = (int)start + r.tested >= n ? start + r.tested - n : start + r.tested;
    it.last_start = is_sp ? -2 : start;
    it.last_tested = is_sp ? 0 : r.tested;
    it.last_count = r.count;
    it.last_value = 0.0;
    it.last_accepted = r.rejected ? 0 : 1;
    if (!r.rejected) {
      if (v + (1e-12 + 4e-16 * (double)n) * (1.0 + v) > it.best_value) {
        const double* __restrict__ mp = it.models + 9 * (int64_t)it.slots[win_base + j];
        double M[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) M[k] = mp[k];
        const uint64_t* __restrict__ bits = R.g_inl;
        it.last_value = ordered_value(
            n, is_sp ? 0 : start, [&](int pos) { return (bits[pos >> 6] >> (pos & 63)) & 1ull; },
            [&](int pos) {
              const double* p = P + 4 * (int64_t)order[pos];
              return it.kind == 0 ? h_sq_residual(p, M) : f_sq_sampson(p, M);
            },
            sq);
        if (it.last_value > it.best_value) {
          it.stop = win_base + j;
          break;
        }
      }
    } else {
      const double de = (double)r.count / (double)n;
      if (de > 0 && fabs(it.delta - de) / it.delta > 0.05) {
        it.delta = de;
        it.A = it.a_table[r.count];
        ++it.delta_changes;
        c = make_chain(it.eps, it.delta, it.A, n);
      }
    }
    j = jn;
  }
  if (is_sp && last >= 0) {
    // the last tested model's inliers in test order
    const int32_t total = inl_count[slot0 + last];
    p_inl = p_keep = 0;
    fetch(last);
    take(last);
    uint64_t* const rec = rec_bits + (int64_t)blockIdx.x * words;
    walk_cells<true>(R, c_last, n, total, rec);
    __syncthreads();
    int32_t* __restrict__ list = sp_list + base;
    int at = 0;
    for (int w = 0; w < nw; ++w) {
      const uint64_t m = rec[w];
      if ((m >> lane) & 1ull) list[at + __popcll(m & ((1ull << lane) - 1ull))] = order[64 * w + lane];
      at += __popcll(m);
    }
  }
  if (lane == 0) items[blockIdx.x] = it;
}

void launch_sprt_walk(hipStream_t st, SprtItem* items, int num_items, int max_slots, const SprtPlan& plan,
                      uint64_t* scratch, const double* pts, const int64_t* pair_pt_off, const int32_t* pair_n,
                      const double* pair_sq_thr, const int32_t* pools, const SpPair* sp_pairs, const SpCell* sp_cells,
                      const int32_t* sp_perm, const int32_t* sp_cell_of, int32_t* sp_list, int max_cells) {
  if (num_items <= 0 || max_slots <= 0) return;
  const int words = plan.words;
  uint64_t* const start = scratch;
  uint64_t* const rec = start + (size_t)words * num_items;
  uint64_t* const inl = rec + (size_t)words * num_items;
  // windows of 256 models, then twice as many each time up to the plan's: a
  // walk often stops early (a best model found), a late one runs to the end
  int win = std::min(256, plan.max_window);
  for (int b = 0; b < max_slots; b += win, win = std::min(2 * win, plan.max_window)) {
    uint64_t* const keep = inl + (size_t)words * num_items * win;
    double* const approx = reinterpret_cast<double*>(keep + (size_t)words * num_items * win);
    int32_t* const kept = reinterpret_cast<int32_t*>(approx + (size_t)num_items * win);
    int32_t* const count = kept + (size_t)num_items * win;
    const int live = std::min(win, max_slots - b);
    hipLaunchKernelGGL(k_sprt_masks, dim3((unsigned)live * (unsigned)num_items), dim3(kMaskThreads),
                       8 * (size_t)std::max(1, (max_cells + 63) / 64), st, items, b, win, live, pts, pair_pt_off,
                       pair_n, pair_sq_thr, pools, sp_pairs, sp_cells, sp_perm, sp_cell_of, words, inl, keep, start, kept,
                       count, approx);
    hipLaunchKernelGGL(k_sprt_walk, dim3((unsigned)num_items), dim3(64), 0, st, items, b, win, pts, pair_pt_off, pair_n,
                       pair_sq_thr, pools, sp_perm, words, inl, keep, start, kept, count, approx, rec, sp_list);
  }
}

}  // namespace gcr
