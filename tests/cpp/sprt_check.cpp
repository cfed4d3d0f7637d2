// Host checks of the SPRT walk: its rules (csrc/sprt_rules.hpp) and the walk
// itself (csrc/dev_sprt.hpp), the headers that the kernels are built from.  The
// walk's 64 lanes run as 64 contexts that meet at every wave operation.  Prints one
// line of counts and returns 0, or names the first case that fails.
#include <ucontext.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <limits>
#include <random>
#include <vector>

#define __device__
#define __forceinline__ inline
#define __popcll __builtin_popcountll
#define __ffsll __builtin_ffsll

namespace gcr {

// ---- a wavefront of contexts ---------------------------------------------------
struct Wave {
  static constexpr size_t kStack = 64 * 1024;
  ucontext_t home, lane[64];
  std::vector<char> stacks = std::vector<char>(64 * kStack);
  int cur = 0;
  bool done[64];
  int met[64];              // wave operations of each lane so far
  uint64_t value[2][64];    // of this operation and, still being read, the last
  std::function<void()> body;

  static Wave& get() {
    static Wave w;
    return w;
  }
  static void entry() {
    Wave& w = get();
    w.body();
    w.done[w.cur] = true;
    swapcontext(&w.lane[w.cur], &w.home);
  }
  // Runs f on the 64 lanes; every lane takes part in every operation.
  void run(std::function<void()> f) {
    body = std::move(f);
    for (int l = 0; l < 64; ++l) {
      getcontext(&lane[l]);
      lane[l].uc_stack.ss_sp = stacks.data() + (size_t)l * kStack;
      lane[l].uc_stack.ss_size = kStack;
      lane[l].uc_link = nullptr;
      makecontext(&lane[l], (void (*)())entry, 0);
      done[l] = false;
      met[l] = 0;
    }
    for (;;) {
      int running = 0;
      for (cur = 0; cur < 64; ++cur)
        if (!done[cur]) {
          swapcontext(&home, &lane[cur]);
          running += done[cur] ? 0 : 1;
        }
      if (running == 0) return;
      if (running != 64) {
        std::printf("FAIL lanes part at a wave operation\n");
        std::exit(1);
      }
    }
  }
  // the values that all lanes bring to their next operation
  const uint64_t* meet(uint64_t v) {
    const int l = cur, at = met[l]++ & 1;
    value[at][l] = v;
    swapcontext(&lane[l], &home);
    return value[at];
  }
};

inline int lane_id() { return Wave::get().cur; }
inline uint64_t ballot64(bool p) {
  const uint64_t* v = Wave::get().meet(p ? 1 : 0);
  uint64_t m = 0;
  for (int l = 0; l < 64; ++l) m |= v[l] << l;
  return m;
}
inline int64_t readlane_i64(int64_t x, int l) { return (int64_t)Wave::get().meet((uint64_t)x)[l]; }
inline uint64_t uni(uint64_t x) { return Wave::get().meet(x)[0]; }
inline int uni(int x) { return (int)(int64_t)Wave::get().meet((uint64_t)(int64_t)x)[0]; }
inline int wave_sum_i32(int x) {
  const uint64_t* v = Wave::get().meet((uint64_t)(int64_t)x);
  int64_t s = 0;
  for (int l = 0; l < 64; ++l) s += (int64_t)v[l];
  return (int)s;
}

}  // namespace gcr

#include "dev_sprt.hpp"

using namespace gcr;

#define CHECK(cond, ...)          \
  do {                            \
    if (!(cond)) {                \
      std::printf("FAIL %s: ", #cond); \
      std::printf(__VA_ARGS__);   \
      std::printf("\n");          \
      std::exit(1);               \
    }                             \
  } while (0)

// Every window of a walk launch is a grid that HIP accepts (fewer than 2^32
// threads, 256 per workgroup), holds a model, and its rows fit the scratch.
static void check_plan() {
  long plans = 0, capped = 0;
  for (int items : {1, 7, 64, 300, 512, 1024, 65535, 1 << 20, 3 << 21})
    for (int n : {1, 63, 64, 65, 4096, 100000})
      for (int slots : {1, 7, 8, 256, 257, 30000, 655360, 1 << 26})
        for (int64_t budget : {(int64_t)1, (int64_t)4096, (int64_t)(32 << 20)}) {
          if ((int64_t)items * ((n + 63) / 64) > (64 << 20)) continue;  // no batch of that size fits the card
          const SprtPlan p = sprt_plan(items, n, slots, budget);
          const int64_t blocks = (int64_t)p.max_window * items;
          CHECK(p.max_window >= 1 && p.max_window <= slots, "items %d n %d slots %d window %d", items, n, slots,
                p.max_window);
          CHECK(blocks * 256 < ((int64_t)1 << 32), "items %d n %d slots %d window %d", items, n, slots, p.max_window);
          CHECK(p.words == (n + 63) / 64, "words");
          // the launch's layout: start and record rows, then of the window's
          // models inlier and kept rows, values, two 32-bit counts
          const size_t rows = (size_t)p.words * items;
          CHECK(p.scratch_words >= 2 * rows + 2 * rows * p.max_window + 2 * (size_t)p.max_window * items,
                "items %d n %d slots %d: %zu words", items, n, slots, p.scratch_words);
          const int64_t bits = 2 * (int64_t)p.words * items * p.max_window;
          CHECK(bits <= budget || p.max_window <= 8, "items %d n %d slots %d: %lld words of rows", items, n, slots,
                (long long)bits);
          ++plans;
          if (p.max_window < slots && p.max_window > 8 && bits < budget / 2) ++capped;
        }
  CHECK(plans > 500 && capped > 0, "%ld plans, %ld bound by the grid", plans, capped);
  std::printf("plans %ld bound by the grid %ld\n", plans, capped);
}

// ---- the walk against the reference's loop ---------------------------------------

static Chain host_chain(double eps, double delta, double A, int n) {
  Chain c;
  c.f_in = delta / eps;
  c.f_out = (1 - delta) / (1 - eps);
  c.A = A;
  c.l_in = std::log(c.f_in);
  c.l_out = std::log(c.f_out);
  c.l_A = std::log(A);
  chain_band(c, n);
  return c;
}

// preemption_sprt.h:299-330
static double threshold(double eps, double delta, double m, double ms) {
  const double C = (1 - delta) * std::log((1 - delta) / (1 - eps)) + delta * std::log(delta / eps);
  const double K = 1.0 / m * C / ms + 1.0;
  double prev = K, a = K;
  for (int i = 0; i < 10; ++i) {
    a = K + std::log(prev);
    if (std::fabs(a - prev) < 1.5e-8) break;
    prev = a;
  }
  return a;
}

struct Case {
  int n, start;
  double eps, delta, A;
  std::vector<uint8_t> inl, keep, first;  // by position; first: a cell begins
};

// One factor at a time in pool order from position start.
static WalkResult plain_pool(const Case& k, const Chain& c) {
  WalkResult r{0, 0, false};
  double lambda = 1.0;
  for (int t = 0; t < k.n && !r.rejected; ++t) {
    const int pos = (k.start + t) % k.n;
    lambda = lambda * (k.inl[pos] ? c.f_in : c.f_out);
    r.count += k.inl[pos];
    ++r.tested;
    r.rejected = lambda > c.A;
  }
  return r;
}

// One factor at a time over the kept cells: a factor that exceeds A is not kept
// and leaves its cell.
static WalkResult plain_cells(const Case& k, const Chain& c, std::vector<uint8_t>& hits) {
  WalkResult r{0, k.n, false};
  hits.assign(k.n, 0);
  double lambda = 1.0;
  bool left = false;
  for (int p = 0; p < k.n; ++p) {
    if (k.first[p]) left = false;
    if (!k.keep[p] || left) continue;
    const double next = lambda * (k.inl[p] ? c.f_in : c.f_out);
    r.count += k.inl[p];
    hits[p] = k.inl[p];
    if (next > c.A) {
      r.rejected = true;
      left = true;
    } else {
      lambda = next;
    }
  }
  return r;
}

static std::vector<uint64_t> pack(const std::vector<uint8_t>& v) {
  std::vector<uint64_t> w((v.size() + 63) / 64, 0);
  for (size_t i = 0; i < v.size(); ++i) w[i / 64] |= (uint64_t)(v[i] != 0) << (i % 64);
  return w;
}

static Case make_case(std::mt19937_64& rng, bool cells) {
  std::uniform_real_distribution<double> u(0.0, 1.0);
  auto log10u = [&](double lo, double hi) { return std::pow(10.0, lo + (hi - lo) * u(rng)); };
  Case k;
  const int sizes[] = {1, 2, 63, 64, 65, 127, 128, 129, 4095, 4096, 4097, 4161};
  k.n = rng() % 4 == 0 ? sizes[rng() % (cells ? 12 : 11)] : 1 + (int)(rng() % (rng() % 8 == 0 ? 6000 : 700));
  k.start = (int)(rng() % k.n);
  k.eps = rng() % 6 == 0 ? (double)(1 + rng() % k.n) / k.n : log10u(-5, -0.02);
  switch (rng() % 7) {
    case 0: k.delta = k.eps; break;
    case 1: k.delta = k.eps * (1 + 1e-13); break;
    case 2: k.delta = k.eps / 10; break;
    case 3: k.delta = (double)(1 + rng() % k.n) / k.n; break;
    default: k.delta = log10u(-5, -0.02);
  }
  const double rates[] = {0.0, 0.02, k.delta, k.eps, 0.5, 0.9, 1.0};
  const double rate = rates[rng() % 7];
  k.inl.resize(k.n);
  for (auto& b : k.inl) b = u(rng) < rate;
  if (rng() % 4 == 0) {
    // long runs of inliers and outliers under a high epsilon: products that
    // sink far and climb back
    k.eps = 1.0 - log10u(-6, -1);
    k.delta = log10u(-3, -0.3);
    bool in = rng() % 2;
    for (int p = 0, run = 0; p < k.n; ++p, --run) {
      if (run == 0) {
        run = 1 + (int)(rng() % (rng() % 2 ? 64 : k.n));
        in = !in;
      }
      k.inl[p] = in;
    }
  }
  k.keep.assign(k.n, 1);
  k.first.assign(k.n, 0);
  if (cells) {
    const double mean = log10u(0, 2.5), kept = u(rng) < 0.3 ? 1.0 : u(rng);
    bool kp = true;
    for (int p = 0; p < k.n; ++p) {
      k.first[p] = p == 0 || u(rng) < 1.0 / mean;
      if (k.first[p]) kp = u(rng) < kept;
      k.keep[p] = kp;
    }
  }
  const double inf = std::numeric_limits<double>::infinity();
  switch (rng() % 12) {
    case 0: k.A = log10u(-3, 3); break;
    case 1: k.A = 1.0; break;
    case 2: {  // exactly a product on the way
      const Chain c = host_chain(k.eps, k.delta, 1.0, k.n);
      double x = 1.0;
      const int upto = 1 + (int)(rng() % k.n);
      for (int t = 0; t < upto; ++t) {
        const int p = cells ? t : (k.start + t) % k.n;
        if (k.keep[p]) x *= k.inl[p] ? c.f_in : c.f_out;
      }
      k.A = x;
      break;
    }
    case 3: {
      const double odd[] = {inf, std::nan(""), 0.0, -1.0, 1e300, 1e-300};
      k.A = odd[rng() % 6];
      break;
    }
    default: k.A = threshold(k.eps, k.delta, 7, 3);
  }
  return k;
}

static void check_walk(bool cells, int trials) {
  std::mt19937_64 rng(cells ? 5 : 3);
  long rejected = 0, accepted = 0, jumps = 0, exact = 0, sunk = 0;
  for (int trial = 0; trial < trials; ++trial) {
    const Case k = make_case(rng, cells);
    const Chain c = host_chain(k.eps, k.delta, k.A, k.n);
    const std::vector<uint64_t> inl = pack(k.inl), keep = pack(k.keep), first = pack(k.first);
    std::vector<uint8_t> both(k.n);
    for (int p = 0; p < k.n; ++p) both[p] = k.inl[p] && (!cells || k.keep[p]);
    const std::vector<uint64_t> rows = cells ? pack(both) : inl;
    int total = 0;
    for (uint8_t b : both) total += b;
    std::vector<uint8_t> hits;
    const WalkResult want = cells ? plain_cells(k, c, hits) : plain_pool(k, c);
    WalkResult got[64];
    std::vector<uint64_t> rec(rows.size(), 0);
    Wave::get().run([&] {
      const size_t l = (size_t)lane_id();
      Rows R;
      R.inl = l < rows.size() ? rows[l] : 0;
      R.keep = cells && l < keep.size() ? keep[l] : 0;
      R.start = cells && l < first.size() ? first[l] : 0;
      R.g_inl = rows.data();
      R.g_keep = keep.data();
      R.g_start = first.data();
      got[l] = cells ? walk_cells<true>(R, c, k.n, total, rec.data()) : walk_pool(R, c, k.start, k.n, total);
    });
    for (int l = 0; l < 64; ++l)
      CHECK(got[l].count == want.count && got[l].rejected == want.rejected && got[l].tested == want.tested,
            "%s trial %d lane %d: n %d start %d eps %.17g delta %.17g A %.17g: count %d/%d tested %d/%d rejected %d/%d",
            cells ? "cells" : "pool", trial, l, k.n, k.start, k.eps, k.delta, k.A, got[l].count, want.count,
            got[l].tested, want.tested, (int)got[l].rejected, (int)want.rejected);
    if (cells) CHECK(rec == pack(hits), "trial %d: recorded inliers", trial);
    (want.rejected ? rejected : accepted) += 1;
    jumps += cells && want.rejected && want.count < total;
    exact += !c.fast || c.unit;
    const double least = total * c.l_in + (k.n - total) * c.l_out;
    sunk += c.fast && least < -700.0;
  }
  CHECK(rejected > trials / 10 && accepted > trials / 10 && exact > 0 && sunk > 0 && (!cells || jumps > 0),
        "%ld %ld %ld %ld %ld", rejected, accepted, jumps, exact, sunk);
  std::printf("%s: rejected %ld accepted %ld left with inliers behind %ld no logarithms %ld sunk %ld\n",
              cells ? "cells" : "pool", rejected, accepted, jumps, exact, sunk);
}

int main(int argc, char** argv) {
  const char* what = argc > 1 ? argv[1] : "";
  if (!std::strcmp(what, "plan")) {
    check_plan();
  } else if (!std::strcmp(what, "pool")) {
    check_walk(false, 10000);
  } else if (!std::strcmp(what, "cells")) {
    check_walk(true, 4000);
  } else {
    std::printf("usage: sprt_check plan|pool|cells\n");
    return 2;
  }
  return 0;
}
