// Host checks of the SPRT walk's rules (csrc/sprt_rules.hpp).  Prints one line
// of counts and returns 0, or names the first case that fails.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "sprt_rules.hpp"

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

int main(int argc, char** argv) {
  const char* what = argc > 1 ? argv[1] : "";
  if (!std::strcmp(what, "plan")) {
    check_plan();
  } else {
    std::printf("usage: sprt_check plan\n");
    return 2;
  }
  return 0;
}
