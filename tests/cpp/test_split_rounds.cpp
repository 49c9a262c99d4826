// CPU check of the cut of marches and walks into chunks
// (miso_amd/csrc/split_rounds.hpp): for many lengths and loads the chosen
// count is the one that a scan of every count up to n chooses, and the call's
// time stays far below a launch's.  Built by tests/cpp/Makefile with g++; run
// by tests/test_split_rounds.py.
#include <chrono>
#include <cmath>
#include <cstdio>
#include <initializer_list>

#include "../../miso_amd/csrc/split_rounds.hpp"

namespace {

// every count in turn, as the rule states it
void scan(int n, long per_chunk, int most, long slots, double start, double even, int &chunk,
          int &nchunks) {
  const int least = most < 1 ? 1 : most;
  double best = 0.0, rounds = 0.0;
  nchunks = 0;
  for (int m = (n + least - 1) / least; m <= n && rounds <= even; ++m) {
    const int c = (n + m - 1) / m;
    if ((n + c - 1) / c != m) continue;  // the same length as fewer chunks'
    const double full = (double)per_chunk * m / slots;
    const double cost = (full <= even ? std::ceil(full) : full + 0.5) * (c + start);
    if (nchunks && cost > 0.98 * best) continue;
    best = cost;
    rounds = full;
    chunk = c;
    nchunks = m;
  }
}

// the launches' rules: slots, start, even
const struct { long slots; double start, even; } RULES[] = {
    {256, 4.0, 2.0}, {768, 4.0, 2.0}, {256, 5.0, 4.0}, {256, 2.5, 4.0}, {512, 2.5, 4.0}};

}  // namespace

// 0: every choice equal; calls receives how many were compared
extern "C" int split_rounds_check(char *msg, int len, int *calls) {
  for (const auto &r : RULES)
    for (int n = 1; n < 70000; n += 1 + n / 9)
      for (long per = 1; per < 3000; per += 1 + per / 3)
        for (int most : {1, 4, 16, 64, 128, 256, 4096}) {
          int a, b, na, nb;
          scan(n, per, most, r.slots, r.start, r.even, a, na);
          misohip::split_rounds(n, per, most, r.slots, r.start, r.even, b, nb);
          ++*calls;
          if (a != b || na != nb) {
            std::snprintf(msg, len, "n %d, %ld blocks, most %d, %ld slots: %d x %d, scan %d x %d",
                          n, per, most, r.slots, nb, b, na, a);
            return 1;
          }
        }
  return 0;
}

// the least time of one call, in microseconds, over a few tries
extern "C" double split_rounds_time(int n, long per_chunk, int most, long slots) {
  double best = 1e30;
  for (int t = 0; t < 7; ++t) {
    int c = 0, m = 0;
    volatile long sink = 0;
    const auto t0 = std::chrono::steady_clock::now();
    for (int i = 0; i < 50; ++i) {
      misohip::split_rounds(n, per_chunk, most, slots, 4.0, 2.0, c, m);
      sink += c;
    }
    const std::chrono::duration<double, std::micro> d = std::chrono::steady_clock::now() - t0;
    best = std::fmin(best, d.count() / 50);
  }
  return best;
}

// the longest walk of a y or z sweep over rows of ni cells
extern "C" int walk_limit_of(int ni, int most, int f64) {
  return misohip::walk_limit(ni, most, f64 != 0);
}

// rows and chunks of the x-y walk
extern "C" void split_xy_of(int nj, int nseg, int npl, int nparts, int most, int *out) {
  misohip::split_xy(nj, nseg, npl, nparts, most, out[0], out[1]);
}
