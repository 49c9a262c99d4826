// How a march or walk is cut into chunks (host code, no HIP).
#pragma once

#include <cmath>

namespace misohip {

// Chunks of a march or walk over n cells, none longer than `most`, in a
// launch of per_chunk blocks each: of all counts the one with the least
// rounds x length, where `slots` blocks run at a time and each costs `start`
// cells more than it covers (its first window is loaded, and its first slopes
// formed, anew).  The last round of a launch is then nearly full, and a small
// grid is spread over the chip as far as the repeated cells allow.  Past
// `even` rounds the blocks no longer end together: half a round is lost at the
// end, and nothing is gained by more chunks (the FP32 z walk of 512^3, 2.7
// rounds of 256 planes: 3.1 ms; 4 of 171: 3.3).  Every chunk starts from the
// fields, so the results do not depend on the split.
//   Only counts with a length of their own are looked at, and none once even a
// full last round could not win: m chunks cost at least the rounds they need
// times the cells they walk, per_chunk / slots x (n + m start).  This runs at
// every launch: 0.3 us for 256 cells, 1.7 for 100000 (every count up to n: 1.3
// and 450).
inline void split_rounds(int n, long per_chunk, int most, long slots, double start, double even,
                         int &chunk, int &nchunks) {
  const int least = most < 1 ? 1 : most;
  const double load = (double)per_chunk / slots;
  double best = 0.0, rounds = 0.0;
  nchunks = 0;
  for (int m = (n + least - 1) / least; m <= n && rounds <= even;) {
    if (nchunks && load * (n + m * start) > best) break;
    const int c = (n + m - 1) / m;
    const double full = (double)per_chunk * m / slots;
    const double cost = (full <= even ? std::ceil(full) : full + 0.5) * (c + start);
    if (!nchunks || cost <= 0.98 * best) {
      best = cost;
      rounds = full;
      chunk = c;
      nchunks = m;
    }
    if (c == 1) break;
    m = (n + c - 2) / (c - 1);  // the fewest chunks shorter than these
  }
}

// Longest walk of the y and z sweeps whose last 64-cell segment along x holds
// `ni` cells or the rest of them.  A wave of at most eight lanes takes 4.8 us a
// plane of a long walk where one of twelve or more takes 1.5 to 2.7 (512 x 512
// rows, 256 planes, FP64; the cause was not found), and less in short ones: z
// sweep of 4 x 512 x 512 1240 us in walks of 256, 830 of 64, 740 of 16 (FP32
// 450, 345, 285); of 12 x 512 x 512 382, 382, 439.  Beside whole segments the
// narrow one is the last to end in FP64: 72 x 512 x 512 2220 us in walks of
// 256, 958 of 128, 934 of 64; 65 x 200 x 600 395, 395, 409 (FP32, 72 x 512 x
// 512: 538, 547, 534; 260^3: 446, 489, 441).
//   Walks of narrow rows alone are cut for four times the blocks that run at a
// time as well (steps of 1 x 100 x 100 in FP64 379 -> 356 us, of 1 x 18 x 649 391
// -> 360, of 8 x 4096 in FP32 105 -> 95).
constexpr int WALK_NARROW = 8, WALK_NARROW_ALONE = 16, WALK_NARROW_LAST = 128;
constexpr int WALK_NARROW_SLOTS = 4;
inline int walk_limit(int ni, int most, bool f64) {
  if ((ni - 1) % 64 + 1 > WALK_NARROW || (ni > 64 && !f64)) return most;
  const int limit = ni > 64 ? WALK_NARROW_LAST : WALK_NARROW_ALONE;
  return most < limit ? most : limit;
}

// The x-y walk over nj rows: nseg waves for each of npl planes, four a block.
// More than one of its blocks fits a CU, but it is bound by VALU issue, so that
// what counts is how evenly they fall on the CUs.  Against walks halved until
// the launch had 2^18 threads, at 64^3 and 205 x 131 x 93 in FP64: 61 -> 49 and
// 229 -> 198 us.
//   A launch of nparts planes, one slab of the overlapped walks, is cut by its
// own blocks where those of the whole walk's cut would leave CUs idle (overlapped
// FP32 step of 128^3 1237 -> 685 us, of 96^3 1211 -> 536, FP64 of 64^3 878 ->
// 492; 256^3, whose slabs fill the chip, 5.61 ms either way).
constexpr int XY_SLOTS = 256;
constexpr double XY_START = 5.0;
inline void split_xy(int nj, int nseg, int npl, int nparts, int most, int &chunk, int &nchunks) {
  auto cut = [&](int planes) {
    split_rounds(nj, ((long)nseg * planes + 3) / 4, most, XY_SLOTS, XY_START, 4.0, chunk, nchunks);
  };
  cut(npl);
  if (nparts && ((long)nseg * nchunks * nparts + 3) / 4 < XY_SLOTS) cut(nparts);
}

}  // namespace misohip
