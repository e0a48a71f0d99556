// CPU check of where the compositing forward keeps its segments (jax-gs_amd/csrc/gs_segments.h),
// built and run by tests/test_segment_slots.py: whatever the lists, no two tiles' slots meet and none
// lies past the buffer; segments cover the lists, and the ends of coarser units are ends of finer ones.
//
// Output (one line): sets of lists, of which packed, faults
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "gs_segments.h"

int main(int argc, char** argv) {
  const long sets = argc > 1 ? atol(argv[1]) : 1000;
  std::mt19937_64 rng(argc > 2 ? strtoull(argv[2], nullptr, 10) : 1ull);
  auto upto = [&](int64_t hi) { return (int64_t)(rng() % (uint64_t)(hi + 1)); };
  long faults = 0, packed_sets = 0;
  for (int lu = 6; lu <= 9; ++lu) {
    for (int j = 0; j < gs::segment_count(lu); ++j) {
      const int b = gs::segment_start(j, lu), e = gs::segment_start(j + 1, lu);
      faults += !(b < e && gs::segments_within(b + 1, lu) == j + 1 && gs::segments_within(e, lu) == j + 1);
      if (lu > 6) faults += gs::segment_start(gs::segments_within(e, lu - 1), lu - 1) != e;
    }
    faults += gs::segment_start(gs::segment_count(lu), lu) != gs::kMaxTileEntries;
  }
  for (long s = 0; s < sets; ++s) {
    const int T = 1 + (int)upto(s % 3 == 0 ? 40 : gs::kFwdOneWaveTiles - 2);
    const int lu = gs::segment_shift(T);
    // lists of a few kinds of length, their sum near the capacity, above it or far below
    const int64_t longest = s % 5 == 0 ? 6000 : (s % 5 == 1 ? 1 : 1 + upto(700));
    std::vector<int64_t> ranges(T + 1, 0);
    for (int t = 0; t < T; ++t) {
      const int kind = (int)upto(3);
      const int64_t n = kind == 0 ? 0 : (kind == 1 ? longest : (kind == 2 ? upto(longest) : (1ll << lu) * upto(3) + upto(2) - 1));
      ranges[t + 1] = ranges[t] + std::max<int64_t>(0, n);
    }
    const int64_t total = ranges[T];
    const int64_t cap = std::max<int64_t>(1, s % 4 == 0 ? total : (s % 4 == 1 ? total / 2 : total + upto(4 * total + 100)));
    const bool packed = gs::segments_packed(T, cap, lu);
    const int64_t slots = gs::segment_slots(T, cap, lu);
    packed_sets += packed;
    faults += slots > (int64_t)T * gs::segment_count(lu);
    int64_t end = 0;  // of the slots of the tiles before
    for (int t = 0; t < T; ++t) {
      // as tile_span clamps them
      const int64_t b = std::min(ranges[t], cap), e = std::min(std::max(ranges[t + 1], b), cap);
      const int n = (int)std::min<int64_t>(e - b, gs::kMaxTileEntries);
      if (n == 0) continue;  // no slot is touched
      const int64_t first = gs::segment_slot(packed, t, (int)b, lu), last = first + gs::segments_within(n, lu);
      faults += !(first >= end && last <= slots);
      end = last;
    }
  }
  std::printf("%ld %ld %ld\n", sets, packed_sets, faults);
  return faults == 0 ? 0 : 1;
}
