// Index arithmetic of kernels that walk ranges of the CSR, apart from the
// kernels so that it can be run on the host at sizes no test can hold.
#pragma once

#include "choose.hpp"  // MGPM_HD

namespace mgpm {

// Lane `lane` of LANES walks the entries [b, e) of one row, UNROLL at a time:
// step(at, ok) gets the positions and which of them are in the range (the
// others repeat the first).  The range's end is what is left of it: positions
// reach 2^32 - 1, and one stepped past e from there wraps to the start of the
// array, below e, while a row has fewer than 2^31 entries.
template <uint32_t LANES, int UNROLL, class F>
MGPM_HD void lane_walk(uint32_t b, uint32_t e, uint32_t lane, const F &step) {
  uint32_t j = b + lane;
  for (int32_t left = static_cast<int32_t>(e - b - lane); left > 0;
       left -= static_cast<int32_t>(LANES * UNROLL)) {
    uint32_t at[UNROLL];
    bool ok[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const uint32_t ahead = LANES * static_cast<uint32_t>(u);
      ok[u] = left > static_cast<int32_t>(ahead);
      at[u] = ok[u] ? j + ahead : j;
    }
    step(at, ok);
    j += LANES * UNROLL;
  }
}

// Where a search of the sorted entries [lo, end) of an array starts and how
// many entries it has left, one at least: searches in lockstep all read while
// the longest one lasts.  One that has nothing to find (not ok, or an empty
// list) stays on the array's first entry: a list that is empty because no arc
// follows it begins past the last one.
struct Window {
  uint32_t lo, len;
};
MGPM_HD Window search_window(uint32_t lo, uint32_t end, bool ok) {
  if (!ok || end <= lo) return {0u, 1u};
  return {lo, end - lo};
}

}  // namespace mgpm
