// row_starts.hpp — which sub-tiles start within a row: shared by the passes
// that note every sub-tile's first row (transpose.hip, spmv_scatter.hip) and the
// host test.
#pragma once

#include <cstdint>

namespace fs {

// The first of n_sub sub-tiles (`items` entries each) that starts at entry e or
// later, n_sub if none does; a row over [a, b) holds the starts of sub-tiles
// [row_sub_tile(a), row_sub_tile(b)).  In [0, n_sub] for any e: a row pointer is
// unchecked here, and e + items - 1 wraps for 64-bit values near the largest
// (the sub-tile came out negative, and its row was written there).
constexpr int64_t row_sub_tile(int64_t e, int64_t items, int64_t n_sub) {
  if (e <= 0) return 0;
  const int64_t q = (e - 1) / items + 1;
  return q < n_sub ? q : n_sub;
}

}  // namespace fs
