// scatter_segments.hpp — how the scattered-product SpMV (spmv_scatter.hip)
// cuts its buckets into segments.  Plain arithmetic: the device plan, the host
// layout and the host test share it.
#pragma once

#include <algorithm>
#include <cstdint>

namespace fs {

// Entries per segment, for nnz entries over `used` buckets: enough segments to
// fill the chip, but a bucket of ordinary size whole.
constexpr uint32_t scatter_segment_items(int64_t nnz, int64_t used) {
  const int64_t fill = std::max<int64_t>(2048, nnz / 1024);
  const int64_t typical = nnz / used + nnz / used / 2;
  return (uint32_t)(typical <= 4 * fill ? std::max(fill, typical) : fill);
}

// Segments of a bucket of c entries, at least one (which writes the zeros of an
// empty bucket).  No c + seg_items: near 2^32 entries in one bucket it wraps.
constexpr uint32_t scatter_bucket_segments(uint32_t c, uint32_t seg_items) {
  return c == 0 ? 1u : c / seg_items + (c % seg_items != 0 ? 1u : 0u);
}

}  // namespace fs
