// Index arithmetic of kernels whose 32-bit indices reach up to 2^31 - 1, free
// of HIP so that the host can test it there.
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define CBX_HD __host__ __device__ __forceinline__
#else
#define CBX_HD inline
#endif

namespace cbx {

// The first index in [lo, end) with row(index) >= key, end if there is none;
// the rows ascend.  Searched for from lo with a step that doubles: one or two
// probes where it is near, a logarithm where not.
template <class Row>
CBX_HD int32_t first_from(Row&& row, int32_t lo, int32_t end, int64_t key) {
  int32_t step = 1, hi = lo;  // rows before lo are below key
  while (hi < end && row(hi) < key) {
    lo = hi + 1;
    hi = end - lo < step ? end : lo + step;  // (lo + step may pass 2^31)
    step = step < 1 << 29 ? step * 2 : step;
  }
  while (lo < hi) {  // in [lo, hi]
    const int32_t mid = lo + (hi - lo) / 2;
    if (row(mid) < key) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// Entry `off` of those from `first` (below end) on, and whether there is one
// (ok): past the end the last entry's index.
CBX_HD int32_t entry_from(int32_t first, int32_t end, int32_t off, bool& ok) {
  const int32_t left = end - first;
  ok = off < left;
  return first + (ok ? off : left - 1);
}

}  // namespace cbx
