// Sizes of the blocks that the caching allocator asks the driver for, free of
// HIP so that the host can test them.
#pragma once

#include <cstddef>

namespace cbx {

// The size of a new block for `bytes`: rounded up to an eighth of its leading
// power of two, so that products whose sizes differ by a few percent (the
// column phases of an MCL expansion) find each other's blocks, but by less than
// kBlockStep, so that the largest products keep the card's memory (unbounded,
// ir and val of R-MAT s20 took 16 GB more than their 156).  Twelve MCL
// expansions of new matrices of 480 to 535 K columns (blocks of 20 to 30 GB):
// 82 to 92 ms each with this bound and without one; with 256 MB two of them took
// 0.4 and 1.6 s to give blocks back, with 16 MB one 3 s.
constexpr size_t kBlockStep = (size_t)1 << 30;
inline size_t block_bytes(size_t bytes) {
  size_t step = 256;
  while (step < kBlockStep && step * 16 <= bytes) step *= 2;
  return (bytes + step - 1) / step * step;
}

}  // namespace cbx
