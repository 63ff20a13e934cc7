// Workgroups of the Krylov sweeps that leave partial sums in a workspace's
// buffer (dots, norms): the buffer's size and how many workgroups a sweep takes.
#pragma once

#include <algorithm>
#include <cstdint>

namespace pgs {

constexpr int kPartBlocks = 1024;  // most workgroups of such a sweep: four per CU

// The buffer holds part_rows(kdim) values per column for each of part_blocks(n)
// workgroups, one per 256 rows or more.
inline int64_t part_blocks(int64_t n) {
  const int64_t rows_per_blk = std::max<int64_t>(256, (n + kPartBlocks - 1) / kPartBlocks);
  return std::max<int64_t>(1, (n + rows_per_blk - 1) / rows_per_blk);
}

// kdim + 1 dots, or the 2 p + 2 of a delayed-CGS2 step (66: the norms of an
// update by up to 4096 workgroups)
inline int64_t part_rows(int64_t kdim) { return std::max<int64_t>(2 * kdim + 2, 66); }

// Workgroups for `want` workgroup-sized pieces of a vector block: part_blocks, or
// more where that leaves over `most` pieces to each, as it does for wide batches
// of few rows; at most `fit`, what the buffer holds, and kPartBlocks.
inline int64_t sweep_blocks(int64_t blocks, int64_t want, int64_t fit, int64_t most) {
  const int64_t more = std::min<int64_t>({kPartBlocks, fit, (want + most - 1) / most});
  return std::max<int64_t>({1, std::min(blocks, want), more});
}

}  // namespace pgs
