// Workgroups of the sweeps that leave partial sums (sweep_blocks), over rows,
// columns and Krylov dimensions: their partials fit the buffer, none of them is
// idle, and no wide batch of few rows is left to a handful of them.
//
// usage: sweep_check   (exit 0 when all hold)
#include <cstdint>
#include <cstdio>

#include "../../pargemslr_amd/csrc/host/sweep_blocks.hpp"

using namespace pgs;

int main() {
  int64_t bad = 0, checked = 0;
  for (int64_t n : {1, 2, 63, 255, 256, 257, 1000, 1001, 4096, 13824, 32768, 110592, 262143, 262145, 2097152})
    for (int64_t nrhs = 1; nrhs <= 64; nrhs *= 2)
      for (int64_t kdim : {1, 10, 50, 127})
        for (int64_t lanes : {64, 128, 256, 512})      // values a workgroup takes at a time
          for (int64_t rows : {(int64_t)2, kdim + 1, 2 * kdim + 2})
            for (int64_t most : {8, 32}) {
              const int64_t want = (n * nrhs + lanes - 1) / lanes;
              const int64_t fit = part_blocks(n) * part_rows(kdim) / rows;
              const int64_t b = sweep_blocks(part_blocks(n), want, fit, most);
              ++checked;
              const bool walks = b * most < want && b < fit && b < kPartBlocks;
              if (b < 1 || b > want || b > fit || b > kPartBlocks || walks) {
                if (++bad < 10)
                  std::printf("n %ld, %ld columns, kdim %ld, %ld rows: %ld workgroups for %ld pieces\n", (long)n,
                              (long)nrhs, (long)kdim, (long)rows, (long)b, (long)want);
              }
            }
  std::printf("%ld sweeps, %ld bad\n", (long)checked, (long)bad);
  return bad ? 1 : 0;
}
