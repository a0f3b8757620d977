// Host run of sfe::for_launches (scriptrs_amd/csrc/sfe_internal.hpp): for
// workgroup sizes and counts around the most that a launch holds, every
// workgroup is in exactly one launch, in order, no launch holds 2^32 threads or
// more, and all but the last start at a multiple of 8.  And the rule that picks
// the workgroup form of the normalisation, sfe::norm_wide.  Prints "bad N".
#include <stdio.h>

#include "sfe_internal.hpp"

int main() {
  long bad = 0;
  for (int threads : {64, 256, 512, 576, 1024}) {
    const int64_t most = (((int64_t)1 << 32) - 1) / threads;
    for (int64_t blocks : {(int64_t)0, (int64_t)1, (int64_t)7, (int64_t)8, most - 9, most - 8, most - 1, most, most + 1,
                           2 * most, 5 * most + 3}) {
      int64_t at = 0;
      int launches = 0;
      const hipError_t e = sfe::for_launches(blocks, threads, [&](int64_t first, unsigned n) {
        bad += first != at || first % 8 != 0 || n == 0 || (int64_t)n * threads >= (int64_t)1 << 32;
        at = first + n;
        ++launches;
        return hipSuccess;
      });
      bad += e != hipSuccess || at != blocks || launches > blocks / (most - 8) + 1;
      if (blocks > most)  // a failed launch ends it
        bad += sfe::for_launches(blocks, threads, [&](int64_t, unsigned) { return hipErrorUnknown; }) != hipErrorUnknown;
    }
  }
  // the workgroup form of the normalisation (sfe::norm_wide), 256 CUs: clips of
  // one length, then ragged ones
  struct { int n, T, wide; } forms[] = {{1, 10, 0}, {1, 256, 0}, {1, 257, 1}, {1, 2000, 1}, {32, 201, 0}, {32, 401, 1},
                                        {33, 401, 0}, {96, 501, 0}, {128, 501, 0}, {129, 501, 1}, {300, 51, 0},
                                        {300, 201, 0}, {2400, 201, 0}, {300, 401, 0}, {300, 448, 0}, {300, 449, 1},
                                        {40, 513, 1}, {96, 1501, 1}, {300, 1501, 1}, {300, 2048, 1}};
  for (auto& f : forms) bad += sfe::norm_wide(f.n, f.T, (int64_t)f.n * f.T, 256) != (f.wide != 0);
  for (auto& f : forms) bad += sfe::norm_wide(f.n, f.T, (int64_t)f.n * f.T / 2, 256) != (f.wide && 8 * f.n <= 768);
  printf("bad %ld\n", bad);
  return bad != 0;
}
