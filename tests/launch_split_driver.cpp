// Host run of sfe::for_launches (scriptrs_amd/csrc/sfe_internal.hpp): for
// workgroup sizes and counts around the most that a launch holds, every
// workgroup is in exactly one launch, in order, no launch holds 2^32 threads or
// more, and all but the last start at a multiple of 8.  Prints "bad N".
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
  printf("bad %ld\n", bad);
  return bad != 0;
}
