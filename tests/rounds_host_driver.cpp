// Host run of the normalisation kernels' addressing (scriptrs_amd/csrc/
// sfe_rounds.hpp) over planned tables: for every item, both workgroup forms,
// every lane and round, the loads of a quad's 4 frames must be the raw slots
// that the table's rule names (sfe_internal.hpp Item), at offsets inside the
// buffer, and past the item outside it.
//
// stdin: cases, each "n" then n lines "start len".  Prints "case <k> quads
// <with> <own> shifted <items>" and at the end "bad <count>".
#include <stdio.h>

#include <vector>

#include "sfe_internal.hpp"
#include "sfe_rounds.hpp"

using sfe::Item;

static long bad = 0;

// One workgroup at quad q0 of item it, rounds [0, rounds).
template <int W>
static void check(int k, int i, const Item& it, int q0, int rounds) {
  const float* raw = reinterpret_cast<const float*>((uintptr_t)1 << 40);
  for (int slab = 0; slab < 8; slab += 7)
    for (int w = 0; w < W; ++w)
      for (int lane = 0; lane < 64; lane += 5) {
        const sfe::Rounds<W> rd(raw, it, slab, lane, w, q0);
        for (int j = 0; j < rounds; ++j) {
          const int64_t q = q0 + 4 * (W * j + w) + lane / 16;
          for (int e = 0; e < 4; ++e) {
            const int shift = it.gshift % sfe::kQuad;
            const uint32_t off = (uint32_t)(shift == 0   ? rd.template elem_off<0>(j, e)
                                            : shift == 1 ? rd.template elem_off<1>(j, e)
                                            : shift == 2 ? rd.template elem_off<2>(j, e)
                                                         : rd.template elem_off<3>(j, e));
            const uint32_t whole = (uint32_t)rd.buf_off(j);
            bool ok;
            if (4 * q >= it.T) {
              ok = off >= (uint32_t)sfe::kNormBufRange && whole >= (uint32_t)sfe::kNormBufRange;
            } else {
              const int64_t f = 4 * q + e;  // in the item's quads, or its last tile's padding
              const bool g = f >= it.f_lo && f <= it.f_hi;
              const int64_t a = (g ? it.grid_off : (f < it.f_lo ? it.out_off : it.tail_off)) +
                                sfe::raw_frame(g ? f + it.gshift : f) + sfe::kRawSlab * slab + 4 * (lane % 16);
              const char* want = reinterpret_cast<const char*>(raw + a);
              ok = off < (uint32_t)sfe::kNormBufRange - 16 && rd.base + off == want;
              if (shift == 0) ok = ok && rd.base + whole + 4 * e == want;
              ok = ok && (16 * W * j + e < rd.left) == (f < it.T);
            }
            if (!ok && bad++ < 20)
              printf("case %d item %d W %d q0 %d slab %d wave %d lane %d round %d frame %d\n", k, i, W, q0, slab, w,
                     lane, j, e);
          }
        }
      }
}

int main() {
  int n, k = 0;
  while (scanf("%d", &n) == 1) {
    std::vector<Item> items(n);
    int64_t fo = 0;
    for (int i = 0; i < n; ++i) {
      long long s, l;
      if (scanf("%lld %lld", &s, &l) != 2) return 2;
      items[i] = sfe::own_item(s, l, 0, sfe::kMel * fo, 0);
      fo += items[i].T;
    }
    sfe::PlanWorkspace ws;
    ws.reserve((size_t)n);
    std::vector<Item> table((size_t)(sfe::kPlanEntriesPerItem + 1) * n);
    size_t n_lm = 0;
    sfe::plan_table(items.data(), n, true, &ws, table.data(), &n_lm);
    int64_t quads = 0, own = 0;
    int shifted = 0;
    for (size_t e = 0; e < n_lm; ++e) quads += table[e].n_units;
    for (int i = 0; i < n; ++i) {
      const Item& it = table[n_lm + i];
      own += (it.T + 3) / 4;
      shifted += it.gshift % sfe::kQuad != 0;
      if (it.T <= sfe::kNormRegFrames) {
        check<4>(k, i, it, 0, sfe::kNormRegFrames / 64);
        check<8>(k, i, it, 0, sfe::kNormRegFrames / 128);
      } else {
        for (int t = 0; t < it.T; t += sfe::kSegFrames) check<4>(k, i, it, t / sfe::kQuad, sfe::kSegFrames / 64);
      }
    }
    printf("case %d quads %lld %lld shifted %d\n", k++, (long long)quads, (long long)own, shifted);
  }
  printf("bad %ld\n", bad);
  return 0;
}
