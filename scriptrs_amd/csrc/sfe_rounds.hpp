// Where the normalisation kernels find their raw log-mel (sfe_kernels.hip), as
// code that the host can run too.
#pragma once

#include "sfe_internal.hpp"

namespace sfe {

// A normalisation workgroup of W waves, lane `lane` of wave w: round j holds
// quad q + 4 W j of the item (q counts from quad q0, a multiple of 4, where the
// workgroup starts) and feature lane % 16 of the slab, at byte off(j) from the
// uniform base (the tile of the item's shared frames where the workgroup
// starts, this slab).  An item's own first quad and last tiles come after its
// shared region (at most kMaxShareFrames frames, then at most 3 tiles for each
// of at most kMaxShareMembers members), so 32-bit byte offsets reach them; an
// item with its own region has all three at out_off.  The region is chosen by
// adding differences under conditions (a choice among several values compiles
// to a table in private memory).
//
// An item that starts SHIFT = gshift % 4 frames into a quad of the shared region
// has its interior quads across two of that region's: frame e of round j is at
// elem_off(j, e).
template <int W>
struct Rounds {
  const char* base;
  uint32_t og, dlo, dhi;
  uint32_t next;  // from the last frame of the shared quad at off(j) to the first of the one after it, less a frame
  int q;          // the lane's quad in round 0
  int qlo, qhi;   // quads [qlo, qhi] are in the shared region
  int left;       // T - 4 q: element e of round j is inside the item where 16 W j + e < left
  static constexpr uint32_t kRound = 4u * kRawTile * W;  // bytes

  __host__ __device__ __forceinline__ Rounds(const float* raw, const Item& it, int slab, int lane, int w, int q0) {
    const int gs = it.gshift / kQuad;
    const int tile0 = (q0 + gs) & ~3;  // quad of the shared region at the base: offsets stay small in any item
    base = reinterpret_cast<const char*>(raw + it.grid_off + raw_quad(tile0) + kRawSlab * slab);
    q = q0 + 4 * w + (lane >> 4);
    og = 4u * (uint32_t)(raw_quad(q + gs - tile0) + 4 * (lane & 15));
    const int64_t own = raw_quad(q) - raw_quad(q + gs) - it.grid_off;
    dlo = 4u * (uint32_t)(it.out_off + own);
    dhi = 4u * (uint32_t)(it.tail_off + own);
    next = 4u * (uint32_t)(raw_quad(q + gs + 1) - raw_quad(q + gs) - kQuad);
    qlo = it.f_lo / kQuad;
    qhi = it.f_hi / kQuad;
    left = it.T - kQuad * q;
  }
  __host__ __device__ __forceinline__ uint32_t off(int j) const {
    uint32_t o = og + kRound * (uint32_t)j + (q + 4 * W * j > qhi ? dhi : 0u);
    if (j == 0) o += q < qlo ? dlo : 0u;  // (the own first quad is quad 0)
    return o;
  }
  // Past the item: an offset past the buffer's range, for which the hardware
  // returns zeros without a memory access.
  __host__ __device__ __forceinline__ int buf_off(int j) const { return 16 * W * j < left ? (int)off(j) : kNormBufRange; }
  // Offset of frame e of round j of an item with gshift % kQuad == SHIFT (past
  // the item, its top bit is set: past the buffer's range too).
  template <int SHIFT>
  __host__ __device__ __forceinline__ int elem_off(int j, int e) const {
    const uint32_t shared = 4u * (SHIFT + e) + (SHIFT + e >= kQuad ? next : 0u);
    const bool own = (q + 4 * W * j > qhi) | (j == 0 && q < qlo);
    return (int)((off(j) + (own ? 4u * e : shared)) | (16 * W * j < left ? 0u : 0x80000000u));
  }
  // Whether every lane of the workgroup holds 4 frames of the item in round j,
  // T frames counted from the workgroup's first.
  static __host__ __device__ __forceinline__ bool full(int j, int T) { return 16 * W * (j + 1) <= T; }
};

}  // namespace sfe
