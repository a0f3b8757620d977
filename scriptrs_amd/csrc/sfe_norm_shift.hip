// The normalisation of calls with items that start inside a quad of their shared
// region (gshift % kQuad != 0), in a code object of its own (sfe_norm.hpp).
#include "sfe_norm.hpp"

namespace sfe {

hipError_t launch_norm_shifted(const float* raw, const Item* items, int n_items, int max_T, int64_t sum_T, int cus,
                               int pad_to, void* out, bool out_bf16, int n_segs, const int32_t* seg_item, void* parts,
                               hipStream_t stream) {
  return launch_norm_form<true>(raw, items, n_items, max_T, sum_T, cus, pad_to, out, out_bf16, n_segs, seg_item, parts,
                                stream);
}

}  // namespace sfe
