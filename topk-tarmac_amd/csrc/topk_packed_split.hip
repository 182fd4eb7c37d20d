// Packed top-k (k <= 8) for fp32 d = 32 and 64 on split-bf16 scores; a
// translation unit of its own so the build compiles it beside the others.
#include "topk_packed.hpp"

namespace tarmac {

hipError_t run_topk_packed_split_wide(const TopkArgs& a) {
  return a.d == 32 ? launch_packed<float, 32, true>(a) : launch_packed<float, 64, true>(a);
}

}  // namespace tarmac
