// One-pass cross-entropy (cross_entropy.hpp) over bf16 logits.
#include "cross_entropy.hpp"

namespace ts_ce {

bool fused_bf16(const FusedArgs& a, bool wide, ts_status* status) {
  return wide ? launch_fused<__bf16, float>(a, status) : launch_fused<__bf16, __bf16>(a, status);
}

}  // namespace ts_ce
