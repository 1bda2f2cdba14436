// One-pass cross-entropy (cross_entropy.hpp) over fp32 logits.
#include "cross_entropy.hpp"

namespace ts_ce {

bool fused_f32(const FusedArgs& a, ts_status* status) {
  return launch_fused<float, float>(a, status);
}

}  // namespace ts_ce
