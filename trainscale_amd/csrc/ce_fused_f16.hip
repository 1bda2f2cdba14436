// One-pass cross-entropy (cross_entropy.hpp) over fp16 logits.
#include "cross_entropy.hpp"

namespace ts_ce {

bool fused_f16(const FusedArgs& a, bool wide, ts_status* status) {
  return wide ? launch_fused<_Float16, float>(a, status) : launch_fused<_Float16, _Float16>(a, status);
}

}  // namespace ts_ce
