// The general attention kernel at D = 128.
#include "attn_fwd.h"

namespace kfmi {

hipError_t launch_fwd128(const AttnParams &p, bool causal, int pro, int st, int blocks, hipStream_t s) {
  return causal ? launch_fwd_c<128, true>(p, pro, st, blocks, s) : launch_fwd_c<128, false>(p, pro, st, blocks, s);
}

}  // namespace kfmi
