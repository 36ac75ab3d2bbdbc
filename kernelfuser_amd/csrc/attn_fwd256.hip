// The general attention kernel at D = 256.
#include "attn_fwd.h"

namespace kfmi {

hipError_t launch_fwd256(const AttnParams &p, bool causal, int pro, int st, int blocks, hipStream_t s) {
  return causal ? launch_fwd_c<256, true>(p, pro, st, blocks, s) : launch_fwd_c<256, false>(p, pro, st, blocks, s);
}

}  // namespace kfmi
