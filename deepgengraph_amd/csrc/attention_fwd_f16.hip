// The 16-bit attention forward (attention_fwd.h) for f16 inputs.
#include "attention_fwd.h"

namespace dgg_attn {

void launch_attn_fwd_f16(const AttnParams& p, int D, bool ref, hipStream_t st) {
  if (D == 64) pick_fwd<F16, 64>(p, ref, st);
  else if (D == 128) pick_fwd<F16, 128>(p, ref, st);
  else pick_fwd<F16, 256>(p, ref, st);
}

}  // namespace dgg_attn
