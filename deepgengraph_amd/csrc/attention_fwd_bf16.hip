// The 16-bit attention forward (attention_fwd.h) for bf16 inputs.
#include "attention_fwd.h"

namespace dgg_attn {

void launch_attn_fwd_bf16(const AttnParams& p, int D, bool ref, hipStream_t st) {
  if (D == 64) pick_fwd<BF16, 64>(p, ref, st);
  else if (D == 128) pick_fwd<BF16, 128>(p, ref, st);
  else pick_fwd<BF16, 256>(p, ref, st);
}

}  // namespace dgg_attn
