// The candidate attention kernel (pfa_cand_attn.h) for f16 inputs.
#include "pfa_cand_attn.h"

namespace pfa {
int cand_attn_launch_f16(const AttnArgs& a, int out_dtype, int D, hipStream_t s) {
  return cand::launch<PFA_F16>(a, out_dtype, D, s);
}
}  // namespace pfa
