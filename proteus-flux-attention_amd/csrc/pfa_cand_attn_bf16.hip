// The candidate attention kernel (pfa_cand_attn.h) for bf16 inputs.
#include "pfa_cand_attn.h"

namespace pfa {
int cand_attn_launch_bf16(const AttnArgs& a, int out_dtype, int D, hipStream_t s) {
  return cand::launch<PFA_BF16>(a, out_dtype, D, s);
}
}  // namespace pfa
