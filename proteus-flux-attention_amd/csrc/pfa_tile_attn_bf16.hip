// The tile attention kernel (pfa_tile_attn.h) for bf16 inputs.
#include "pfa_tile_attn.h"

namespace pfa {
int tile_attn_launch_bf16(const AttnArgs& a, int out_dtype, int D, hipStream_t s) {
  return tile::launch<PFA_BF16>(a, out_dtype, D, s);
}
}  // namespace pfa
