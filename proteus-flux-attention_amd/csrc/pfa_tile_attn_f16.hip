// The tile attention kernel (pfa_tile_attn.h) for f16 inputs.
#include "pfa_tile_attn.h"

namespace pfa {
int tile_attn_launch_f16(const AttnArgs& a, int out_dtype, int D, hipStream_t s) {
  return tile::launch<PFA_F16>(a, out_dtype, D, s);
}
}  // namespace pfa
