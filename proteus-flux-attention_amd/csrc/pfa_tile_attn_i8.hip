// The tile attention kernel (pfa_tile_attn.h) for i8 inputs.
#include "pfa_tile_attn.h"

namespace pfa {
int tile_attn_launch_i8(const AttnArgs& a, int out_dtype, int D, hipStream_t s) {
  return tile::launch<PFA_I8>(a, out_dtype, D, s);
}
}  // namespace pfa
