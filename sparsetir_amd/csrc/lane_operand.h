// MFMA operands made in registers, and results of eight neighbouring features per lane (gfx950).
#pragma once
#include "common.h"

namespace stir {

typedef uint32_t Words4 __attribute__((ext_vector_type(4)));

// Lane (c, g) of a wavefront holds 8 features from each of 8 rows (k), 16 bytes a row in x[0 .. 7].  Word w of the rows 2 d and
// 2 d + 1 holds the features 2 w and 2 w + 1 of both; one v_perm makes word d of the B operand of either, whose column is c.
// So eight operands, one for each feature of a lane, cost 32 v_perm and no LDS, and a lane ends up with eight neighbouring
// features of a row of the result.  This is the operand of feature 2 w + odd.
template <typename Rows>
__device__ __forceinline__ Words4 operand_of(const Rows& x, int w, int odd) {
  Words4 b;
#pragma unroll
  for (int d = 0; d < 4; ++d)
    b[d] = __builtin_amdgcn_perm(x[2 * d + 1][w], x[2 * d][w], odd ? 0x07060302 : 0x05040100);
  return b;
}

// Eight floats of a lane, dealt out among the four lanes of a quad so that store s (0, 1) of four floats by each lane fills 64
// bytes: floats 16 s + 4 (lane % 4) ... of the quad's 32.  As they are, a store would leave every other 16 bytes to the next
// (condensed product, 169 k rows, 8-row tiles, 128 features, fp32 result 88.7 us, dealt out 68.3).
__device__ __forceinline__ void deal_out(const float (&v)[8], float (&out)[2][4]) {
  const bool second = threadIdx.x & 1;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    // lanes 0, 1 of a quad take from lane 2 s, lanes 2, 3 from lane 2 s + 1
    const int a0 = __builtin_amdgcn_mov_dpp(__float_as_int(v[e]), 0x50, 0xf, 0xf, true);
    const int b0 = __builtin_amdgcn_mov_dpp(__float_as_int(v[4 + e]), 0x50, 0xf, 0xf, true);
    const int a1 = __builtin_amdgcn_mov_dpp(__float_as_int(v[e]), 0xfa, 0xf, 0xf, true);
    const int b1 = __builtin_amdgcn_mov_dpp(__float_as_int(v[4 + e]), 0xfa, 0xf, 0xf, true);
    out[0][e] = __int_as_float(second ? b0 : a0);
    out[1][e] = __int_as_float(second ? b1 : a1);
  }
}

}  // namespace stir
