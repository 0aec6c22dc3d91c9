// MFMA operands made in registers (gfx950).
#pragma once
#include "common.h"

namespace stir {

typedef uint32_t Words4 __attribute__((ext_vector_type(4)));
// Eight 16-bit values in a caller's array, which may start at any element of an allocation: loads and stores of 16 bytes take any
// address, but nothing may be made of an alignment that is not there.
typedef uint32_t Halves8 __attribute__((ext_vector_type(4), aligned(2)));

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

}  // namespace stir
