// Sixteen bytes through to the memory that all XCDs see, and from there: what workgroups of one launch leave for
// each other.  As four-byte atomics a partial tile took four masked writes per 16 bytes; a release or acquire at
// device scope would write back or invalidate a whole L2.
#pragma once
#include "common.h"

namespace stir {

// Buffer instructions with the bit that a device-wide atomic load or store sets (sc1), rather than inline assembly:
// the compiler knows when the result of a load is there and which registers a store still reads.
class CoherentPiece {
 public:
  typedef uint32_t Four __attribute__((ext_vector_type(4)));
  // `bytes` (below 2^32) from a 16-byte aligned address that is the same for all lanes
  __device__ __forceinline__ CoherentPiece(float* base, uint32_t bytes)
      : r_(__builtin_amdgcn_make_buffer_rsrc(base, 0, bytes, 0x00027000)) {}
  // offsets in floats, a multiple of four
  __device__ __forceinline__ float4 load(uint32_t at) const {
    return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r_, 4 * at, 0, kSc1));
  }
  // has arrived when the wavefront's vmcnt is zero
  __device__ __forceinline__ void store(uint32_t at, const float4& v) const {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(Four, v), r_, 4 * at, 0, kSc1);
  }

 private:
  static constexpr int kSc1 = 16;
  __amdgpu_buffer_rsrc_t r_;
};

}  // namespace stir
