// Sixteen bytes through to the memory that all XCDs see, and from there: what workgroups of one launch leave for
// each other.  As four-byte atomics a partial tile took four masked writes per 16 bytes; a release or acquire at
// device scope would write back or invalidate a whole L2.
#pragma once
#include "common.h"

namespace stir {

typedef float f32x4c __attribute__((ext_vector_type(4)));

// Has arrived when the wavefront's vmcnt is zero.
__device__ __forceinline__ void coherent_store(float* p, const f32x4c& v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1" : : "v"(p), "v"(v) : "memory");
}

// v[u] = the four floats at p[u], all eight in flight together.  One statement, the wait included: to the compiler
// the result of a load it does not know of is there at once, and it may move it before a wait that stands apart.
__device__ __forceinline__ void coherent_load(f32x4c (&v)[8], const float* const (&p)[8]) {
  asm volatile(
      "global_load_dwordx4 %0, %8, off sc1\n\t"
      "global_load_dwordx4 %1, %9, off sc1\n\t"
      "global_load_dwordx4 %2, %10, off sc1\n\t"
      "global_load_dwordx4 %3, %11, off sc1\n\t"
      "global_load_dwordx4 %4, %12, off sc1\n\t"
      "global_load_dwordx4 %5, %13, off sc1\n\t"
      "global_load_dwordx4 %6, %14, off sc1\n\t"
      "global_load_dwordx4 %7, %15, off sc1\n\t"
      "s_waitcnt vmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
      : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[6]), "v"(p[7])
      : "memory");
}

}  // namespace stir
