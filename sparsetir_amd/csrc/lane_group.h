// Feature rows spread over lane groups: what the SpMM kernels share.  A group of G lanes holds a row of
// feat <= 4 * G * REP floats, lane l of it the chunks of four features from 4 * l and 4 * (l + G) on.
#pragma once
#include "common.h"

namespace stir {

// four consecutive floats; a row of B whose width is no multiple of four starts at any float, and a
// 16-byte load only needs its address to be a multiple of four bytes
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ float4 ld4(const float* p) {
  const f32x4u v = *reinterpret_cast<const f32x4u*>(p);
  return make_float4(v[0], v[1], v[2], v[3]);
}

// Feature widths: a lane's chunk number r is the four features from c0 = 4 * (lane in group + r * G)
// on.  In a row whose width is no multiple of four the last chunk would reach into the next row (or
// past the end of B): it is loaded from feat - 4 instead, four features of this row again; a store
// writes the shared ones twice with the same value, an addition moves the ones that are not shared to
// the front first (tail_chunk).
__device__ __forceinline__ int chunk_offset(int c0, int feat) { return min(c0, feat - 4); }

__device__ __forceinline__ float4 tail_chunk(float4 a, int over) {  // over: features of `a` before c0
  if (over & 1) a = make_float4(a.y, a.z, a.w, 0.f);
  if (over & 2) a = make_float4(a.z, a.w, 0.f, 0.f);
  return a;
}

__device__ __forceinline__ void fma4(float4& acc, float a, const float4& x) {
  acc.x = fmaf(a, x.x, acc.x);
  acc.y = fmaf(a, x.y, acc.y);
  acc.z = fmaf(a, x.z, acc.z);
  acc.w = fmaf(a, x.w, acc.w);
}

// 0..5: lane groups of 4, 8, 16, 32, 64 lanes and 64 lanes x 2 float4 cover feat; -1: the kernel of
// one lane per feature (a row narrower than one float4, or wider than two per lane).  Widths that are
// no multiple of 4 take the same kernels (chunk_offset): 169 k nodes, 1.17 M edges with hubs on both
// sides, 47 features: 1750 us with one lane per feature (the chain of the hub row), 52 us with these.
inline int vector_class(int feat) {
  if (feat < 4 || feat > 512) return -1;
  int c = 0;
  while ((16 << c) < feat) ++c;
  return c;
}

// Feature slices: workgroup L of slice_grid(slices, blocks) takes block `block` (which may lie behind the last:
// nothing to do) of slice `slice`.  Workgroups are dispatched round-robin over the 8 XCDs, each with its own L2:
// an XCD works on an eighth of the slices, so it gathers from that much of B.  A slice is dealt out in
// ceil(8 / slices) interleaved pieces, so that an XCD with a part of one has blocks of all its kinds.
constexpr int kXcds = 8;
inline int64_t slice_grid(int slices, int64_t blocks) {
  if (slices == 1) return blocks;
  const int pieces = (kXcds + slices - 1) / slices;
  return kXcds * ceil_div(slices * pieces * ceil_div(blocks, pieces), kXcds);
}
__device__ __forceinline__ void slice_block(int64_t L, int slices, int64_t blocks, int& slice, int64_t& block) {
  const int pieces = (kXcds + slices - 1) / slices;
  const int64_t piece = (blocks + pieces - 1) / pieces, all = slices * pieces * piece;
  const int64_t per = (all + kXcds - 1) / kXcds, t = (L & (kXcds - 1)) * per + L / kXcds;
  if (t >= all || L / kXcds >= per) {
    slice = 0, block = blocks;
    return;
  }
  slice = (int)(t / (pieces * piece));
  const int64_t p = t - slice * (pieces * piece);
  block = p % piece * pieces + p / piece;
}

// csr_balanced.hip: the product of merged rows (see spmm.hip) by workgroups of equal work, added to C, where
// merged_balanced says that this is the better way.
bool merged_balanced(int32_t m, int32_t n, int32_t feat, int64_t slots);
int launch_merged_balanced(int32_t m, int32_t n, int32_t feat, int64_t slots, const float* const* d_vals,
                           const float* d_B, float* d_C, const int32_t* d_slot_ptr, const int32_t* d_cols,
                           hipStream_t st);

}  // namespace stir
