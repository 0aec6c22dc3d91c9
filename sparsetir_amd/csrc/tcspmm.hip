// SpMM on the gfx950 matrix cores over the condensed format of ConDense: the rows of the
// sparse matrix are cut into tiles of t rows (t = 8, 16 -- the two sizes the reference's
// examples/spmm/bench_tc_spmm.py:584-585,670 condenses with -- or 32); inside a tile the distinct
// columns are gathered g = 16 at a time into dense t x 16 blocks A[jo] (zero where the row has no
// entry):
//   C[io*t + ii, f] = sum over groups jo of tile io, ji < 16:  A[jo, ii, ji] * B[indices[jo, ji], f]
// fp16 inputs, fp32 accumulation, fp16 or fp32 output.
//
// With a plan (stir_tc_plan: the long tiles listed once, longest first, in pieces) a product is one launch of
// tcspmm_units_kernel, or of tcspmm_direct_kernel above 64 features (tc_form).  Bound by the gather of rows of B where there
// are tiles enough, else by the chain id -> row of B -> product of the longest unit.  Before, the tiles of up to 16 steps went as below and the pieces of the others in a
// second launch, a workgroup of 16 wavefronts each.  Tiles of 16 rows, power-law rows of up to 500 to 17.5 k nonzeros,
// uniform columns, us: 25.9 k rows, 626 k nonzeros, 32 features 22.4 -> 10.8; 167 k, 3.8 M, 32: 83 -> 66; 24 k, 244 k,
// 64: 22.2 -> 10.8; 200 k, 4 M, 64: 101 -> 90; 33 k, 648 k, 224: 61 -> 48; 169 k, 1.17 M, 128: 62.1 -> 62.7 over the
// same arrays again and again, 70.3 -> 63.4 where other arrays are used in between (skewed columns 47 -> 49).
//
// Without a plan: a workgroup of four wavefronts owns (row tile, 128 features), a wavefront t rows x 32 features.
// A step covers two groups (32 gathered rows of B): A[jo] is already in MFMA A-operand order (a lane's 8 k values
// are contiguous), the 32 gathered rows of B go through LDS, interleaved into (k, k+1) pairs on the way,
// double-buffered, with the next step's gathers in flight during the multiply.  Tiles of 32 rows multiply with
// two v_mfma_f32_32x32x16_f16 per step (one per group); tiles of 16 rows with v_mfma_f32_16x16x32_f16, whose k
// extent of 32 is the step's two groups, once per 16 features; tiles of 8 rows are the upper half of a 16-row
// operand whose other rows are zero.
//
// A row tile that touches thousands of distinct columns (a hub row of a power-law graph) would be
// one long serial chain in one workgroup.  With fp32 output such tiles are cut into up to kSplit
// units of at least kUnitSteps steps that add their results with atomics; a first launch clears the rows
// of those tiles.  With fp16 output partial sums would be rounded once per unit; there, tiles of
// more than kLongSteps steps are left to a second launch (tcspmm_long_kernel) whose workgroups
// have 16 wavefronts that split the steps of the tile among them and add their fp32 partial sums
// through LDS before the one write of the tile.
#include <algorithm>
#include <vector>

#include "coherent.h"
#include "common.h"
#include "lane_operand.h"
#include "../../include/sparsetir_amd.h"

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

typedef float f32x4 __attribute__((ext_vector_type(4)));
using stir::Halves8;
// as stored at any element of C
typedef float Float4 __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kTileF = 128;
constexpr int kGroup = 16;  // g
constexpr int kUnitSteps = 16;  // steps (of two groups) per unit of a long tile
constexpr int kSplit = 16;      // most units per tile (second grid dimension of the split launch)
constexpr int kLongSteps = 16;  // fp16 output: tiles with more steps go to the second launch
constexpr int kLongScan = 8;    // ... each workgroup of which looks at this many row tiles
constexpr int kLongNT = 2;      // ... whose workgroups own 32 * kLongNT features and have 32 / kLongNT * 4 wavefronts

__device__ __forceinline__ int tile_steps(const int32_t* __restrict__ indptr, int64_t io) {
  const int64_t rows_total = (int64_t)(indptr[io + 1] - indptr[io]) * kGroup;
  return (int)((rows_total + 31) / 32);
}

// ---- what differs between the row-tile sizes: the accumulators of a wavefront for (T rows) x
// (32 features), the A operand of a step, and the multiply of a step out of the staged rows of B.
// WIDE = 32-row tiles on the 32x32x16 instruction; otherwise 16-row operands on 16x16x32.
template <bool WIDE>
struct TcAcc;
template <>
struct TcAcc<true> {
  static constexpr int kRegs = 16;
  f32x16 r;
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int v = 0; v < 16; ++v) r[v] = 0.f;
  }
  __device__ __forceinline__ float get(int v) const { return r[v]; }
  // register v of lane l is this row / feature of the wavefront's tile
  static __device__ __forceinline__ int row(int v, int l) { return (v & 3) + 4 * (l >> 5) + 8 * (v >> 2); }
  static __device__ __forceinline__ int col(int v, int l) { return l & 31; }
};
template <>
struct TcAcc<false> {
  static constexpr int kRegs = 8;  // two 16x16 tiles side by side
  f32x4 r[2];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int v = 0; v < 8; ++v) r[v >> 2][v & 3] = 0.f;
  }
  __device__ __forceinline__ float get(int v) const { return r[v >> 2][v & 3]; }
  static __device__ __forceinline__ int row(int v, int l) { return 4 * (l >> 4) + (v & 3); }
  static __device__ __forceinline__ int col(int v, int l) { return 16 * (v >> 2) + (l & 15); }
};

// A[jo] and A[jo + 1] as the A operand(s) of a step (zero past the tile's last group).
// T = 32: lane (n = l % 32, h = l / 32) holds A[jo + d][n][8h .. 8h+7] in a[d].
// T <= 16: lane (i = l % 16, q = l / 16) holds k = 8q .. 8q+7 of the step's 32, i.e.
// A[jo + q/2][i][8(q%2) ..], in a[0]; rows i >= T of the operand are zero.
template <int T>
__device__ __forceinline__ void tc_load_a(u32x4 (&a)[2], const uint16_t* __restrict__ A, int64_t jo, int64_t g_end,
                                          int lane) {
  a[0] = a[1] = u32x4{0, 0, 0, 0};
  if constexpr (T == 32) {
    const int n = lane & 31, h = lane >> 5;
    a[0] = *reinterpret_cast<const Halves8*>(A + (jo * 32 + n) * kGroup + 8 * h);
    if (jo + 1 < g_end) a[1] = *reinterpret_cast<const Halves8*>(A + ((jo + 1) * 32 + n) * kGroup + 8 * h);
  } else {
    const int i = lane & 15, q = lane >> 4;
    const int64_t grp = jo + (q >> 1);
    if (i < T && grp < g_end) a[0] = *reinterpret_cast<const Halves8*>(A + (grp * T + i) * kGroup + 8 * (q & 1));
  }
}

// Where 16-byte-aligned feature offset `col` of k pair `kp` lives inside its staged row of STRIDE
// words (a power of two).  The 16-row multiply reads rows 4q .. 4q+3 for q = l / 16 at 16
// consecutive features: rotating a row by 16 (kp / 4) words puts the four q on different banks.
template <int T, int STRIDE>
__device__ __forceinline__ int tc_stage_col(int kp, int col) {
  if constexpr (T == 32) return col;
  else return (col + 16 * (kp >> 2)) & (STRIDE - 1);
}

// acc += A-operand(s) x the 32 staged rows of B, features col0 .. col0+31 of the staged rows
// xs[16 k pairs][STRIDE]
template <int T, int STRIDE>
__device__ __forceinline__ void tc_multiply(TcAcc<T == 32>& acc, const u32x4 (&a)[2], const uint32_t* xs, int col0,
                                            int lane) {
  if constexpr (T == 32) {
    const int n = lane & 31, h = lane >> 5;
    u32x4 b0, b1;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      b0[d] = xs[(4 * h + d) * STRIDE + col0 + n];      // rows 8h .. 8h+7 of the first group
      b1[d] = xs[(8 + 4 * h + d) * STRIDE + col0 + n];  // rows 8h .. 8h+7 of the second group
    }
    acc.r = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a[0]), __builtin_bit_cast(f16x8, b0),
                                                  acc.r, 0, 0, 0);
    acc.r = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a[1]), __builtin_bit_cast(f16x8, b1),
                                                  acc.r, 0, 0, 0);
  } else {
    const int n = lane & 15, q = lane >> 4;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const int c = tc_stage_col<T, STRIDE>(4 * q, col0 + 16 * nt) + n;
      u32x4 b;
#pragma unroll
      for (int d = 0; d < 4; ++d) b[d] = xs[(4 * q + d) * STRIDE + c];  // rows 8q .. 8q+7 of the step
      acc.r[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[0]),
                                                        __builtin_bit_cast(f16x8, b), acc.r[nt], 0, 0, 0);
    }
  }
}

// Clears the fp32 rows of the tiles that the split launch accumulates into.  grid (mb * f_tiles)
__global__ __launch_bounds__(256) void tcspmm_clear_long_kernel(int tile, int feat, int64_t mb, int f_tiles,
                                                                float* __restrict__ C,
                                                                const int32_t* __restrict__ indptr) {
  const int f_tile = (int)(blockIdx.x % f_tiles);
  const int64_t io = blockIdx.x / f_tiles;
  if (io >= mb || tile_steps(indptr, io) <= kUnitSteps) return;
  const int f0 = f_tile * kTileF;
  for (int e = threadIdx.x; e < tile * kTileF; e += 256) {
    const int row = e / kTileF, f = f0 + e % kTileF;
    if (f < feat) C[(io * tile + row) * feat + f] = 0.f;
  }
}

// OUT: 0 = fp16 output, 1 = fp32 output.  SPLIT: grid is (mb * f_tiles, kSplit); the units of a
// long tile take equal shares of its steps and add with atomics, unit 0 of a short tile stores.
template <int T, int OUT, bool SPLIT>
__global__ __launch_bounds__(256) void tcspmm_kernel(int feat, int64_t mb, int f_tiles,
                                                     const uint16_t* __restrict__ A,
                                                     const uint16_t* __restrict__ B, void* __restrict__ C,
                                                     const int32_t* __restrict__ indptr,
                                                     const int32_t* __restrict__ indices) {
  __shared__ __attribute__((aligned(16))) uint32_t xs[2][16 * kTileF];  // [buffer][k pair][feature]
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int f_tile = (int)(blockIdx.x % f_tiles);
  const int64_t io = blockIdx.x / f_tiles;
  if (io >= mb) return;
  const int f0 = f_tile * kTileF;
  const int kp = tid >> 4, fc = tid & 15;  // staging role: k pair, 8-feature chunk
  const bool stage_live = f0 + fc * 8 < feat;
  const int stage_at = kp * kTileF + tc_stage_col<T, kTileF>(kp, fc * 8);

  TcAcc<T == 32> acc;
  acc.clear();

  const int64_t g_begin = indptr[io], g_end = indptr[io + 1];
  const int64_t rows_total = (g_end - g_begin) * kGroup;  // gathered rows of B for this tile
  const int steps = (int)((rows_total + 31) / 32);
  const int32_t* rowlist = indices + g_begin * kGroup;
  if constexpr (OUT == 0) {
    if (steps > kLongSteps) return;  // left to the launch for long tiles; uniform over the workgroup
  }
  int it_begin = 0, it_end = steps;
  bool add = false;
  if constexpr (SPLIT) {
    const int u = blockIdx.y;
    if (steps > kUnitSteps) {
      add = true;
      const int len = max(kUnitSteps, (steps + kSplit - 1) / kSplit);  // even shares beyond kSplit units
      it_begin = u * len;
      it_end = min(steps, it_begin + len);
      if (it_begin >= it_end) return;  // uniform over the workgroup
    } else if (u > 0) {
      return;
    }
  }

  // The row ids of a step are requested one step before its rows of B, so that a step costs one
  // memory round trip, not two in a row.
  int row_a = 0, row_b = 0;
  auto fetch_ids = [&](int it) {
    const int64_t k = (int64_t)it * 32 + 2 * kp;
    row_a = row_b = 0;
    if (k < rows_total) row_a = rowlist[k], row_b = rowlist[k + 1];  // the same group: both exist
  };
  u32x4 r0, r1, a_next[2];
  auto fetch = [&](int it) {
    tc_load_a<T>(a_next, A, g_begin + 2 * it, g_end, lane);
    r0 = r1 = u32x4{0, 0, 0, 0};
    const int64_t k = (int64_t)it * 32 + 2 * kp;
    if (stage_live && k < rows_total) {
      r0 = *reinterpret_cast<const Halves8*>(B + (int64_t)row_a * feat + f0 + fc * 8);
      r1 = *reinterpret_cast<const Halves8*>(B + (int64_t)row_b * feat + f0 + fc * 8);
    }
    if (it + 1 < it_end) fetch_ids(it + 1);
  };

  if (it_begin < it_end) {
    fetch_ids(it_begin);
    fetch(it_begin);
  }
  for (int it = it_begin; it < it_end; ++it) {
    const int buf = it & 1;
    const u32x4 a_now[2] = {a_next[0], a_next[1]};
    u32x4 lo, hi;
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      lo[2 * d] = __builtin_amdgcn_perm(r1[d], r0[d], 0x05040100);
      lo[2 * d + 1] = __builtin_amdgcn_perm(r1[d], r0[d], 0x07060302);
      hi[2 * d] = __builtin_amdgcn_perm(r1[d + 2], r0[d + 2], 0x05040100);
      hi[2 * d + 1] = __builtin_amdgcn_perm(r1[d + 2], r0[d + 2], 0x07060302);
    }
    *reinterpret_cast<u32x4*>(&xs[buf][stage_at]) = lo;
    *reinterpret_cast<u32x4*>(&xs[buf][stage_at + 4]) = hi;
    if (it + 1 < it_end) fetch(it + 1);
    __syncthreads();
    tc_multiply<T, kTileF>(acc, a_now, xs[buf], wave * 32, lane);
  }
  const int fcol = f0 + wave * 32;
  if (fcol >= feat) return;
#pragma unroll
  for (int v = 0; v < TcAcc<T == 32>::kRegs; ++v) {
    const int row = TcAcc<T == 32>::row(v, lane);
    if (T < 16 && row >= T) continue;
    const int64_t off = (io * T + row) * feat + fcol + TcAcc<T == 32>::col(v, lane);
    if constexpr (OUT == 1) {
      if (add)
        __hip_atomic_fetch_add(static_cast<float*>(C) + off, acc.get(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      else
        static_cast<float*>(C)[off] = acc.get(v);
    } else {
      const _Float16 hv = (_Float16)acc.get(v);
      static_cast<uint16_t*>(C)[off] = __builtin_bit_cast(uint16_t, hv);
    }
  }
}

// The steps [s_begin, s_end) of row tile io for the features [f0, f0 + 32 * NTL), by a workgroup of
// 32 / NTL wavefronts: 8 with all four 32-feature accumulators of a 128-feature slice, or (what is
// launched) 16 with two -- 64 features; half the accumulators and half the staged bytes per
// wavefront, so that 16 fit the register file.  Wavefront w takes steps s_begin + w, + WAVES, ...,
// gathers the step's 32 rows of B itself (lane: k pairs kp, kp + KP, ... and 8-feature chunk
// fc) into its own piece of LDS -- no workgroup barrier in the loop, the LDS operations of one
// wavefront execute in order -- and the partial results are added through LDS, one 32-feature
// tile at a time; store(row in tile, feature, sum) receives every sum once.  The steps are a chain
// per wavefront (a step is a round trip to memory): more wavefronts per tile shorten it.
// lds: WAVES * 16 * 32 * NTL words (64 KB either way).  Ends with LDS reads: a caller that goes on
// to another tile puts a workgroup barrier in between.
template <int T, int NTL, class Store>
__device__ __forceinline__ void tcspmm_long_steps(uint32_t* __restrict__ lds, int feat, int64_t io, int f0,
                                                  int s_begin, int s_end, const uint16_t* __restrict__ A,
                                                  const uint16_t* __restrict__ B,
                                                  const int32_t* __restrict__ indptr,
                                                  const int32_t* __restrict__ indices, Store store) {
  using Acc = TcAcc<T == 32>;
  constexpr int WAVES = 32 / NTL;  // wavefronts per workgroup
  constexpr int TF = 32 * NTL;     // features per workgroup
  constexpr int CH = TF / 8;       // 8-feature chunks of a staged row
  constexpr int KP = 64 / CH;      // k pairs a wavefront stages at once
  constexpr int Q = 16 / KP;       // ... times Q = the 16 k pairs of a step
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kp = lane / CH, fc = lane % CH;
  const bool stage_live = f0 + fc * 8 < feat;
  uint32_t* xs = lds + wave * (16 * TF);  // [k pair][feature]
  const int64_t g_begin = indptr[io], g_end = indptr[io + 1];
  const int64_t rows_total = (g_end - g_begin) * kGroup;
  const int32_t* rowlist = indices + g_begin * kGroup;

  Acc acc[NTL];
#pragma unroll
  for (int t = 0; t < NTL; ++t) acc[t].clear();

  // row ids one step (of this wavefront) before the rows of B, as in the kernel above
  int row_a[Q], row_b[Q];
  auto fetch_ids = [&](int it) {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int64_t k = (int64_t)it * 32 + 2 * (kp + KP * q);
      row_a[q] = row_b[q] = 0;
      if (k < rows_total) row_a[q] = rowlist[k], row_b[q] = rowlist[k + 1];
    }
  };
  u32x4 r0[Q], r1[Q], a_next[2];
  auto fetch = [&](int it) {
    tc_load_a<T>(a_next, A, g_begin + 2 * it, g_end, lane);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      r0[q] = r1[q] = u32x4{0, 0, 0, 0};
      const int64_t k = (int64_t)it * 32 + 2 * (kp + KP * q);
      if (stage_live && k < rows_total) {
        r0[q] = *reinterpret_cast<const Halves8*>(B + (int64_t)row_a[q] * feat + f0 + fc * 8);
        r1[q] = *reinterpret_cast<const Halves8*>(B + (int64_t)row_b[q] * feat + f0 + fc * 8);
      }
    }
    if (it + WAVES < s_end) fetch_ids(it + WAVES);
  };

  // a wavefront without a step (fewer steps than wavefronts) only takes part in the sums
  if (s_begin + wave < s_end) {
    fetch_ids(s_begin + wave);
    fetch(s_begin + wave);
  }
  for (int it = s_begin + wave; it < s_end; it += WAVES) {
    const u32x4 a_now[2] = {a_next[0], a_next[1]};
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      u32x4 lo, hi;
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        lo[2 * d] = __builtin_amdgcn_perm(r1[q][d], r0[q][d], 0x05040100);
        lo[2 * d + 1] = __builtin_amdgcn_perm(r1[q][d], r0[q][d], 0x07060302);
        hi[2 * d] = __builtin_amdgcn_perm(r1[q][d + 2], r0[q][d + 2], 0x05040100);
        hi[2 * d + 1] = __builtin_amdgcn_perm(r1[q][d + 2], r0[q][d + 2], 0x07060302);
      }
      const int at = (kp + KP * q) * TF + tc_stage_col<T, TF>(kp + KP * q, fc * 8);
      *reinterpret_cast<u32x4*>(xs + at) = lo;
      *reinterpret_cast<u32x4*>(xs + at + 4) = hi;
    }
    if (it + WAVES < s_end) fetch(it + WAVES);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int t = 0; t < NTL; ++t) tc_multiply<T, TF>(acc[t], a_now, xs, t * 32, lane);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_wave_barrier();  // the next step's stores come after these reads
  }

  // ---- the partial tiles, one 32-feature tile at a time: a thread sums register v of lane l
  // over the wavefronts
  constexpr int REGS = Acc::kRegs;
  float* red = reinterpret_cast<float*>(lds);  // [wavefront][register][lane], at most 4 KB per wavefront
#pragma unroll
  for (int t = 0; t < NTL; ++t) {
    __syncthreads();  // staging pieces (t = 0) or the sums of the tile before are done with
#pragma unroll
    for (int v = 0; v < REGS; ++v) red[(wave * REGS + v) * 64 + lane] = acc[t].get(v);
    __syncthreads();
    for (int e = tid; e < REGS * 64; e += 64 * WAVES) {
      const int v = e >> 6, l = e & 63;
      float sum = 0.f;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) sum += red[(w * REGS + v) * 64 + l];
      const int row = Acc::row(v, l);
      const int fcol = f0 + t * 32 + Acc::col(v, l);
      if (fcol < feat && row < T) store(row, fcol, sum);
    }
  }
}

// fp16 output without a plan: the tiles the kernel above skips (more than kLongSteps steps).
template <int T, int NTL>
__global__ __launch_bounds__(64 * (32 / NTL)) void tcspmm_long_kernel(int feat, int64_t mb, int f_tiles,
                                                                      const uint16_t* __restrict__ A,
                                                                      const uint16_t* __restrict__ B,
                                                                      void* __restrict__ C,
                                                                      const int32_t* __restrict__ indptr,
                                                                      const int32_t* __restrict__ indices) {
  extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
  const int lane = threadIdx.x & 63;
  const int f0 = (int)(blockIdx.x % f_tiles) * (32 * NTL);
  // A workgroup looks at kLongScan row tiles and works on the long ones among them (most have
  // none): a workgroup per tile would start tens of thousands that only find out that their tile
  // is short, each holding 64 KB of LDS while it does.  Its tiles lie a whole grid apart -- long
  // tiles come in runs (the hub rows of a graph sorted by degree) and would otherwise queue up in
  // one workgroup.
  const int64_t io_stride = gridDim.x / f_tiles;
  // which of them are long: lane k asks for the group range of the k-th tile, all at once
  uint64_t todo;
  {
    const int64_t io = blockIdx.x / f_tiles + (int64_t)lane * io_stride;
    int64_t groups = 0;
    if (lane < kLongScan && io < mb) groups = indptr[io + 1] - indptr[io];
    todo = __ballot((groups * kGroup + 31) / 32 > kLongSteps);
  }
  bool used_lds = false;
  while (todo) {
    const int k_tile = __ffsll((long long)todo) - 1;
    todo &= todo - 1;
    const int64_t io = blockIdx.x / f_tiles + (int64_t)k_tile * io_stride;
    if (used_lds) __syncthreads();  // the sums of the tile before have been read
    used_lds = true;
    tcspmm_long_steps<T, NTL>(lds, feat, io, f0, 0, tile_steps(indptr, io), A, B, indptr, indices,
                              [&](int row, int fcol, float sum) {
                                const _Float16 hv = (_Float16)sum;
                                static_cast<uint16_t*>(C)[(io * T + row) * feat + fcol] = __builtin_bit_cast(uint16_t, hv);
                              });
  }
}

// ---- with a plan (stir_tc_plan): one launch of units, each a whole row tile or a piece of a long one.  Tiles of more
// than kWholeSteps steps are listed once by the plan, the longest first, and come before the others in the launch;
// those that the launch would end on are cut into pieces.  A unit is a workgroup of W wavefronts for (T rows) x (32 * NTL
// features) that take its steps in turn: wavefront w the steps w, w + W, ..., each with an image of its step's 32
// gathered rows of B in its own LDS -- no workgroup barrier in the loop, the LDS operations of one wavefront
// execute in order -- and the partial results meet in LDS at the end.  The image is the rows as they are, 16-byte
// unit c of row k at place c ^ swizzle(k), and comes out in MFMA operand order through the transposing read
// ds_read_b64_tr_b16 (see bsr_tile in bsr.hip; the XOR keeps the two blocks of 16 lanes that the LDS serves
// together on distinct banks).
// The pieces of a long tile leave fp32 partial tiles in the plan's scratch memory, and the workgroup that
// finishes last among the pieces of a tile (per feature tile: a counter in device memory, which that workgroup
// sets back to zero) adds them up in piece order and rounds once: the same bits whichever workgroup comes last.
// The partial tiles are written and read with device-coherent accesses (they pass the XCD's L2), so that no
// workgroup has to write back or invalidate a whole L2, as a release or acquire at device scope does.
constexpr int kWholeSteps = 32;
// A tile of more than this part of all steps is cut: about the units that run at a time, so that what is left whole
// ends with the others.  Pieces cost memory for partial tiles, at most 2 * kShares of them.  us with every tile above
// 32 steps cut / with parts of 4096 / 2048 / 1024 / 512 / 128: 169 k rows, 1.17 M nonzeros with hubs, 128 features, 16
// rows 62.1 / 62.0 / 61.9 / 61.3 / 63.2 / 166; 200 k, 4 M, 64, 32 rows 118 / 118 / 108 / 107 / 115 / 204; the same,
// skewed columns, 16 rows 57.3 / 57.2 / 56.7 / 62.8 / 80.2 / 80.4; 40 k, 1 M, 128, 32 rows 45.6 / 45.1 / 45.2 / 45.1 /
// 42.8 / 58.9.
constexpr int kShares = 2048;

struct TcPiece {
  int32_t tile, step_begin, step_end;
  int32_t slot;        // partial tile in the scratch memory; -1: the whole tile
  int32_t first_slot;  // of the tile's pieces
  int32_t pieces;      // of the tile
  int32_t multi;       // number of the tile among the long tiles
  int32_t pad;
};

typedef __fp16 tr16x4 __attribute__((__vector_size__(4 * sizeof(__fp16))));  // result type of the transposing LDS read
#define STIR_LDS __attribute__((address_space(3)))

// 8 consecutive k of one feature per lane: two transposing reads `next` bytes (four rows of k) apart
__device__ __forceinline__ f16x8 tc_read_b(const char* at, int next) {
  union {
    tr16x4 t[2];
    f16x8 v;
  } u;
  u.t[0] = __builtin_amdgcn_ds_read_tr16_b64_v4f16((STIR_LDS tr16x4*)(at));
  u.t[1] = __builtin_amdgcn_ds_read_tr16_b64_v4f16((STIR_LDS tr16x4*)(at + next));
  return u.v;
}

// four consecutive features of a row of C; aligned: as one store
template <int OUT>
__device__ __forceinline__ void tc_store4(void* C, int64_t off, const float4& v, bool aligned) {
  if constexpr (OUT == 1) {
    float* q = static_cast<float*>(C) + off;
    if (aligned)
      *reinterpret_cast<float4*>(q) = v;
    else
      q[0] = v.x, q[1] = v.y, q[2] = v.z, q[3] = v.w;
  } else {
    const _Float16 h[4] = {(_Float16)v.x, (_Float16)v.y, (_Float16)v.z, (_Float16)v.w};
    uint16_t* q = static_cast<uint16_t*>(C) + off;
    if (aligned) {
      uint2 out;
      out.x = (uint32_t)__builtin_bit_cast(uint16_t, h[0]) | ((uint32_t)__builtin_bit_cast(uint16_t, h[1]) << 16);
      out.y = (uint32_t)__builtin_bit_cast(uint16_t, h[2]) | ((uint32_t)__builtin_bit_cast(uint16_t, h[3]) << 16);
      *reinterpret_cast<uint2*>(q) = out;
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) q[u] = __builtin_bit_cast(uint16_t, h[u]);
    }
  }
}

// What a workgroup does that has left a partial tile (of one feature tile) in memory.
template <int T, int TF, int W, int OUT>
__device__ __forceinline__ void tc_add_pieces(const TcPiece& pc, int64_t io, int f_tile, int f_tiles, int feat, void* C,
                                              int aligned, float* scratch, uint32_t* arrived) {
  // Every wavefront waits until its stores have arrived, then one thread counts the workgroup
  // in: whoever counts last finds the partial tiles of all the others in memory.
  __shared__ int last_of_tile;
  const int tid = threadIdx.x, f0 = f_tile * TF;
  const int64_t elems = (int64_t)T * feat;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    uint32_t* counter = arrived + (int64_t)pc.multi * f_tiles + f_tile;
    const uint32_t before = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const bool last = before + 1 == (uint32_t)pc.pieces;
    if (last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
    last_of_tile = last;
  }
  __syncthreads();
  if (!last_of_tile) return;
  // C[tile, f0 .. f0 + TF) = the partial tiles added in piece order, rounded once
  float* first = scratch + (int64_t)pc.first_slot * elems;
  for (int w = tid; w < T * (TF / 4); w += 64 * W) {
    const int row = w / (TF / 4), fcol = f0 + (w % (TF / 4)) * 4;
    if (fcol >= feat) continue;
    const int64_t e = (int64_t)row * feat + fcol;
    float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int p0 = 0; p0 < pc.pieces; p0 += 8) {
      float4 y[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        y[u] = stir::CoherentPiece(first + min(p0 + u, pc.pieces - 1) * elems, (uint32_t)(elems * 4)).load((uint32_t)e);
      __builtin_amdgcn_sched_barrier(0);  // all eight, then the sums
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (p0 + u < pc.pieces) sum.x += y[u].x, sum.y += y[u].y, sum.z += y[u].z, sum.w += y[u].w;
    }
    tc_store4<OUT>(C, io * elems + e, sum, aligned);
  }
}

template <int T, int NTL, int W, int OUT>
__global__ __launch_bounds__(64 * W) void tcspmm_units_kernel(int feat, int64_t mb, int f_tiles, int64_t n_pieces,
                                                              const TcPiece* __restrict__ pieces,
                                                              const uint16_t* __restrict__ A,
                                                              const uint16_t* __restrict__ B, void* __restrict__ C,
                                                              int aligned, float* scratch, uint32_t* arrived,
                                                              const int32_t* __restrict__ indptr,
                                                              const int32_t* __restrict__ indices) {
  using Acc = TcAcc<T == 32>;
  static_assert(NTL == 1 || NTL == 2, "wider units: tcspmm_direct_kernel");
  constexpr int TF = 32 * NTL;
  constexpr int FCN = TF / 8;             // 16-byte units of a staged row
  constexpr int LOADS = FCN / 2;          // ... of a step's 32 rows per lane
  constexpr int XB = 32 * TF * 2;         // bytes of a wavefront's image
  constexpr int REGS = Acc::kRegs;
  constexpr int ATONCE = NTL * 8 / REGS ? NTL * 8 / REGS : 1;  // 32-feature tiles summed at a time: what fits
  constexpr int RB = ATONCE * REGS * 64 * 4;                   // bytes per wavefront of a sum
  __shared__ __attribute__((aligned(16))) char lds[W * (XB > RB ? XB : RB)];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int f_tile = (int)(blockIdx.x % f_tiles);
  const int64_t unit = blockIdx.x / f_tiles;
  const int f0 = f_tile * TF;
  TcPiece pc;
  pc.slot = -1;
  int64_t io = unit - n_pieces;
  int s_begin = 0, s_end = 0;
  if (unit < n_pieces) {
    pc = pieces[unit];
    io = pc.tile;
    // a plan made from other contents of indptr: stay inside the tile as it is now
    s_begin = pc.step_begin, s_end = min(pc.step_end, tile_steps(indptr, io));
  } else {
    if (io >= mb) return;
    s_end = tile_steps(indptr, io);
    if (s_end > kWholeSteps) return;  // in the list
  }
  const int64_t g_begin = indptr[io], g_end = indptr[io + 1];
  const int64_t rows_total = (g_end - g_begin) * kGroup;
  const int32_t* rowlist = indices + g_begin * kGroup;
  char* image = lds + wave * XB;

  auto swizzle = [](int k) {
    return (FCN == 4 ? 0 : 4 * ((k >> 1) & 1)) ^ (T == 32 ? 0 : 2 * ((k >> 3) & 1));
  };
  // staging role: unit c of the rows k0 + u * (64 / FCN)
  const int c = lane % FCN, k0 = lane / FCN;
  const bool live = f0 + 8 * c < feat;
  uint32_t put[LOADS];
#pragma unroll
  for (int u = 0; u < LOADS; ++u) {
    const int k = k0 + u * (64 / FCN);
    put[u] = (uint32_t)((k * FCN + (c ^ swizzle(k))) * 16);
  }
  // operand role: a block of 16 lanes reads four rows of two units
  const int sl = lane & 15, kr = sl >> 2;
  uint32_t get[NTL][T == 32 ? 1 : 2];
#pragma unroll
  for (int t = 0; t < NTL; ++t) {
    if constexpr (T == 32) {
      const int k = 8 * (lane >> 5) + kr, cc = 4 * t + 2 * ((lane >> 4) & 1) + ((sl & 3) >> 1);
      get[t][0] = (uint32_t)((k * FCN + (cc ^ swizzle(k))) * 16 + (sl & 1) * 8);
    } else {
      const int k = 8 * (lane >> 4) + kr;
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        const int cc = 4 * t + 2 * nt + ((sl & 3) >> 1);
        get[t][nt] = (uint32_t)((k * FCN + (cc ^ swizzle(k))) * 16 + (sl & 1) * 8);
      }
    }
  }

  Acc acc[NTL];
#pragma unroll
  for (int t = 0; t < NTL; ++t) acc[t].clear();

  // The row ids of a step are requested a step (of this wavefront) before its rows of B, so that a step costs
  // one memory round trip, not two in a row.
  int id = 0;
  auto fetch_ids = [&](int it) {
    const int64_t k = (int64_t)it * 32 + (lane & 31);
    id = k < rows_total ? rowlist[k] : -1;  // the second group of a tile's last step may not exist
  };
  u32x4 x[LOADS], a_next[2];
  auto fetch = [&](int it) {
    tc_load_a<T>(a_next, A, g_begin + 2 * it, g_end, lane);
#pragma unroll
    for (int u = 0; u < LOADS; ++u) {
      const int row = __shfl(id, k0 + u * (64 / FCN), 64);
      x[u] = u32x4{0, 0, 0, 0};
      if (live && row >= 0) x[u] = *reinterpret_cast<const Halves8*>(B + (int64_t)row * feat + f0 + 8 * c);
    }
    if (it + W < s_end) fetch_ids(it + W);
  };
  if (s_begin + wave < s_end) {
    fetch_ids(s_begin + wave);
    fetch(s_begin + wave);
  }
  for (int it = s_begin + wave; it < s_end; it += W) {
    const u32x4 a[2] = {a_next[0], a_next[1]};
#pragma unroll
    for (int u = 0; u < LOADS; ++u) *reinterpret_cast<u32x4*>(image + put[u]) = x[u];
    if (it + W < s_end) fetch(it + W);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int t = 0; t < NTL; ++t) {
      if constexpr (T == 32) {
#pragma unroll
        for (int d = 0; d < 2; ++d)
          acc[t].r = __builtin_amdgcn_mfma_f32_32x32x16_f16(
              __builtin_bit_cast(f16x8, a[d]), tc_read_b(image + get[t][0] + 16 * d * FCN * 16, 4 * FCN * 16),
              acc[t].r, 0, 0, 0);
      } else {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          acc[t].r[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
              __builtin_bit_cast(f16x8, a[0]), tc_read_b(image + get[t][nt], 4 * FCN * 16), acc[t].r[nt], 0, 0, 0);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_wave_barrier();  // the next step's stores come after these reads
  }

  // ---- the sums over the wavefronts, four consecutive features per thread
  const int used = min(W, s_end - s_begin);
  const int64_t elems = (int64_t)T * feat;
  float* red = reinterpret_cast<float*>(lds);  // [wavefront][tile][register][lane]
  const bool part = pc.slot >= 0;
  const stir::CoherentPiece partial(scratch + (part ? (int64_t)pc.slot * elems : 0), part ? (uint32_t)(elems * 4) : 0u);
#pragma unroll
  for (int t0 = 0; t0 < NTL; t0 += ATONCE) {
    __syncthreads();  // images, or the sums before, are done with
#pragma unroll
    for (int t = 0; t < ATONCE; ++t)
#pragma unroll
      for (int v = 0; v < REGS; ++v) red[((wave * ATONCE + t) * REGS + v) * 64 + lane] = acc[t0 + t].get(v);
    __syncthreads();
    for (int e = tid; e < T * ATONCE * 8; e += 64 * W) {
      const int row = e / (ATONCE * 8), t = e % (ATONCE * 8) / 8, col = e % 8 * 4;
      const int v = T == 32 ? (row & 3) + 4 * (row >> 3) : (row & 3) + 4 * (col >> 4);
      const int l = T == 32 ? col + 32 * ((row >> 2) & 1) : (col & 15) + 16 * (row >> 2);
      float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
      for (int w = 0; w < used; ++w) {
        const float4 o = *reinterpret_cast<const float4*>(red + ((w * ATONCE + t) * REGS + v) * 64 + l);
        sum.x += o.x, sum.y += o.y, sum.z += o.z, sum.w += o.w;
      }
      const int fcol = f0 + (t0 + t) * 32 + col;
      if (fcol >= feat) continue;
      if (!part) {
        tc_store4<OUT>(C, (io * T + row) * feat + fcol, sum, aligned);
      } else {
        partial.store((uint32_t)(row * feat + fcol), sum);
      }
    }
  }
  if (part) tc_add_pieces<T, TF, W, OUT>(pc, io, f_tile, f_tiles, feat, C, aligned, scratch, arrived);
}

// A unit of 128 features with the operands made in registers (lane_operand.h): a lane loads 8 features of the eight gathered
// rows 8 g ... 8 g + 7 of a step, and the row ids it needs for that; no LDS but for the sums over the W wavefronts at the
// end.  Narrower units, whose rows of B are less than 256 bytes, stay with the kernel above: 8 or 4 bytes a lane fill an L1 at
// 19 TB/s, 16 bytes at 33.  Through LDS / in registers, us: 169 k rows, 1.17 M nonzeros, 128 features, tiles of 16 rows 63.3 /
// 57.9, of 32 72 / 65.4; 100 k, 1 M, 256 features, 16 rows 90.4 / 84.4; 150 k, 3 M, skewed columns, 128 86.8 / 81.0.  Bound by the rows of B
// that miss an L2 (8.2 TB/s for rows out of 32 MB).
// D steps of a wavefront are on their way.  With two, a SIMD has registers for 4 / 3 / 2 wavefronts (tiles of 8 / 16 / 32 rows) and
// 32-row tiles leave 64 KB of sums for four wavefronts, 32 KB for two: few units at a time where tiles have a step or two for a
// wavefront, which hide nothing in themselves.  With one it has 5 / 4 / 3, and 32-row tiles pass half of their sums at a time
// through half of the LDS (tc_form says where which pays).
template <int T, int W, int OUT, int D>
__global__ __launch_bounds__(64 * W, T == 8 ? 4 : (T == 32 ? 2 : 3) + (D == 1)) void tcspmm_direct_kernel(
    int feat, int64_t mb, int f_tiles, int64_t n_pieces, const TcPiece* __restrict__ pieces, const uint16_t* __restrict__ A,
    const uint16_t* __restrict__ B, void* __restrict__ C, int aligned, float* scratch, uint32_t* arrived,
    const int32_t* __restrict__ indptr, const int32_t* __restrict__ indices) {
  constexpr int TF = 128, RH = T == 32 ? 2 : 1;  // RH: operands of 16 rows
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int f_tile = (int)(blockIdx.x % f_tiles);
  const int64_t unit = blockIdx.x / f_tiles;
  const int f0 = f_tile * TF;
  TcPiece pc;
  pc.slot = -1;
  int64_t io = unit - n_pieces;
  int s_begin = 0, s_end = 0;
  if (unit < n_pieces) {
    pc = pieces[unit];
    io = pc.tile;
    // a plan made from other contents of indptr: stay inside the tile as it is now
    s_begin = pc.step_begin, s_end = min(pc.step_end, tile_steps(indptr, io));
  } else {
    if (io >= mb) return;
    s_end = tile_steps(indptr, io);
    if (s_end > kWholeSteps) return;  // in the list
  }
  const int64_t g_begin = indptr[io];
  const int groups = (int)(indptr[io + 1] - g_begin);
  const int32_t* rowlist = indices + g_begin * kGroup;
  const uint16_t* Bf = B + min(f0 + 8 * c, feat - 8);  // features beyond feat repeat the last ones: nobody stores them

  f32x4 acc[RH][8];
#pragma unroll
  for (int r = 0; r < RH; ++r)
#pragma unroll
    for (int t = 0; t < 8; ++t) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Of a lane's group 2 step + g / 2; of one that is not there, what the group before it has: zeros are put in its place
  // when the step is multiplied, and nothing is asked for that does not exist.
  typedef int32_t Ids __attribute__((ext_vector_type(4), aligned(4)));
  auto group_of = [&](int step) { return min(2 * step + (g >> 1), groups - 1); };
  Ids ids[2];
  u32x4 x[D][8], a[D][RH];
  auto load_ids = [&](int step) {
    const int32_t* p = rowlist + group_of(step) * kGroup + 8 * (g & 1);
    ids[0] = *reinterpret_cast<const Ids*>(p), ids[1] = *reinterpret_cast<const Ids*>(p + 4);
  };
  auto fetch = [&](int s, int step) {  // whose ids are there
#pragma unroll
    for (int r = 0; r < RH; ++r) {
      a[s][r] = u32x4{0, 0, 0, 0};  // rows T ... 15 of the operand
      if (T >= 16 || c < T)
        a[s][r] = *reinterpret_cast<const Halves8*>(A + ((g_begin + group_of(step)) * T + 16 * r + c) * kGroup + 8 * (g & 1));
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) x[s][q] = *reinterpret_cast<const Halves8*>(Bf + (int64_t)ids[q / 4][q % 4] * feat);
  };
  auto multiply = [&](int s, int step) {
    if (2 * step + 1 >= groups) {
      const uint32_t there = g < 2 ? ~0u : 0u;
#pragma unroll
      for (int r = 0; r < RH; ++r)
#pragma unroll
        for (int d = 0; d < 4; ++d) a[s][r][d] &= there;
#pragma unroll
      for (int q = 0; q < 8; ++q)
#pragma unroll
        for (int w = 0; w < 4; ++w) x[s][q][w] &= there;
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const f16x8 b = __builtin_bit_cast(f16x8, stir::operand_of(x[s], t / 2, t % 2));
#pragma unroll
      for (int r = 0; r < RH; ++r)
        acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[s][r]), b, acc[r][t], 0, 0, 0);
    }
  };
  // wavefront w takes the steps w, w + W, ...; the ids of a step are asked for a step (of its own) before its rows of B
  int left = s_end - s_begin > wave ? (s_end - s_begin - wave + W - 1) / W : 0;
  if (left > 0) {
    int step = s_begin + wave;
    const auto later = [&](int by) { return min(step + by * W, s_end - 1); };
    load_ids(step);
    if constexpr (D == 1) {
#pragma unroll 1
      for (; left > 0; --left, step += W) {
        fetch(0, step);
        load_ids(later(1));
        multiply(0, step);
      }
    } else {
      fetch(0, step);
      load_ids(later(1));
      if (left > 1) fetch(1, step + W);
      load_ids(later(2));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
      for (; left >= 4; left -= 2) {
#pragma unroll
        for (int s = 0; s < 2; ++s, step += W) {
          multiply(s, step);
          __builtin_amdgcn_sched_barrier(0);
          fetch(s, step + 2 * W);
          load_ids(later(3));
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      multiply(0, step);  // one to three are left
      if (left > 2) fetch(0, step + 2 * W);
      if (left > 1) multiply(1, step + W);
      if (left > 2) multiply(0, step + 2 * W);
    }
  }

  // ---- the sums over the wavefronts, `ROUND` operands of 16 rows at a time: each adds 4 ROUND / W of the rows a lane has.
  // acc[r][t][v] is row 16 r + 4 g + v, feature 8 c + t.  Sixteen-bit results leave as they lie; floats are read four features to a
  // lane in the order of the row, so that a store is of whole lines (halves of lines: 169 k rows, 8-row tiles, 128 features 68.5
  // us, now 66.5).
  constexpr int ROUND = D == 1 ? 1 : RH;
  __shared__ __attribute__((aligned(16))) f32x4 sums[W][4 * ROUND][2][64];  // [e][lane ^ 8 e]: eight lanes in row order share no bank
  const int used = min(W, s_end - s_begin);
  const int64_t elems = (int64_t)T * feat;
  const bool part = pc.slot >= 0;
  const stir::CoherentPiece partial(scratch + (part ? (int64_t)pc.slot * elems : 0), part ? (uint32_t)(elems * 4) : 0u);
#pragma unroll
  for (int r0 = 0; r0 < RH; r0 += ROUND) {
    if (r0) __syncthreads();  // the sums before have been read
    if (wave < used) {
#pragma unroll
      for (int at = 0; at < 4 * ROUND; ++at)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const auto& o = acc[r0 + (at >> 2)];
          sums[wave][at][e][lane ^ (8 * e)] = f32x4{o[4 * e][at & 3], o[4 * e + 1][at & 3], o[4 * e + 2][at & 3], o[4 * e + 3][at & 3]};
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4 * ROUND / W; ++q) {
      const int from = wave * (4 * ROUND / W) + q, at = 4 * r0 + from;
      const bool floats = OUT == 1 || part;
      f32x4 o[2];
      int place[2];  // of o[i] in sums: lane ^ 8 e, with 64 e
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int piece = 64 * i + lane, e = floats ? piece & 1 : i;  // in row order: row piece / 32, features 4 (piece % 32) ...
        place[i] = 64 * e + ((floats ? piece >> 1 : lane) ^ (8 * e));
        o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int w = 0; w < W; ++w) {
        if (w >= used) continue;
#pragma unroll
        for (int i = 0; i < 2; ++i) o[i] += sums[w][from][0][place[i]];
      }
      if (!floats) {
        const int row = 16 * (at >> 2) + 4 * g + (at & 3);
        u32x4 w;
#pragma unroll
        for (int t = 0; t < 4; ++t)
          w[t] = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)o[t / 2][2 * (t % 2)]) |
                 (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)o[t / 2][2 * (t % 2) + 1]) << 16;
        if (f0 + 8 * c < feat && (T >= 16 || row < T))
          *reinterpret_cast<Halves8*>(static_cast<uint16_t*>(C) + (io * T + row) * feat + f0 + 8 * c) = w;
        continue;
      }
#pragma unroll
      for (int i = 0; i < (T == 8 ? 1 : 2); ++i) {  // of 8 rows the other half is no rows
        const int row = 16 * (at >> 2) + 8 * i + 4 * (lane >> 5) + (at & 3), fcol = f0 + 4 * (lane & 31);
        if (fcol >= feat) continue;
        const float4 v = make_float4(o[i][0], o[i][1], o[i][2], o[i][3]);
        if (part) partial.store((uint32_t)(row * feat + fcol), v);
        else *reinterpret_cast<Float4*>(static_cast<float*>(C) + (io * T + row) * feat + fcol) = Float4{v.x, v.y, v.z, v.w};
      }
    }
  }
  if (part) tc_add_pieces<T, TF, W, OUT>(pc, io, f_tile, f_tiles, feat, C, aligned, scratch, arrived);
}

constexpr int kLongTF = 32 * kLongNT, kLongWaves = 32 / kLongNT;
constexpr size_t kLongLds = size_t(kLongWaves) * 16 * kLongTF * sizeof(uint32_t);

int check_args(int32_t out_dtype, int32_t mb, int32_t tile_size, int32_t group_size, int32_t feat, int64_t nnzb,
               const void* d_A, const void* d_B, void* d_C, const int32_t* d_indptr, const int32_t* d_indices) {
  STIR_REQUIRE(out_dtype == STIR_F16 || out_dtype == STIR_F32, "tc_spmm: out_dtype must be STIR_F16 or STIR_F32");
  STIR_REQUIRE((tile_size == 8 || tile_size == 16 || tile_size == 32) && group_size == kGroup,
               "tc_spmm: tile_size=%d group_size=%d; the MFMA path needs t in {8, 16, 32} and g=16", tile_size,
               group_size);
  STIR_REQUIRE(mb >= 0 && nnzb >= 0, "tc_spmm: bad sizes");
  STIR_REQUIRE(feat > 0 && feat % 32 == 0, "tc_spmm: feat=%d must be a multiple of 32", feat);
  STIR_REQUIRE(mb == 0 || (d_B && d_C && d_indptr && (nnzb == 0 || (d_A && d_indices))),
               "tc_spmm: null pointer argument");
  return 0;
}

template <int T>
int launch_unplanned(bool out32, int32_t mb, int32_t feat, const uint16_t* A, const uint16_t* B, void* d_C,
                     const int32_t* d_indptr, const int32_t* d_indices, hipStream_t st) {
  const int f_tiles = (int)stir::ceil_div(feat, kTileF);
  const int64_t blocks = (int64_t)mb * f_tiles;
  STIR_REQUIRE(blocks < (int64_t(1) << 31), "tc_spmm: too many tiles for one launch");
  if (out32) {
    hipLaunchKernelGGL(tcspmm_clear_long_kernel, dim3((unsigned)blocks), dim3(256), 0, st, T, feat, (int64_t)mb,
                       f_tiles, static_cast<float*>(d_C), d_indptr);
    STIR_LAUNCH_CHECK();
    hipLaunchKernelGGL((tcspmm_kernel<T, 1, true>), dim3((unsigned)blocks, kSplit), dim3(256), 0, st, feat,
                       (int64_t)mb, f_tiles, A, B, d_C, d_indptr, d_indices);
  } else {
    // the two launches write different row tiles
    const int long_f_tiles = (int)stir::ceil_div(feat, kLongTF);
    const int64_t long_blocks = stir::ceil_div((int64_t)mb, kLongScan) * long_f_tiles;
    STIR_REQUIRE(long_blocks < (int64_t(1) << 31), "tc_spmm: too many tiles for one launch");
    hipLaunchKernelGGL((tcspmm_kernel<T, 0, false>), dim3((unsigned)blocks), dim3(256), 0, st, feat, (int64_t)mb,
                       f_tiles, A, B, d_C, d_indptr, d_indices);
    STIR_LAUNCH_CHECK();
    hipLaunchKernelGGL((tcspmm_long_kernel<T, kLongNT>), dim3((unsigned)long_blocks), dim3(64 * kLongWaves), kLongLds,
                       st, feat, (int64_t)mb, long_f_tiles, A, B, d_C, d_indptr, d_indices);
  }
  STIR_LAUNCH_CHECK();
  return 0;
}

// How a product with a plan is launched.
struct TcForm {
  int tiles;      // of 32 features to a unit: 4 by tcspmm_direct_kernel, else by tcspmm_units_kernel
  int waves;      // to a unit
  bool one_step;  // tcspmm_direct_kernel with one step of a wavefront on its way
};

TcForm tc_form(int T, bool out32, int64_t mb, int feat, int64_t nnzb, int64_t n_pieces) {
  // Units of 128 features above 64 (tcspmm_direct_kernel), their last one however full; us with units of 64 features, by the
  // other kernel, / of 128: 20 k rows, 300 k nonzeros, 128 features 16.2 / 14.4, 100 k, 500 k, 96 33.6 / 26.0, 120 k, 600 k, 160
  // 61.2 / 53.7, 60 k, 900 k, 192 66.1 / 56.4; 33 k, 160 features, 8-, 16-, 32-row tiles of 5 to 20 steps 0.82 to 0.98 of the time;
  // and of 64 features alone 60 k, 900 k 25.7 / 29.5, 200 k, 4 M 66 / 80.  Two exceptions:
  //   128 features, many 8-row tiles of several steps: there is little of A to fetch twice, and the two units of 64 of a tile are
  //   neighbours, so that every other XCD has the same half of B in its L2: 50 k rows, 1.25 M nonzeros (6.5 steps) 42 / 47, 169 k,
  //   4.2 M 154 / 165, skewed columns 123 / 135 (but of 50 k rows 40 / 35); 4 steps 116 / 110, 2.2 steps 29.9 / 30.1, 4125 tiles of
  //   6.3 steps 26.4 / 25.2;
  //   32 features in a unit of 128 of their own, 32-row tiles, of which hardly a turn is resident (64 KB of sums each): 12 k rows, 49
  //   k nonzeros, 160 features 10.2 / 10.9; with units of 32 KB below that is no reason: 33 k, 165 k, 160 15.7 / 15.3.  Of 8-row tiles
  //   where the empty part is about what another turn is of: 14 k, 370 k, 160 20.7 / 22.1 (1300 to 2000 tiles 0.95 to 0.97 of the
  //   time, 2.4 to 13 steps; fewer 1.02, more 0.99 to 1.4).
  const int64_t wide_units = (mb + n_pieces) * stir::ceil_div(feat, 128);
  const bool halves = T == 8 && feat == 128 && mb >= 6000 && nnzb >= 9 * mb;
  const bool lone = feat % 128 == 32 && (T == 32 ? wide_units < 1300 : T == 8 && wide_units >= 2600 && wide_units < 4000);
  const int tiles = feat <= 32 ? 1 : feat > 64 && !halves && !lone ? 4 : 2;
  const int64_t units = (mb + n_pieces) * stir::ceil_div(feat, 32 * tiles);
  // Four wavefronts shorten a unit, two leave fewer of them without a step: 64 features, 25 k tiles of 1.5 and of 5.2
  // steps 49.3 against 36.5 and 71.7 against 57.5 us; 3025 tiles of 2.7 steps 12.5 against 13.7, 3125 of 14.7
  // 35.5 against 38.3 us; 32 features, 12.5 k tiles of 2.7 steps 25.3 against 27.6, 25 k of 1.5 31.6 against 28.1.
  const int waves = units >= (tiles == 4 ? 5000 : 8000) && (tiles > 1 || nnzb < 4 * mb) ? 2 : 4;
  // One step on its way (of two) where more units at a time count for more than the loads of a wavefront behind its products; us
  // with one / two:
  //   8-row tiles: four wavefronts 0.98 to 1.02, and many units of two: 169 k rows, 1.9 M nonzeros, 192 features (42 k units) 100.5 /
  //   104.1, 850 k 72.5 / 75.5; but 33 k, 200 k, 192 (8250) 25.7 / 24.6, 20 k, 80 k, 224 (5000) 20.3 / 18.6;
  //   32-row tiles, four wavefronts, from three turns of 64 KB on: 75 k rows, 375 k nonzeros, 192 features 33.4 / 40.1, 60 k, 300 k,
  //   skewed columns 27.7 / 33.3; less of them 20 k, 80 k, 128 (625 units) 16.1 / 15.8;
  //   two wavefronts, a last unit at most half full and a step or two for each: 169 k rows, 850 k nonzeros of skewed columns, 192
  //   features, 32 rows 85 / 91.7, 16-bit results 69.4 / 76.3, 16 rows (2.7 steps) 80.3 / 83.3, 16-bit 57.7 / 63.1; but of uniform
  //   columns 81.9 / 84.3 and 68.4 / 65.7, and with more steps 1.01 to 1.04 of the time.
  const bool part_empty = feat % 128 != 0 && feat % 128 <= 64;
  const bool one_step = T == 8    ? waves == 4 || units >= 20000
                        : T == 16 ? waves == 2 && part_empty && nnzb < (out32 ? 6 : 5) * mb
                        : waves == 4 ? units >= 1300
                                     : part_empty && nnzb < 10 * mb;
  return {tiles, waves, tiles == 4 && one_step};
}

template <int T>
int launch_planned(bool out32, int32_t mb, int32_t feat, int64_t nnzb, int64_t n_pieces, const TcPiece* d_pieces, float* d_scratch,
                   uint32_t* d_arrived, const uint16_t* A, const uint16_t* B, void* d_C, const int32_t* d_indptr,
                   const int32_t* d_indices, hipStream_t st) {
  const TcForm form = tc_form(T, out32, mb, feat, nnzb, n_pieces);
  const int f_tiles = (int)stir::ceil_div(feat, 32 * form.tiles);
  const int64_t blocks = (mb + n_pieces) * f_tiles;
  STIR_REQUIRE(blocks < (int64_t(1) << 31), "tc_spmm: too many tiles for one launch");
  const int aligned = reinterpret_cast<uintptr_t>(d_C) % (out32 ? 16 : 8) == 0;
#define STIR_TC_GO(KERNEL, W)                                                                                        \
  hipLaunchKernelGGL(KERNEL, dim3((unsigned)blocks), dim3(64 * W), 0, st, feat, (int64_t)mb, f_tiles, n_pieces,      \
                     d_pieces, A, B, d_C, aligned, d_scratch, d_arrived, d_indptr, d_indices)
#define STIR_TC(NTL, W)                                                                                              \
  do {                                                                                                               \
    if (out32) STIR_TC_GO((tcspmm_units_kernel<T, NTL, W, 1>), W);                                                   \
    else STIR_TC_GO((tcspmm_units_kernel<T, NTL, W, 0>), W);                                                         \
  } while (0)
#define STIR_TC_D(W, D)                                                                                              \
  do {                                                                                                               \
    if (out32) STIR_TC_GO((tcspmm_direct_kernel<T, W, 1, D>), W);                                                    \
    else STIR_TC_GO((tcspmm_direct_kernel<T, W, 0, D>), W);                                                          \
  } while (0)
  if (form.tiles == 1) {
    if (form.waves == 2) STIR_TC(1, 2); else STIR_TC(1, 4);
  } else if (form.tiles == 2) {
    if (form.waves == 2) STIR_TC(2, 2); else STIR_TC(2, 4);
  } else if constexpr (T == 8) {
    if (form.waves == 4) STIR_TC_D(4, 1);
    else if (form.one_step) STIR_TC_D(2, 1);
    else STIR_TC_D(2, 2);
  } else if constexpr (T == 16) {
    if (form.waves == 4) STIR_TC_D(4, 2);
    else if (form.one_step) STIR_TC_D(2, 1);
    else STIR_TC_D(2, 2);
  } else {
    if (form.waves == 4 && form.one_step) STIR_TC_D(4, 1);
    else if (form.waves == 4) STIR_TC_D(4, 2);
    else if (form.one_step) STIR_TC_D(2, 1);
    else STIR_TC_D(2, 2);
  }
#undef STIR_TC_D
#undef STIR_TC
#undef STIR_TC_GO
  STIR_LAUNCH_CHECK();
  return 0;
}

}  // namespace

// The form of a product with a plan of so many pieces: tiles of 32 features to a unit, 8 times the wavefronts, 64 for one
// step on its way; -1 for what no product is.  For the tests, which say what they cover.
extern "C" int stir_tc_form(int32_t tile_size, int32_t out_dtype, int32_t mb, int32_t feat, int64_t nnzb, int64_t n_pieces) {
  if ((tile_size != 8 && tile_size != 16 && tile_size != 32) || (out_dtype != STIR_F16 && out_dtype != STIR_F32) || mb <= 0 ||
      feat <= 0 || nnzb < 0 || n_pieces < 0)
    return -1;
  const TcForm f = tc_form(tile_size, out_dtype == STIR_F32, mb, feat, nnzb, n_pieces);
  return f.tiles + 8 * f.waves + 64 * f.one_step;
}

extern "C" int stir_tc_spmm_f16(int32_t out_dtype, int32_t mb, int32_t tile_size, int32_t group_size,
                                int32_t feat, int64_t nnzb, const void* d_A, const void* d_B, void* d_C,
                                const int32_t* d_indptr, const int32_t* d_indices, void* stream) {
  if (check_args(out_dtype, mb, tile_size, group_size, feat, nnzb, d_A, d_B, d_C, d_indptr, d_indices)) return -1;
  if (mb == 0) return 0;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint16_t* A = static_cast<const uint16_t*>(d_A);
  const uint16_t* B = static_cast<const uint16_t*>(d_B);
  const bool out32 = out_dtype == STIR_F32;
  switch (tile_size) {
    case 8: return launch_unplanned<8>(out32, mb, feat, A, B, d_C, d_indptr, d_indices, st);
    case 16: return launch_unplanned<16>(out32, mb, feat, A, B, d_C, d_indptr, d_indices, st);
    default: return launch_unplanned<32>(out32, mb, feat, A, B, d_C, d_indptr, d_indices, st);
  }
}

struct stir_tc_plan {
  int32_t mb = 0;
  int device = 0;
  int64_t n_pieces = 0, n_multi = 0, slots = 0;
  TcPiece* d_pieces = nullptr;
  // Counters, and behind them the partial tiles, made anew by the launch that needs more.  A counter per cut tile and
  // feature tile: the pieces that have finished in the running launch; zero between launches (the workgroup that
  // counts last clears its counter).
  uint32_t* d_arrived = nullptr;
  size_t arrived_bytes = 0, scratch_bytes = 0;
};

extern "C" int stir_tc_plan_destroy(stir_tc_plan* plan) {
  if (!plan) return 0;
  if (plan->d_pieces) (void)hipFree(plan->d_pieces);
  if (plan->d_arrived) (void)hipFree(plan->d_arrived);
  delete plan;
  return 0;
}

extern "C" int stir_tc_plan_create(stir_tc_plan** plan, int32_t mb, const int32_t* d_indptr, void* stream) {
  STIR_REQUIRE(plan, "tc_plan_create: plan is null");
  STIR_REQUIRE(mb >= 0 && (mb == 0 || d_indptr), "tc_plan_create: bad arguments");
  hipStream_t st = static_cast<hipStream_t>(stream);
  std::vector<int32_t> ptr(size_t(mb) + 1, 0);
  if (mb > 0) {
    STIR_HIP(hipMemcpyAsync(ptr.data(), d_indptr, sizeof(int32_t) * ptr.size(), hipMemcpyDeviceToHost, st));
    STIR_HIP(hipStreamSynchronize(st));
  }
  // the long tiles, longest first (ties in tile order)
  std::vector<std::pair<int32_t, int32_t>> longs;  // (steps, tile)
  int64_t all_steps = 0;
  for (int32_t io = 0; io < mb; ++io) {
    STIR_REQUIRE(ptr[io] <= ptr[io + 1], "tc_plan_create: indptr decreases at tile %d", io);
    const int64_t steps = ((int64_t)(ptr[io + 1] - ptr[io]) * kGroup + 31) / 32;
    if (steps > kWholeSteps) longs.emplace_back((int32_t)steps, io);
    all_steps += steps;
  }
  const int64_t most = std::max<int64_t>(kWholeSteps, all_steps / kShares);
  std::stable_sort(longs.begin(), longs.end(),
                   [](const std::pair<int32_t, int32_t>& a, const std::pair<int32_t, int32_t>& b) { return a.first > b.first; });
  std::vector<TcPiece> pieces;
  int64_t slots = 0, n_multi = 0;
  for (const auto& lt : longs) {
    const int32_t steps = lt.first, io = lt.second;
    const int32_t n = (int32_t)((steps + most - 1) / most);  // pieces of equal length
    const int32_t len = (steps + n - 1) / n;
    STIR_REQUIRE(slots + n < (int64_t(1) << 31), "tc_plan_create: too many pieces");
    for (int32_t p = 0; p < n; ++p)
      pieces.push_back(TcPiece{io, p * len, std::min(steps, (p + 1) * len), n > 1 ? (int32_t)(slots + p) : -1,
                               (int32_t)slots, n, (int32_t)n_multi, 0});
    if (n > 1) slots += n, ++n_multi;
  }
  stir_tc_plan* p = new stir_tc_plan();
  p->mb = mb;
  p->n_pieces = (int64_t)pieces.size();
  p->n_multi = n_multi;
  p->slots = slots;
  hipError_t e = hipGetDevice(&p->device);
  if (e == hipSuccess && !pieces.empty()) {
    e = hipMalloc(reinterpret_cast<void**>(&p->d_pieces), sizeof(TcPiece) * pieces.size());
    if (e == hipSuccess)
      e = hipMemcpyAsync(p->d_pieces, pieces.data(), sizeof(TcPiece) * pieces.size(), hipMemcpyHostToDevice, st);
  }
  if (e == hipSuccess) e = hipStreamSynchronize(st);  // the host vectors go away
  if (e != hipSuccess) {
    stir_tc_plan_destroy(p);
    return stir::fail("tc_plan_create: %s", hipGetErrorString(e));
  }
  *plan = p;
  return 0;
}

extern "C" size_t stir_tc_plan_counter_bytes(const stir_tc_plan* plan, int32_t feat) {
  if (!plan || feat <= 0) return 0;
  return (size_t(plan->n_multi) * size_t(stir::ceil_div(feat, 32)) * sizeof(uint32_t) + 255) / 256 * 256;
}

extern "C" size_t stir_tc_plan_partial_bytes(const stir_tc_plan* plan, int32_t tile_size, int32_t feat) {
  if (!plan || tile_size <= 0 || feat <= 0) return 0;
  return size_t(plan->slots) * size_t(tile_size) * size_t(feat) * sizeof(float);
}

extern "C" int stir_tc_spmm_f16_workspace(const stir_tc_plan* plan, int32_t out_dtype, int32_t mb, int32_t tile_size,
                                          int32_t group_size, int32_t feat, int64_t nnzb, const void* d_A,
                                          const void* d_B, void* d_C, const int32_t* d_indptr, const int32_t* d_indices,
                                          void* d_counters, void* d_partials, void* stream) {
  STIR_REQUIRE(plan, "tc_spmm_planned: plan is null");
  if (check_args(out_dtype, mb, tile_size, group_size, feat, nnzb, d_A, d_B, d_C, d_indptr, d_indices)) return -1;
  STIR_REQUIRE(plan->mb == mb, "tc_spmm_planned: the plan was made for %d row tiles, not %d", plan->mb, mb);
  int device = 0;
  STIR_HIP(hipGetDevice(&device));
  STIR_REQUIRE(device == plan->device, "tc_spmm_planned: the plan lives on device %d, the current device is %d",
               plan->device, device);
  STIR_REQUIRE(plan->n_multi == 0 || (d_counters && d_partials), "tc_spmm_planned: null workspace");
  if (mb == 0) return 0;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint16_t* A = static_cast<const uint16_t*>(d_A);
  const uint16_t* B = static_cast<const uint16_t*>(d_B);
  const bool out32 = out_dtype == STIR_F32;
  float* partials = static_cast<float*>(d_partials);
  uint32_t* counters = static_cast<uint32_t*>(d_counters);
  switch (tile_size) {
    case 8:
      return launch_planned<8>(out32, mb, feat, nnzb, plan->n_pieces, plan->d_pieces, partials, counters, A, B, d_C,
                               d_indptr, d_indices, st);
    case 16:
      return launch_planned<16>(out32, mb, feat, nnzb, plan->n_pieces, plan->d_pieces, partials, counters, A, B, d_C,
                                d_indptr, d_indices, st);
    default:
      return launch_planned<32>(out32, mb, feat, nnzb, plan->n_pieces, plan->d_pieces, partials, counters, A, B, d_C,
                                d_indptr, d_indices, st);
  }
}

extern "C" int stir_tc_spmm_f16_planned(stir_tc_plan* plan, int32_t out_dtype, int32_t mb, int32_t tile_size,
                                        int32_t group_size, int32_t feat, int64_t nnzb, const void* d_A,
                                        const void* d_B, void* d_C, const int32_t* d_indptr,
                                        const int32_t* d_indices, void* stream) {
  STIR_REQUIRE(plan, "tc_spmm_planned: plan is null");
  // memory of the plan is made only for a call that goes on to launch
  if (check_args(out_dtype, mb, tile_size, group_size, feat, nnzb, d_A, d_B, d_C, d_indptr, d_indices)) return -1;
  int device = 0;
  STIR_HIP(hipGetDevice(&device));
  const size_t counters = stir_tc_plan_counter_bytes(plan, feat), partials = stir_tc_plan_partial_bytes(plan, tile_size, feat);
  if (plan->mb == mb && plan->device == device && mb > 0 &&
      (counters > plan->arrived_bytes || partials > plan->scratch_bytes)) {
    const size_t more_counters = std::max(counters, plan->arrived_bytes);
    const size_t more_partials = std::max(partials, plan->scratch_bytes);
    if (plan->d_arrived) STIR_HIP(hipFree(plan->d_arrived));
    plan->d_arrived = nullptr;
    plan->arrived_bytes = plan->scratch_bytes = 0;
    STIR_HIP(hipMalloc(reinterpret_cast<void**>(&plan->d_arrived), more_counters + more_partials));
    STIR_HIP(hipMemsetAsync(plan->d_arrived, 0, more_counters, static_cast<hipStream_t>(stream)));
    plan->arrived_bytes = more_counters, plan->scratch_bytes = more_partials;
  }
  char* scratch = reinterpret_cast<char*>(plan->d_arrived);
  return stir_tc_spmm_f16_workspace(plan, out_dtype, mb, tile_size, group_size, feat, nnzb, d_A, d_B, d_C, d_indptr, d_indices,
                                    scratch, scratch ? scratch + plan->arrived_bytes : nullptr, stream);
}
