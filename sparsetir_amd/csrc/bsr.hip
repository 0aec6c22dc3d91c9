// BSR SpMM on the gfx950 matrix cores: Y[i-th block row] = sum over stored blocks p of
// A_p (blk x blk) * X[indices[p]-th block of rows], 16-bit inputs, fp32 accumulation.
//
// Slices of 32 rows, 16 where the block is an odd multiple of that: a wavefront owns them x 128 or 256 features, loads the
// rows of X into registers eight features to a lane and makes the MFMA B operand (8 consecutive k of one feature per lane)
// out of them with v_perm: no LDS and no other wavefront is in the way (bsr_direct_kernel, bsr_wave_kernel,
// bsr16_direct_kernel, bsr16_wave_kernel).  In small launches, and in larger ones of 16-row slices, the wavefronts of a
// workgroup take the steps of one tile in turn.
// Slices of 64 rows (blocks that are a multiple of 64, where there are many): a workgroup of four wavefronts owns 64 rows
// and a 128*NT-wide slice of the feature axis; both operands go through LDS (bsr_tile).  Small launches of long block rows
// whose tiles of 128 features leave CUs idle, whatever the block, by bsr_split_kernel.
#include <hip/hip_fp16.h>

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "lane_operand.h"
#include "../../include/sparsetir_amd.h"

namespace {

using stir::Halves8;
using stir::kWave;

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __fp16 tr16x4 __attribute__((__vector_size__(4 * sizeof(__fp16))));  // result type of the transposing LDS read
#define STIR_LDS __attribute__((address_space(3)))

constexpr int kTileF = 128;  // features per workgroup
constexpr int kTileK = 32;   // k rows staged per step
constexpr int kWaveF = 256;  // features per wavefront where a wavefront owns a tile

template <bool BF16>
__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

template <bool BF16>
__device__ __forceinline__ uint16_t to16(float v) {
  if constexpr (BF16) {
    return __builtin_bit_cast(uint16_t, (__bf16)v);  // v_cvt_pk_bf16_f32: nearest even, NaN stays a (quiet) NaN
  } else {
    _Float16 h = (_Float16)v;
    return __builtin_bit_cast(uint16_t, h);
  }
}

// Workgroup -> (slice, feature tile).  Workgroups are dispatched round-robin over the 8 XCDs, each with
// its own L2.  All slices of one feature tile read the same columns of X (nb*blk rows x TF features): the
// tiles are numbered feature tile by feature tile and XCD x takes the x-th eighth of them, so it works on an
// eighth of the feature tiles, one after the other, whatever their number.  (Feature tiles dealt out whole left
// XCDs idle when there were not 8 k of them, and dealt out in turn put all of X through every L2:
// 5 feature tiles, 327 x 370 blocks of 32, 1216 features: 201 -> 122 us; 10 feature tiles, 98 x 90 blocks of
// 64, 2432 features: 102 -> 79 us.)  The grid is 8 * ceil(slices * f_tiles / 8) workgroups.
__device__ __forceinline__ bool decode_tile(int64_t L, int64_t slices, int f_tiles, int64_t& slice,
                                            int& f_tile) {
  const int64_t total = slices * f_tiles, per = (total + 7) >> 3;
  const int64_t t = (L & 7) * per + (L >> 3);
  f_tile = (int)(t / slices);
  slice = t % slices;
  return (L >> 3) < per && t < total;
}

// The same when the block rows are numbered by rank (row_of_rank), `sub` slices each that stay together: they read the
// same X.  Where XCDs share a feature tile, each takes ranks from the whole range in proportion to its share, so that
// none has the long ones.  With n of them here and m at another XCD, the k-th here comes after those there whose
// (2 k' + 1) / m is smaller than (2 k + 1) / n.
__device__ __forceinline__ bool decode_ranked(int64_t L, int64_t slices, int sub, int f_tiles, int64_t& slice,
                                              int& f_tile) {
  const int64_t rows = slices / sub, total = rows * f_tiles, per = (total + 7) >> 3;
  const int x = (int)(L & 7);
  const uint32_t at = (uint32_t)(L >> 3);
  const int64_t t = x * per + at / sub;
  if (at / sub >= per || t >= total) return false;
  f_tile = (int)(t / rows);
  const int64_t lo = f_tile * rows, hi = lo + rows;
  const int64_t first = max(x * per, lo), n = min((x + 1) * per, hi) - first, k = t - first;
  int64_t rank = k;
  for (int y = (int)(lo / per); y < 8 && y * per < hi; ++y) {
    if (y == x) continue;
    const int64_t m = min((y + 1) * per, hi) - max(y * per, lo);
    rank += ((2 * k + 1) * m + n - (y > x)) / (2 * n);
  }
  slice = rank * sub + at % sub;
  return true;
}

// The block row of rank `rank` when the block rows are ordered by their number of blocks, longest first, equal ones
// by number.  Workgroups of a launch that walk block rows of equal length side by side move through X together (block
// columns ascend in a block row) and share a window of it in L2, one turn of resident workgroups after the other:
// nothing synchronises them, the order only decides what L2 holds.  Every wavefront finds the row from indptr by
// itself, the length of that rank by halving, then the place among the rows of that length.  More block rows than a
// wavefront can hold are ranked in equal groups, one after the other: 2048 x 512 blocks of 32, 10 %, 4096 features 1574 us,
// 2562 as they come; 1500 x 400, 8 %, 2048 features 354, 498; 2048 x 1024 blocks of 16, 10 %, 1024 features 306, 432.
constexpr int kRankChunks = 16;
constexpr int kRankRows = kRankChunks * kWave;  // block rows whose lengths a wavefront can hold
__device__ __forceinline__ int row_of_rank(const int32_t* __restrict__ indptr, int rows, int rank) {
  const int groups = (rows + kRankRows - 1) / kRankRows, size = (rows + groups - 1) / groups;
  const int first = rank / size * size;
  indptr += first, rank -= first, rows = min(size, rows - first);
  const int lane = threadIdx.x & 63;
  int len[kRankChunks], most = 0, least = INT32_MAX;
#pragma unroll
  for (int q = 0; q < kRankChunks; ++q) {
    const int i = q * kWave + lane;
    len[q] = -1;
    if (i < rows) {
      len[q] = indptr[i + 1] - indptr[i];
      most = max(most, len[q]), least = min(least, len[q]);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    most = max(most, __shfl_xor(most, off, kWave));
    least = min(least, __shfl_xor(least, off, kWave));
  }
  auto reach = [&](int at_least) {  // rows of that length or longer
    int n = 0;
#pragma unroll
    for (int q = 0; q < kRankChunks; ++q)
      if (q * kWave < rows) n += __popcll(__ballot(len[q] >= at_least));
    return n;
  };
  // the longest length that more than `rank` rows reach
  int lo = __builtin_amdgcn_readfirstlane(least), hi = __builtin_amdgcn_readfirstlane(most) + 1;
  while (hi - lo > 1) {
    const int mid = lo + ((hi - lo) >> 1);
    if (reach(mid) > rank) lo = mid; else hi = mid;
  }
  int left = rank - reach(lo + 1), row = 0;  // rows of that length before the one wanted
#pragma unroll
  for (int q = 0; q < kRankChunks; ++q) {
    if (q * kWave >= rows) continue;
    const uint64_t same = __ballot(len[q] == lo);
    const int n = __popcll(same);
    if (left >= 0 && left < n) {
      const bool wanted = ((same >> lane) & 1) && __popcll(same & ((uint64_t(1) << lane) - 1)) == left;
      row = q * kWave + __ffsll((unsigned long long)__ballot(wanted)) - 1;
    }
    left -= n;
  }
  return first + row;
}

// 8 consecutive k of one feature per lane, from a feature-contiguous image: two transposing reads `next`
// bytes (four rows of k) apart
__device__ __forceinline__ u32x4 read_b(const char* at, int next) {
  const tr16x4 t0 = __builtin_amdgcn_ds_read_tr16_b64_v4f16((STIR_LDS tr16x4*)(at));
  const tr16x4 t1 = __builtin_amdgcn_ds_read_tr16_b64_v4f16((STIR_LDS tr16x4*)(at + next));
  const u32x2 lo = __builtin_bit_cast(u32x2, t0), hi = __builtin_bit_cast(u32x2, t1);
  return u32x4{lo[0], lo[1], hi[0], hi[1]};
}

// `bytes` from an address that is the same for all lanes; a lane that asks for what lies beyond gets zeros
__device__ __forceinline__ __amdgpu_buffer_rsrc_t window(const uint16_t* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(base), 0, bytes, 0x00020000);
}

// 32 rows of Y from row `row0`, features f0 .. f0 + 32 T, from a wavefront's accumulators: acc[t][v] is row (v%4) + 4h +
// 8(v/4), column n of the t-th 32x32 tile.  16-bit results go through 2048 T bytes of LDS of the wavefront's own into
// 16-byte stores (2-byte stores take eight times the instructions: 73 of 605 us at 16384 x 16384, 10 %, 4096
// features), fp32 results as they are, a line per 32 lanes.
template <bool BF16, int OUT, int T>
__device__ __forceinline__ void store_rows(char* __restrict__ own, const f32x16 (&acc)[T], void* __restrict__ Y,
                                           int64_t row0, int feat, int f0) {
  const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
  if constexpr (OUT == 1) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      if (f0 + 32 * t >= feat) continue;
      float* first = static_cast<float*>(Y) + (row0 + 4 * h) * feat + f0 + 32 * t + n;
#pragma unroll
      for (int v = 0; v < 16; ++v)
        __builtin_nontemporal_store(acc[t][v], first + (int64_t)((v & 3) + 8 * (v >> 2)) * feat);
    }
  } else {
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        *reinterpret_cast<uint16_t*>(own + (((v & 3) + 4 * h + 8 * (v >> 2)) * 32 * T + 32 * t + n) * 2) =
            to16<BF16>(acc[t][v]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    constexpr int UN = 4 * T;  // 16-byte units per row
#pragma unroll
    for (int q = 0; q < 2 * T; ++q) {
      const int at = kWave * q + lane, row = at / UN, u = at % UN;
      const u32x4 w = *reinterpret_cast<const u32x4*>(own + at * 16);
      if (f0 + 8 * u < feat)
        __builtin_nontemporal_store(Halves8(w), reinterpret_cast<Halves8*>(static_cast<uint16_t*>(Y) + (row0 + row) * feat + f0 +
                                                                8 * u));
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// One tile of the output: the 32*RS rows [bi0, bi0 + 32*RS) of stored block row i times the
// features [f0, f0 + 128*NT).  256 threads = 4 wavefronts; wavefront w owns features
// [32*NT*w, 32*NT*(w+1)) of the tile and RS*NT 32x32 accumulators.  RS = 2 (blocks of 64 rows and
// more): two adjacent 32-row slices of a block row, so every X fragment read from LDS feeds two
// MFMAs and the X tile is fetched once for 64 rows.
//
// Per step (one stored block, 32 of its k columns) the workgroup brings a 32 x 128*NT tile of X
// and the 32*RS x 32 piece of the block into LDS -- each thread loads 16-byte chunks, consecutive
// lanes consecutive chunks of a row of X -- while the previous step is multiplied (two LDS
// stages, one barrier per step).  LDS keeps X feature-contiguous, in 16-byte units of 8 features:
// unit (k, c) sits at (k/4)*4*FCN + (k%4)*FCN + (c ^ 4*(k%4)), FCN = units per row.  The MFMA B
// operand (8 consecutive k for one feature per lane) comes out of that image through the
// transposing read ds_read_b64_tr_b16, which hands lane i of a block of 16 lanes four consecutive
// k of column i when the lanes address rows k .. k+3, four features each.  The LDS serves such a
// read 32 lanes at a time from 64 banks: two blocks of 16 lanes, each reading two units in each of
// four rows whose stride is a multiple of all banks, so the XOR has to move the four rows of a
// block to four different groups of four units (c ^ 4*(k%4); with c ^ 2*(k%4) two rows of the two
// blocks met in the same banks and every read took twice its cycles).  The 16-byte stores of a row
// (8 lanes and 8 consecutive units per cycle) stay on distinct banks under either XOR.
// The block piece is fetched once per workgroup (8*RS bytes per thread) and laid out by k chunk so
// that a lane's A operand is one 16-byte read.
// lds: 2 * (64*128*NT + 2048*RS) bytes.
template <bool BF16, int OUT, int NT, int RS>  // OUT: 0 = same 16-bit type as the inputs, 1 = fp32
__device__ __forceinline__ void bsr_tile(char* __restrict__ lds, int blk, int feat, int i, int i_out, int bi0,
                                         int f0, const uint16_t* __restrict__ A,
                                         const uint16_t* __restrict__ X, void* __restrict__ Y,
                                         const int32_t* __restrict__ indptr,
                                         const int32_t* __restrict__ indices) {
  constexpr int TF = kTileF * NT;
  constexpr int FCN = TF / 8;            // 16-byte units per tile row
  constexpr int XB = kTileK * TF * 2;    // bytes of X per stage
  constexpr int SB = XB + 2048 * RS;     // bytes per stage
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;

  // staging role: 2*NT chunks of X per thread, of the eight rows from 8 * wave on; a chunk beyond feat reads as zero
  uint32_t xoff[2 * NT], xdst[2 * NT];
#pragma unroll
  for (int q = 0; q < 2 * NT; ++q) {
    const int idx = 64 * q + lane, c = idx % FCN, kw = idx / FCN, k = 8 * wave + kw;
    xoff[q] = f0 + 8 * c < feat ? (uint32_t)(kw * feat + 8 * c) * 2 : ~15u;  // bytes from the wavefront's first
    xdst[q] = (uint32_t)(((k >> 2) * 4 * FCN + (k & 3) * FCN + (c ^ (4 * (k & 3)))) * 16);
  }
  const uint16_t* Xw = X + (int64_t)(8 * wave) * feat + f0;
  // ... and 8*RS bytes of the block: RS = 1: half of the unit (chunk tid/64, row (tid/2)%32);
  // RS = 2: the unit (slice tid/128, chunk (tid/32)%4, row tid%32)
  uint32_t aoff;
  if constexpr (RS == 1)
    aoff = (uint32_t)(((tid >> 1) & 31) * blk + (tid >> 6) * 8 + (tid & 1) * 4) * 2;
  else
    aoff = (uint32_t)((32 * (tid >> 7) + (tid & 31)) * blk + ((tid >> 5) & 3) * 8) * 2;
  // operand reads, bytes inside a stage
  const int sl = lane & 15, half16 = (lane >> 4) & 1;
  uint32_t bread[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int kr = sl >> 2, c = (wave * NT + t) * 4 + 2 * half16 + ((sl & 3) >> 1);
    bread[t] = (uint32_t)(((2 * h) * 4 * FCN + kr * FCN + (c ^ (4 * kr))) * 16 + (sl & 1) * 8);
  }
  const uint32_t aread = XB + (h * 32 + n) * 16;

  f32x16 acc[RS][NT];
#pragma unroll
  for (int rs = 0; rs < RS; ++rs)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[rs][t][v] = 0.f;

  const int p_begin = indptr[i];
  const int nblk = indptr[i + 1] - p_begin;
  const int steps = nblk * (blk / kTileK);

  // The step to fetch next: block pb of the row, k offset k0; nothing beyond the last, so that no load depends on a
  // branch.  The block columns of the 64 blocks in hand and of the next 64 are in registers, one per lane: asked for
  // one by one, each block waited for a scalar load (430 x 120 blocks of 32, 1120 features, by this kernel 62.5 -> 59.3 us).
  // Two to four steps in registers at a time gain 3 to 10 % with two workgroups to a CU, sizes that other forms take, and
  // lose 3 to 15 % on larger ones.
  int pb = 0, k0 = 0;
  int j_lane = lane < nblk ? indices[p_begin + lane] : 0;
  int j_more = kWave + lane < nblk ? indices[p_begin + kWave + lane] : 0;
  u32x4 xr[2 * NT], ar;  // RS = 1 uses the first two words of ar
  auto fetch = [&]() {
    const bool live = pb < nblk;
    const int j = __builtin_amdgcn_readlane(j_lane, pb & (kWave - 1));
    const auto rx = window(Xw + ((int64_t)j * blk + k0) * feat, live ? 16u * feat : 0);
    const auto ra =
        window(A + (int64_t)(p_begin + pb) * blk * blk + (int64_t)bi0 * blk + k0, live ? 64u * RS * blk : 0);
#pragma unroll
    for (int q = 0; q < 2 * NT; ++q) xr[q] = __builtin_amdgcn_raw_buffer_load_b128(rx, xoff[q], 0, 0);
    if constexpr (RS == 1) {
      const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(ra, aoff, 0, 0);
      ar[0] = v[0], ar[1] = v[1];
    } else {
      ar = __builtin_amdgcn_raw_buffer_load_b128(ra, aoff, 0, 0);
    }
    k0 += kTileK;
    if (k0 == blk) {
      k0 = 0, ++pb;
      if ((pb & (kWave - 1)) == 0) {
        j_lane = j_more;
        j_more = pb + kWave + lane < nblk ? indices[p_begin + pb + kWave + lane] : 0;
      }
    }
  };
  fetch();
  for (int it = 0; it < steps; ++it) {
    char* stage = lds + (it & 1) * SB;
#pragma unroll
    for (int q = 0; q < 2 * NT; ++q) *reinterpret_cast<u32x4*>(stage + xdst[q]) = xr[q];
    if constexpr (RS == 1)
      *reinterpret_cast<u32x2*>(stage + XB + tid * 8) = u32x2{ar[0], ar[1]};
    else
      *reinterpret_cast<u32x4*>(stage + XB + tid * 16) = ar;
    fetch();
    __syncthreads();  // stage `it` is complete; the other stage's readers passed the previous barrier
    u32x4 a[RS][2];
#pragma unroll
    for (int rs = 0; rs < RS; ++rs)
#pragma unroll
      for (int m = 0; m < 2; ++m) a[rs][m] = *reinterpret_cast<const u32x4*>(stage + aread + rs * 2048 + m * 1024);
#pragma unroll
    for (int m = 0; m < 2; ++m) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const u32x4 b = read_b(stage + bread[t] + (4 * m) * FCN * 64, FCN * 64);
#pragma unroll
        for (int rs = 0; rs < RS; ++rs) acc[rs][t] = mfma32<BF16>(a[rs][m], b, acc[rs][t]);
      }
    }
  }
  if constexpr (OUT == 0) __syncthreads();  // the stages are free
#pragma unroll
  for (int rs = 0; rs < RS; ++rs)
    store_rows<BF16, OUT>(lds + wave * 2048 * NT, acc[rs], Y, (int64_t)i_out * blk + bi0 + 32 * rs, feat,
                          f0 + wave * NT * 32);
}

// The other order, for tall blocks (by_rows): XCD x owns the block rows i = x, x + 8, ... and
// walks, for each, the slices of the block row inside every feature tile before the next feature
// tile.  The workgroups that are resident together on an XCD then share the blocks of A of their
// block row (fetched into that L2 once instead of once per feature tile) and, between the slices
// of a block row, its tiles of X.
__device__ __forceinline__ bool decode_tile_by_rows(int64_t L, int64_t block_rows, int sub, int f_tiles,
                                                    int64_t& slice, int& f_tile) {
  const int xcd = (int)(L & 7);
  const int64_t t = L >> 3;
  const int64_t i = xcd + 8 * (t / ((int64_t)sub * f_tiles));
  f_tile = (int)((t / sub) % f_tiles);
  slice = i * sub + t % sub;
  return i < block_rows;
}

// One workgroup per tile, 1-D grid (see decode_tile).
template <bool BF16, int OUT, int NT, int RS>
__global__ __launch_bounds__(256) void bsr_spmm_kernel(int blk, int feat, int64_t slices, int f_tiles, int by_rows,
                                                       int ranked,
                                                       const uint16_t* __restrict__ A,
                                                       const uint16_t* __restrict__ X, void* __restrict__ Y,
                                                       const int32_t* __restrict__ indptr,
                                                       const int32_t* __restrict__ indices,
                                                       const int32_t* __restrict__ row_ids) {
  constexpr int TF = kTileF * NT;
  __shared__ __attribute__((aligned(16))) char xs[2 * (kTileK * TF * 2 + 2048 * RS)];
  int64_t slice;
  int f_tile;
  const int sub = blk / (32 * RS);  // slices of 32*RS rows per block row
  if (RS == 1) by_rows = ranked = 0;  // blocks of 64 rows and more only: see bsr_form
  if (by_rows) {
    if (!decode_tile_by_rows(blockIdx.x, slices / sub, sub, f_tiles, slice, f_tile)) return;
  } else if (ranked ? !decode_ranked(blockIdx.x, slices, sub, f_tiles, slice, f_tile)
                    : !decode_tile(blockIdx.x, slices, f_tiles, slice, f_tile)) {
    return;
  }
  // the same for all lanes, which the divisions hide from the compiler
  slice = __builtin_amdgcn_readfirstlane((int)slice), f_tile = __builtin_amdgcn_readfirstlane(f_tile);
  int i = (int)slice / sub;
  const int bi0 = ((int)slice % sub) * (32 * RS);
  if (ranked) i = __builtin_amdgcn_readfirstlane(row_of_rank(indptr, (int)(slices / sub), i));
  // doubly-compressed form: stored block row i is block row row_ids[i] of the output
  const int i_out = row_ids ? row_ids[i] : i;
  bsr_tile<BF16, OUT, NT, RS>(xs, blk, feat, i, i_out, bi0, f_tile * TF, A, X, Y, indptr, indices);
}

// ------------------------------------------------------------------ blocks of 16 k+16 rows
// Block sides that are a multiple of 16 but not of 32 (the reference's schedule splits both block
// axes by 16, examples/blocksparse/bsr_spmm.py:379-380): 16-row slices on v_mfma_f32_16x16x32,
// whose k extent of 32 is two 16-column chunks of the block row's blocks in storage order.
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <bool BF16>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                  0, 0);
}

// ------------------------------------------------------------------ 32-row slices, X in registers
// Lane (c, g) of a wavefront loads 8 features from each of 8 consecutive rows of X, 16 bytes a row, and makes eight MFMA
// operands of them (lane_operand.h): the loads are whole 256- or 512-byte pieces of a row, and eight neighbouring features of a
// row of Y are one 16-byte store.
using stir::operand_of;

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// Results of a wavefront whose lane (n, h), n of LANES, has eight neighbouring features, 8 n ..., of row 4 h of Y behind `row`: as
// they are, 16 bytes a lane, if they have 16 bits.  Floats first go through 2 KB of LDS into row order, four features to a lane
// and the rows one behind the other, so that a store is of whole lines: with halves of lines (an exchange within quads) 437 x 33
// blocks of 32, 1 step, 2720 features took 48.7 us, now 33.4, 452 x 51, 3 steps, 3840 66.5, 49.6.
// The place of piece e (features 4 e ...) of a lane is XORed by 8 e: eight lanes in row order share no bank.
template <int LANES>
__device__ __forceinline__ int piece_place(int h, int n, int e) { return (2 * h + e) * LANES + (n ^ (8 * e)); }

template <bool BF16, int OUT, int LANES>
__device__ __forceinline__ void store_rows8(void* __restrict__ Y, int64_t row, int feat, int f0, int lane, const float (&v)[8],
                                            f32x4* stage) {
  const int n = lane % LANES, h = lane / LANES;
  if constexpr (OUT == 1) {
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int e = 0; e < 2; ++e)
      stage[piece_place<LANES>(h, n, e)] = f32x4{v[4 * e], v[4 * e + 1], v[4 * e + 2], v[4 * e + 3]};
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int at = kWave * i + lane, r = at / (2 * LANES), u = at % (2 * LANES);
      const f32x4 d = stage[piece_place<LANES>(r, u >> 1, u & 1)];
      if (f0 + 4 * u < feat)
        __builtin_nontemporal_store(f32x4u{d[0], d[1], d[2], d[3]},
                                    reinterpret_cast<f32x4u*>(static_cast<float*>(Y) + (row + 4 * r) * feat + f0 + 4 * u));
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  } else {
    u32x4 w;
#pragma unroll
    for (int t = 0; t < 4; ++t) w[t] = to16<BF16>(v[2 * t]) | (uint32_t)to16<BF16>(v[2 * t + 1]) << 16;
    if (f0 + 8 * n < feat)
      __builtin_nontemporal_store(Halves8(w), reinterpret_cast<Halves8*>(static_cast<uint16_t*>(Y) + (row + 4 * h) * feat + f0 + 8 * n));
  }
}

// The same for what several wavefronts left in LDS, `used` of them: lane (c, g), c of 16, of wavefront w has its pieces e at
// part[w * stride + 64 e + (lane ^ 8 e)].
template <bool BF16, int OUT, int W>
__device__ __forceinline__ void add_up8(const f32x4* part, int stride, int used, void* __restrict__ Y, int64_t row, int feat, int f0,
                                        int lane) {
  f32x4 o[2];
  int place[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int at = kWave * i + lane, e = OUT == 1 ? at & 1 : i;
    place[i] = 64 * e + ((OUT == 1 ? at >> 1 : lane) ^ (8 * e));
    o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int w = 0; w < W; ++w) {
    if (w >= used) continue;
#pragma unroll
    for (int i = 0; i < 2; ++i) o[i] += part[w * stride + place[i]];
  }
  if constexpr (OUT == 1) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = 2 * i + (lane >> 5), u = lane & 31;
      if (f0 + 4 * u < feat)
        __builtin_nontemporal_store(f32x4u{o[i][0], o[i][1], o[i][2], o[i][3]},
                                    reinterpret_cast<f32x4u*>(static_cast<float*>(Y) + (row + 4 * r) * feat + f0 + 4 * u));
    }
  } else {
    const float v[8] = {o[0][0], o[0][1], o[0][2], o[0][3], o[1][0], o[1][1], o[1][2], o[1][3]};
    store_rows8<BF16, OUT, 16>(Y, row, feat, f0, lane, v, nullptr);
  }
}

// A tile of 32 rows x 128 features, 16 accumulators of v_mfma_f32_16x16x32, a step of 32 k in eight loads of X and two of A.
// W wavefronts take the steps of a block row in turn and meet in LDS at the end (W = 1: none does).
// D steps are on their way; nothing is asked for beyond the last one: a load outside its window costs as much as another
// (128 x 128 blocks of 32, 512 features, four wavefronts 9.8 -> 9.1 us).
// Against four wavefronts that shared 128 features through LDS and met at a barrier per step, us as part of a graph:
// 128 x 128 blocks of 32, 10 %, 512 features 11.1 -> 9.1 (W = 4); 256 x 256, 512 features 24.0 -> 20.1 (W = 1; 2 now); 209 x 46, 2
// steps a row, 1216 features 9.3 -> 7.8 (W = 1); against eight wavefronts with 64
// features through LDS: 197 x 193, 37 steps, 224 features 23.0 -> 16.3 (W = 4), 131 x 322, 78 steps, 128 features 18.7 ->
// 14.9 (W = 8).  Small launches are bound by the trips to memory one after the other -- indptr, block columns, rows of X,
// 2.8 us with the launch -- and then by X and A coming through the L2s, which hold neither (config above: 22 MB, 2.7 us).
template <bool BF16, int OUT, int W, int D = 2>
__global__ __launch_bounds__(W * kWave, D == 1 ? 4 : W == 1 ? 3 : 2) void bsr_direct_kernel(
    int blk, int feat, int64_t slices, int f_tiles, const uint16_t* __restrict__ A, const uint16_t* __restrict__ X,
    void* __restrict__ Y, const int32_t* __restrict__ indptr, const int32_t* __restrict__ indices,
    const int32_t* __restrict__ row_ids) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  int64_t slice;
  int f_tile;
  if (!decode_tile(blockIdx.x, slices, f_tiles, slice, f_tile)) return;
  // the same for all lanes, which the divisions hide from the compiler
  slice = __builtin_amdgcn_readfirstlane((int)slice), f_tile = __builtin_amdgcn_readfirstlane(f_tile);
  const int sub = blk / 32;  // slices per block row = steps per block
  const int i = (int)slice / sub, bi0 = (int)slice % sub * 32;
  const int i_out = row_ids ? row_ids[i] : i;
  const int f0 = f_tile * kTileF;
  // rows 8 g ... 8 g + 7 of a step's 32; features beyond feat repeat the last ones: nobody stores them
  const uint32_t xoff = (uint32_t)(8 * g * feat + min(8 * c, feat - f0 - 8)) * 2;
  const uint32_t aoff = (uint32_t)((bi0 + c) * blk + 8 * g) * 2;

  f32x4 acc[2][8];
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int t = 0; t < 8; ++t) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int p_begin = indptr[i], nblk = indptr[i + 1] - p_begin;
  const int steps = nblk * sub, first = W == 1 ? 0 : wave;
  if (first < steps) {
    const int32_t* cols = indices + p_begin;
    int left = (steps - first + W - 1) / W;
    int block = first / sub, col = first % sub;  // of the step to fetch next
    u32x4 x[D][8], a[D][2];
    auto fetch = [&](int s) {
      const int j = cols[min(block, nblk - 1)];
      const auto ra = window(A + (int64_t)(p_begin + block) * blk * blk + 32 * col, (uint32_t)(blk * blk - 32 * col) * 2);
#pragma unroll
      for (int r = 0; r < 2; ++r) a[s][r] = __builtin_amdgcn_raw_buffer_load_b128(ra, aoff + 32 * r * blk, 0, 0);
      const auto rx = window(X + ((int64_t)j * blk + 32 * col) * feat + f0, 64u * feat);
#pragma unroll
      for (int q = 0; q < 8; ++q) x[s][q] = __builtin_amdgcn_raw_buffer_load_b128(rx, xoff, q * 2 * feat, 0);
      block += W / sub, col += W % sub;
      if (col >= sub) col -= sub, ++block;
    };
    auto multiply = [&](int s) {
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const u32x4 b = operand_of(x[s], t / 2, t % 2);
#pragma unroll
        for (int r = 0; r < 2; ++r) acc[r][t] = mfma16<BF16>(a[s][r], b, acc[r][t]);
      }
    };
    if constexpr (D == 1) {
      fetch(0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
      for (; left > 1; --left) {
        multiply(0);
        __builtin_amdgcn_sched_barrier(0);
        fetch(0);
        __builtin_amdgcn_sched_barrier(0);
      }
      multiply(0);
    } else {
      fetch(0);
      if (left > 1) fetch(1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
      for (; left >= 2 * D; left -= D) {
#pragma unroll
        for (int s = 0; s < D; ++s) {
          multiply(s);
          __builtin_amdgcn_sched_barrier(0);
          fetch(s);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      multiply(0);  // one to three are left
      if (left > 2) fetch(0);
      if (left > 1) multiply(1);
      if (left > 2) multiply(0);
    }
  }

  // acc[r][t][v] is row 16 r + 4 g + v, feature 8 c + t
  const int64_t row0 = (int64_t)i_out * blk + bi0;
  if constexpr (W == 1) {
    __shared__ f32x4 stage[OUT == 1 ? 2 * kWave : 1];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float o[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) o[t] = acc[r][t][v];
        store_rows8<BF16, OUT, 16>(Y, row0 + 16 * r + v, feat, f0, lane, o, stage);
      }
  } else {
    // each wavefront adds 8 / W of the eight rows a lane has
    __shared__ __attribute__((aligned(16))) f32x4 part[W][8][2][kWave];
    const int used = min(steps, W);
    if (wave < used) {
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int e = 0; e < 2; ++e)
            part[wave][4 * r + v][e][lane ^ (8 * e)] =
                f32x4{acc[r][4 * e][v], acc[r][4 * e + 1][v], acc[r][4 * e + 2][v], acc[r][4 * e + 3][v]};
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 8 / W; ++q) {
      const int at = wave * (8 / W) + q;
      add_up8<BF16, OUT, W>(part[0][at][0], 8 * 2 * kWave, used, Y, row0 + 16 * (at >> 2) + (at & 3), feat, f0, lane);
    }
  }
}

// ---- 16-row slices
// A step is two chunks of 16 columns, and of the k slots 8 g ... of lane group g four are rows of the first and four of the
// second, in A and X alike: so a load of X is of one chunk, whose place is the same for all lanes.  The groups have the rows 0, 8,
// 4, 12 ... of a chunk: A comes 16 bytes a lane, columns 8 (g & 1) ... of chunk g / 2, and two swaps of half wavefronts put it
// so.  All offsets are in lanes' registers: an empty window's loads with scalar ones are not relied on to be zeros.
__device__ __forceinline__ u32x4 two_chunks(u32x4 a) {
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    const u32x2 t = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(a[w], a[w + 2], false, false));
    a[w] = t[0], a[w + 2] = t[1];
  }
  return a;
}
__device__ __forceinline__ int first_row(int g) { return 8 * (g & 1) + 4 * (g >> 1); }

// The sums of `used` of the W wavefronts at a tile, which have 4 / W (eight: the first four one) of a lane's four rows each; part:
// those of this tile.
template <bool BF16, int OUT, int W>
__device__ __forceinline__ void add_up(const f32x4 (&acc)[8], f32x4 (&part)[W][4][2][kWave], int wave, int lane, int used,
                                       void* __restrict__ Y, int64_t row0, int feat, int f0) {
  if (wave < used) {
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int e = 0; e < 2; ++e)
        part[wave][v][e][lane ^ (8 * e)] = f32x4{acc[4 * e][v], acc[4 * e + 1][v], acc[4 * e + 2][v], acc[4 * e + 3][v]};
  }
  __syncthreads();
  for (int v = wave; v < 4; v += W) add_up8<BF16, OUT, W>(part[0][v][0], 4 * 2 * kWave, used, Y, row0 + v, feat, f0, lane);
}

// A tile of 16 rows x 128 features, eight accumulators of v_mfma_f32_16x16x32; W wavefronts take the steps in turn.  T such tiles
// side by side to a workgroup, whose wavefronts find each other's A in L1.  D steps of a wavefront are on their way.
// Against X through LDS (wavefronts with 128 or 256 features, or four that met at a barrier per step), us: 398 x 310 blocks of
// 16, 19 steps, 576 features 34 -> 20.5 (W = 4); 749 x 92, 8 steps, 160 features 15.4 -> 9.1 (T = 2); 342 x 83, 4 steps, 1728
// features 18.5 -> 14.8 (W = 1); 154 tiles of 80 steps 16.8 -> 13.0 (W = 8).  LDS, which X passed twice, had been as busy as the
// L1s.  Bound by the L1s and the trips to memory at small sizes, by X from beyond L2 at large ones.  A by two loads of 8 bytes a
// lane, without the swaps: 3 % slower, blocks of 48 and 80 5 to 8 %.
template <bool BF16, int OUT, int W, int T, bool ONE, int D = 2>
__global__ __launch_bounds__(W * T * kWave, D == 1 ? 5 : W == 1 ? 4 : 2) void bsr16_direct_kernel(
    int blk, int feat, int64_t slices, int f_tiles, int ranked, const uint16_t* __restrict__ A,
    const uint16_t* __restrict__ X, void* __restrict__ Y, const int32_t* __restrict__ indptr,
    const int32_t* __restrict__ indices, const int32_t* __restrict__ row_ids) {
  if (ONE) blk = 16;
  const int sub = blk / 16;  // 16-row slices per block row = 16-column chunks per block
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6) % W;
  const int c = lane & 15, g = lane >> 4;
  int64_t slice;
  int f_tile;
  if (W * T == 1 && ranked ? !decode_ranked(blockIdx.x, slices, sub, f_tiles, slice, f_tile)
                           : !decode_tile(blockIdx.x, slices, f_tiles, slice, f_tile))
    return;
  // the same for all lanes, which the divisions hide from the compiler
  slice = __builtin_amdgcn_readfirstlane((int)slice), f_tile = __builtin_amdgcn_readfirstlane(f_tile);
  int i = (int)slice / sub;
  const int bi0 = (int)slice % sub * 16;
  if (W * T == 1 && ranked) i = __builtin_amdgcn_readfirstlane(row_of_rank(indptr, (int)(slices / sub), i));
  const int i_out = row_ids ? row_ids[i] : i;
  const int f0 = (f_tile * T + __builtin_amdgcn_readfirstlane(tid >> 6) / W) * kTileF;  // feat and beyond: a tile without work
  // features beyond feat repeat the last ones: nobody stores them
  uint32_t xoff[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) xoff[q] = (uint32_t)((first_row(g) + q) * feat + min(8 * c, feat - f0 - 8)) * 2;
  const uint32_t aoff = (uint32_t)((bi0 + c) * blk + 8 * (g & 1)) * 2;

  f32x4 acc[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int p_begin = indptr[i], nblk = indptr[i + 1] - p_begin;
  const int chunks = nblk * sub, steps = T > 1 && f0 >= feat ? 0 : (chunks + 1) / 2, first = W == 1 ? 0 : wave;
  if (first < steps) {
    const int32_t* cols = indices + p_begin;
    int left = (steps - first + W - 1) / W;
    int block = 2 * first / sub, col = 2 * first % sub;  // of the step to fetch next
    u32x4 x[D][8], a[D];
    auto fetch = [&](int s) {
      const auto ra = window(A + (int64_t)(p_begin + block) * blk * blk, (uint32_t)(min(nblk - block, 2) * blk * blk) * 2);
      const int over = ONE || col + 1 == sub;  // the second chunk is the first of the next block
      const int apart = over ? blk * blk - 16 * col : 16;
      a[s] = __builtin_amdgcn_raw_buffer_load_b128(ra, aoff + (16 * col + (g >> 1) * apart) * 2, 0, 0);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int at = block + (b && over), k0 = ONE || (b && over) ? 0 : 16 * (col + b);
        const bool live = at < nblk;
        const int j = cols[min(at, nblk - 1)];
        const auto rx = window(X + ((int64_t)j * blk + k0) * feat + f0, live ? 32u * feat : 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) x[s][4 * b + q] = __builtin_amdgcn_raw_buffer_load_b128(rx, xoff[q], 0, 0);
      }
      block += 2 * W / sub, col += 2 * W % sub;
      if (col >= sub) col -= sub, ++block;
    };
    auto multiply = [&](int s) {
      const u32x4 rows = two_chunks(a[s]);
#pragma unroll
      for (int t = 0; t < 8; ++t) acc[t] = mfma16<BF16>(rows, operand_of(x[s], t / 2, t % 2), acc[t]);
    };
    if constexpr (D == 1) {
      fetch(0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
      for (; left > 1; --left) {
        multiply(0);
        __builtin_amdgcn_sched_barrier(0);
        fetch(0);
        __builtin_amdgcn_sched_barrier(0);
      }
      multiply(0);
    } else {
      fetch(0);
      if (left > 1) fetch(1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
      for (; left >= 2 * D; left -= D) {
#pragma unroll
        for (int s = 0; s < D; ++s) {
          multiply(s);
          __builtin_amdgcn_sched_barrier(0);
          fetch(s);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      multiply(0);  // one to three are left
      if (left > 2) fetch(0);
      if (left > 1) multiply(1);
      if (left > 2) multiply(0);
    }
  }

  // acc[t][v] is row 4 g + v, feature 8 c + t
  const int64_t row0 = (int64_t)i_out * blk + bi0;
  if constexpr (W == 1) {
    static_assert(T == 1, "one wavefront to a workgroup");
    __shared__ f32x4 stage[OUT == 1 ? 2 * kWave : 1];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float o[8];
#pragma unroll
      for (int t = 0; t < 8; ++t) o[t] = acc[t][v];
      store_rows8<BF16, OUT, 16>(Y, row0 + v, feat, f0, lane, o, stage);
    }
  } else {
    __shared__ __attribute__((aligned(16))) f32x4 part[T][W][4][2][kWave];
    add_up<BF16, OUT, W>(acc, part[(tid >> 6) / W], wave, lane, min(steps, W), Y, row0, feat, f0);
  }
}

// A tile of 16 rows x 256 features, sixteen accumulators, in two halves of 128 features: as soon as the last operand of a half is
// made, the next step's half is asked for.  By a wavefront (blocks of 16), or by four that take the steps in turn (the others).
// The columns come by scalar loads, a step ahead: a vector load of them on a branch in the loop made every wait in it one for
// all loads (11 % slower).
// 1024 x 300 blocks of 16, 12 steps, 1024 features 52 us with X through LDS, 43.7; 1024 x 1024, 51 steps 174 -> 161 ranked, where
// X comes from beyond the L2s either way 16384 x 16384, 10 %, 4096 features 611 to 632 -> 606 to 619, 30 % more of it missing L2.
template <bool BF16, int OUT, bool ONE>
__global__ __launch_bounds__((ONE ? 1 : 4) * kWave, 3) void bsr16_wave_kernel(
    int blk, int feat, int64_t slices, int f_tiles, int ranked, const uint16_t* __restrict__ A,
    const uint16_t* __restrict__ X, void* __restrict__ Y, const int32_t* __restrict__ indptr,
    const int32_t* __restrict__ indices, const int32_t* __restrict__ row_ids) {
  constexpr int W = ONE ? 1 : 4;
  if (ONE) blk = 16;
  const int sub = blk / 16;
  int64_t slice;
  int f_tile;
  if (ranked ? !decode_ranked(blockIdx.x, slices, sub, f_tiles, slice, f_tile)
             : !decode_tile(blockIdx.x, slices, f_tiles, slice, f_tile))
    return;
  const int lane = threadIdx.x & 63, wave = W == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  // the same for all lanes, which the divisions hide from the compiler
  slice = __builtin_amdgcn_readfirstlane((int)slice), f_tile = __builtin_amdgcn_readfirstlane(f_tile);
  int i = (int)slice / sub;
  const int bi0 = (int)slice % sub * 16;
  if (ranked) i = __builtin_amdgcn_readfirstlane(row_of_rank(indptr, (int)(slices / sub), i));
  const int i_out = row_ids ? row_ids[i] : i;
  const int f0 = f_tile * kWaveF;
  uint32_t xoff[2][4];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int q = 0; q < 4; ++q) xoff[m][q] = (uint32_t)((first_row(g) + q) * feat + min(128 * m + 8 * c, feat - f0 - 8)) * 2;
  const uint32_t aoff = (uint32_t)((bi0 + c) * blk + 8 * (g & 1)) * 2;

  f32x4 acc[2][8];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int t = 0; t < 8; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int p_begin = indptr[i], nblk = indptr[i + 1] - p_begin;
  const int steps = (nblk * sub + 1) / 2, mine = W == 1 ? steps : (steps - wave + W - 1) / W;
  const int32_t* cols = indices + p_begin;
  int block = 2 * wave / sub, col = 2 * wave % sub;  // of the step after the one that is being fetched
  int at[2], j[2], k0[2], at_n[2], j_n[2], k0_n[2];  // the chunks of either
  auto look = [&]() {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const bool over = ONE ? b != 0 : col + b == sub;
      at_n[b] = block + over, k0_n[b] = ONE || over ? 0 : 16 * (col + b);
      j_n[b] = cols[min(at_n[b], nblk - 1)];
    }
    block += 2 * W / sub, col += 2 * W % sub;
    if (col >= sub) col -= sub, ++block;
  };
  auto next = [&]() {
#pragma unroll
    for (int b = 0; b < 2; ++b) at[b] = at_n[b], j[b] = j_n[b], k0[b] = k0_n[b];
    look();
  };
  u32x4 x[2][8];
  u32x4 ar;
  auto fetch_a = [&]() {
    const uint32_t block_bytes = 2u * blk * blk, bytes = at[0] < nblk ? (at[0] + 1 < nblk ? 2 * block_bytes : block_bytes) : 0;
    const auto ra = window(A + (int64_t)(p_begin + at[0]) * blk * blk, bytes);
    ar = __builtin_amdgcn_raw_buffer_load_b128(ra, aoff + (k0[0] + (g >> 1) * ((at[1] - at[0]) * blk * blk + k0[1] - k0[0])) * 2, 0, 0);
  };
  auto fetch_x = [&](int m) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const auto rx = window(X + ((int64_t)j[b] * blk + k0[b]) * feat + f0, at[b] < nblk ? 32u * feat : 0);
#pragma unroll
      for (int q = 0; q < 4; ++q) x[m][4 * b + q] = __builtin_amdgcn_raw_buffer_load_b128(rx, xoff[m][q], 0, 0);
    }
  };
  if (mine > 0) {
    look(), next(), fetch_a(), fetch_x(0), fetch_x(1);
#pragma unroll 1
    for (int it = 0; it < mine; ++it) {
      const u32x4 a = two_chunks(ar);
      next(), fetch_a();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        u32x4 b[2][2];
        auto pick = [&](int w) { b[w % 2][0] = operand_of(x[m], w, 0), b[w % 2][1] = operand_of(x[m], w, 1); };
        pick(0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          if (w < 3) pick(w + 1); else fetch_x(m);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int e = 0; e < 2; ++e) acc[m][2 * w + e] = mfma16<BF16>(a, b[w % 2][e], acc[m][2 * w + e]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }
  const int64_t row0 = (int64_t)i_out * blk + bi0;
  if constexpr (W == 1) {
    __shared__ f32x4 stage[OUT == 1 ? 2 * kWave : 1];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float o[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) o[t] = acc[m][t][v];
        store_rows8<BF16, OUT, 16>(Y, row0 + v, feat, f0 + 128 * m, lane, o, stage);
      }
  } else {
    __shared__ __attribute__((aligned(16))) f32x4 part[W][4][2][kWave];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      if (m) __syncthreads();
      add_up<BF16, OUT, W>(acc[m], part, wave, lane, min(steps, W), Y, row0, feat, f0 + 128 * m);
    }
  }
}

// ---- 32-row slices by a wavefront
// A wavefront owns 32 rows x 256 features, eight accumulators of v_mfma_f32_32x32x16: a step of 32 k is two halves of eight
// loads of X; as soon as the last operand of a half is made, the next step's half is asked for, so that 8 wavefronts per CU
// have 128 KB on their way.  A comes in 16-byte pieces in memory order, a step ahead, and through 2 KB of LDS of the
// wavefront's own into operand order: asked for in operand order, a load touches 32 half lines and costs twice as much.
// With the ranked order (row_of_rank) the wavefronts of an XCD stay within reach of each other in X: 16384 x 16384,
// 10 % blocks of 32, 4096 features, fp16: 565 us in plain order, 378 ranked; 416 with X through LDS, 393 with A in operand
// order.  Bound by the L2s: 7.7 GB through the L1s (233 us at the 33 TB/s that 16 bytes a lane reach) and 1.75 GB of misses,
// of which 0.86 are A, read once per feature tile: the products alone take 155 us, the loads alone 366, X without A 267, X
// out of L2 beside A 286.  Not bound by latency: four wavefronts per CU with two or three steps each on their way 410 us.
// Two feature tiles side by side on an XCD share A but not the window of X (520 us); A past the L2 is slower (465).
template <bool BF16, int OUT>
__global__ __launch_bounds__(kWave, 2) void bsr_wave_kernel(int blk, int feat, int64_t slices, int f_tiles, int ranked,
                                                            const uint16_t* __restrict__ A,
                                                            const uint16_t* __restrict__ X, void* __restrict__ Y,
                                                            const int32_t* __restrict__ indptr,
                                                            const int32_t* __restrict__ indices,
                                                            const int32_t* __restrict__ row_ids) {
  constexpr int FT = kWaveF / 32;  // accumulators
  __shared__ __attribute__((aligned(16))) u32x4 piece[2 * kWave];
  const int sub = blk / 32;
  int64_t slice;
  int f_tile;
  if (ranked ? !decode_ranked(blockIdx.x, slices, sub, f_tiles, slice, f_tile)
             : !decode_tile(blockIdx.x, slices, f_tiles, slice, f_tile))
    return;
  const int lane = threadIdx.x, n = lane & 31, h = lane >> 5;
  // the same for all lanes, which the divisions hide from the compiler
  slice = __builtin_amdgcn_readfirstlane((int)slice), f_tile = __builtin_amdgcn_readfirstlane(f_tile);
  int i = (int)slice / sub;
  const int bi0 = ((int)slice % sub) * 32;
  if (ranked) i = __builtin_amdgcn_readfirstlane(row_of_rank(indptr, (int)(slices / sub), i));
  const int i_out = row_ids ? row_ids[i] : i;
  const int f0 = f_tile * kWaveF;
  // rows 16 m + 8 h ... + 7 of a step's 32; features beyond feat repeat the last ones: nobody stores them
  const uint32_t xoff = (uint32_t)(8 * h * feat + min(8 * n, feat - f0 - 8)) * 2;
  const uint32_t aoff = (uint32_t)((bi0 + lane / 4) * blk + 8 * (lane % 4)) * 2;

  f32x16 acc[FT];
#pragma unroll
  for (int t = 0; t < FT; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[t][v] = 0.f;

  const int p_begin = indptr[i], nblk = indptr[i + 1] - p_begin;
  const int steps = nblk * sub;
  if (steps > 0) {
    // the step to fetch next: block `block`, k offset k0; nothing beyond the last, so that no load depends on a branch
    const int32_t* cols = indices + p_begin;
    int block = 0, k0 = 0, j = cols[0], j_next = cols[min(1, nblk - 1)];
    u32x4 x[2][8], ar[2], a[2];
    auto fetch_a = [&]() {
      // the window begins inside A also when it is empty: nothing rests on what a scalar offset does to an empty one
      const auto ra = window(A + (int64_t)(p_begin + min(block, nblk - 1)) * blk * blk + k0,
                             block < nblk ? (uint32_t)(blk * blk - k0) * 2 : 0);
#pragma unroll
      for (int m = 0; m < 2; ++m) ar[m] = __builtin_amdgcn_raw_buffer_load_b128(ra, aoff, m * 32 * blk, 0);
    };
    auto fetch_x = [&](int m) {
      const auto rx = window(X + ((int64_t)j * blk + k0) * feat + f0, block < nblk ? 64u * feat : 0);
#pragma unroll
      for (int q = 0; q < 8; ++q) x[m][q] = __builtin_amdgcn_raw_buffer_load_b128(rx, xoff, (16 * m + q) * 2 * feat, 0);
    };
    auto advance = [&]() {
      k0 += 32;
      const bool over = k0 == blk;
      k0 = over ? 0 : k0, block += over, j = over ? j_next : j;
      j_next = cols[min(block + 1, nblk - 1)];
    };
    fetch_a(), fetch_x(0), fetch_x(1), advance();
#pragma unroll 1
    for (int it = 0; it < steps; ++it) {
      // piece 64 m + l is row 16 m + l / 4, k 8 (l % 4) ...
#pragma unroll
      for (int m = 0; m < 2; ++m) piece[(lane % 4) * 32 + 16 * m + lane / 4] = ar[m];
      fetch_a();
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int m = 0; m < 2; ++m) a[m] = piece[(2 * m + h) * 32 + n];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        u32x4 b[2][2];
        auto pick = [&](int w) { b[w % 2][0] = operand_of(x[m], w, 0), b[w % 2][1] = operand_of(x[m], w, 1); };
        pick(0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          if (w < 3) pick(w + 1); else fetch_x(m);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int e = 0; e < 2; ++e) acc[2 * w + e] = mfma32<BF16>(a[m], b[w % 2][e], acc[2 * w + e]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      advance();
    }
  }
  // acc[t][v] is row (v % 4) + 4 h + 8 (v / 4), feature 8 n + t
  const int64_t row0 = (int64_t)i_out * blk + bi0;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    float o[8];
#pragma unroll
    for (int t = 0; t < FT; ++t) o[t] = acc[t][v];
    store_rows8<BF16, OUT, 32>(Y, row0 + (v & 3) + 8 * (v >> 2), feat, f0, lane, o, reinterpret_cast<f32x4*>(piece));
  }
}

// ------------------------------------------------------------------ small launches
// With a few workgroups per CU the run time is the chain of steps of the longest block row, each a memory
// round trip.  Here the eight wavefronts of a workgroup take the steps of a block row (ROWS = 32 or 16 of its
// rows, 64 features) in turn: wavefront w the steps w, w + 8, ..., each with an X tile of its own in LDS (no
// workgroup barrier in the loop: the LDS operations of one wavefront execute in order); the eight partial
// results are added through LDS at the end.
// The X tile is 32 rows of 8 units of 16 bytes; unit (k, c) sits at place c ^ 4 * (k / 2 % 2) of its row -- two
// rows fill the 64 banks -- and, ROWS = 16, ^ 2 * (k / 8 % 2): the two blocks of 16 lanes that
// a transposing read serves together ask for the same units of k groups eight rows apart there.
// Against four wavefronts that took the k halves of each step: 40 x 510 blocks of 32, 18 %, 288 features
// 27.4 -> 15.9 us; 358 x 998 blocks of 16, 64 features (which had no such form) 39 -> 11.8 us.
constexpr int kSplitWaves = 8;
constexpr int kSplitF = 64;

template <bool BF16, int OUT, int ROWS>
__global__ __launch_bounds__(64 * kSplitWaves) void bsr_split_kernel(int blk, int feat, int64_t slices, int f_tiles,
                                                                     const uint16_t* __restrict__ A,
                                                                     const uint16_t* __restrict__ X,
                                                                     void* __restrict__ Y,
                                                                     const int32_t* __restrict__ indptr,
                                                                     const int32_t* __restrict__ indices,
                                                                     const int32_t* __restrict__ row_ids) {
  constexpr int FCN = kSplitF / 8;
  constexpr int XB = kTileK * kSplitF * 2;          // bytes of a wavefront's X tile
  constexpr int TILES = ROWS == 32 ? 2 : 4;         // 32- or 16-feature tiles
  constexpr int REGS = ROWS == 32 ? 16 : 4;         // accumulator registers of one
  constexpr int ELEMS = TILES * REGS * kWave;       // floats of a partial result
  __shared__ __attribute__((aligned(16))) char lds[kSplitWaves * (XB > ELEMS * 4 ? XB : ELEMS * 4)];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int64_t slice;
  int f_tile;
  if (!decode_tile(blockIdx.x, slices, f_tiles, slice, f_tile)) return;
  const int sub = blk / ROWS;
  const int i = (int)(slice / sub), bi0 = (int)(slice % sub) * ROWS;
  const int i_out = row_ids ? row_ids[i] : i;
  const int f0 = f_tile * kSplitF;
  char* stage = lds + wave * XB;
  // staging role: unit xc of the rows k = 8 u + kq
  const int xc = lane & 7, kq = lane >> 3;
  const bool xlive = f0 + 8 * xc < feat;
  const uint32_t xoff = (uint32_t)(kq * feat + 8 * xc);
  uint32_t xdst[4];
#pragma unroll
  for (int u = 0; u < 4; ++u)
    xdst[u] = (uint32_t)(((8 * u + kq) * FCN + (xc ^ (4 * ((kq >> 1) & 1)) ^ (ROWS == 16 ? 2 * (u & 1) : 0))) * 16);
  // operand role
  const int n = ROWS == 32 ? lane & 31 : lane & 15, h = ROWS == 32 ? lane >> 5 : lane >> 4;
  const int sl = lane & 15, kr = sl >> 2;
  uint32_t bread[TILES];
#pragma unroll
  for (int t = 0; t < TILES; ++t) {
    const int c = ROWS == 32 ? 4 * t + 2 * ((lane >> 4) & 1) + ((sl & 3) >> 1) : 2 * t + ((sl & 3) >> 1);
    const int place = c ^ (4 * (kr >> 1)) ^ (ROWS == 16 ? 2 * (h & 1) : 0);
    bread[t] = (uint32_t)(((8 * h + kr) * FCN + place) * 16 + (sl & 1) * 8);
  }

  const int p_begin = indptr[i];
  const int nblk = indptr[i + 1] - p_begin;
  const int ksteps = blk / kTileK;                       // ROWS = 32: steps per block
  const int chunks = nblk * sub;                         // ROWS = 16: two per step
  const int steps = ROWS == 32 ? nblk * ksteps : (chunks + 1) / 2;
  // The block columns of the row's first 64 blocks are fetched once, one per lane: looking them up
  // step by step would put a second memory round trip in front of every step's loads of X.
  const int j_lane = lane < nblk ? indices[p_begin + lane] : 0;
  auto column = [&](int b) -> int64_t {
    return b < kWave ? __builtin_amdgcn_readlane(j_lane, b) : indices[p_begin + b];
  };

  u32x4 xr[4], ar[2];
  auto fetch = [&](int it) {
    if constexpr (ROWS == 32) {
      const int b = it / ksteps, k0 = (it - b * ksteps) * kTileK;
      const uint16_t* ab = A + (int64_t)(p_begin + b) * blk * blk + (int64_t)(bi0 + n) * blk + k0 + 8 * h;
      ar[0] = *reinterpret_cast<const Halves8*>(ab);
      ar[1] = *reinterpret_cast<const Halves8*>(ab + 16);
      const uint16_t* xb = X + (column(b) * blk + k0) * feat + f0 + xoff;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        xr[u] = u32x4{0, 0, 0, 0};
        if (xlive) xr[u] = *reinterpret_cast<const Halves8*>(xb + (int64_t)(8 * u) * feat);
      }
    } else {
      const int c0 = 2 * it, b0 = c0 / sub, b1 = (c0 + 1) / sub;
      const bool two = c0 + 1 < chunks;
      const int ba = h >> 1 ? b1 : b0, ca = c0 + (h >> 1) - ba * sub;
      ar[0] = u32x4{0, 0, 0, 0};
      if (h < 2 || two)
        ar[0] = *reinterpret_cast<const Halves8*>(A + (int64_t)(p_begin + ba) * blk * blk + (int64_t)(bi0 + n) * blk +
                                                16 * ca + 8 * (h & 1));
      const uint16_t* x0 = X + (column(b0) * blk + 16 * (c0 - b0 * sub)) * feat + f0 + xoff;
      const uint16_t* x1 = X + (column(two ? b1 : b0) * blk + 16 * (two ? c0 + 1 - b1 * sub : 0)) * feat + f0 + xoff;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        xr[u] = u32x4{0, 0, 0, 0};
        if (xlive && (u < 2 || two))
          xr[u] = *reinterpret_cast<const Halves8*>((u < 2 ? x0 : x1) + (int64_t)(8 * (u & 1)) * feat);
      }
    }
  };

  typename std::conditional<ROWS == 32, f32x16, f32x4>::type acc[TILES];
#pragma unroll
  for (int t = 0; t < TILES; ++t)
#pragma unroll
    for (int v = 0; v < REGS; ++v) acc[t][v] = 0.f;

  if (wave < steps) fetch(wave);
  for (int it = wave; it < steps; it += kSplitWaves) {
    const u32x4 a0 = ar[0], a1 = ar[1];
#pragma unroll
    for (int u = 0; u < 4; ++u) *reinterpret_cast<u32x4*>(stage + xdst[u]) = xr[u];
    if (it + kSplitWaves < steps) fetch(it + kSplitWaves);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      if constexpr (ROWS == 32) {
        acc[t] = mfma32<BF16>(a0, read_b(stage + bread[t], 4 * FCN * 16), acc[t]);
        acc[t] = mfma32<BF16>(a1, read_b(stage + bread[t] + 16 * FCN * 16, 4 * FCN * 16), acc[t]);
      } else {
        acc[t] = mfma16<BF16>(a0, read_b(stage + bread[t], 4 * FCN * 16), acc[t]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_wave_barrier();  // the next step's stores come after these reads
  }

  // ---- add the partial results
  __syncthreads();  // every wavefront is done with its tile
  float* red = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int t = 0; t < TILES; ++t)
#pragma unroll
    for (int v = 0; v < REGS; ++v) red[wave * ELEMS + (t * REGS + v) * kWave + lane] = acc[t][v];
  __syncthreads();
  const int used = min(steps, kSplitWaves);
#pragma unroll
  for (int e0 = 0; e0 < ELEMS; e0 += 64 * kSplitWaves) {
    const int e = e0 + tid, l = e & 63, v = (e >> 6) % REGS, t = (e >> 6) / REGS;
    float sum = 0.f;
    for (int w = 0; w < used; ++w) sum += red[w * ELEMS + e];
    int row, col;
    if constexpr (ROWS == 32)
      row = (v & 3) + 4 * (l >> 5) + 8 * (v >> 2), col = f0 + 32 * t + (l & 31);
    else
      row = 4 * (l >> 4) + v, col = f0 + 16 * t + (l & 15);
    if (col >= feat) continue;
    const int64_t off = ((int64_t)i_out * blk + bi0 + row) * feat + col;
    if constexpr (OUT == 1)
      static_cast<float*>(Y)[off] = sum;
    else
      static_cast<uint16_t*>(Y)[off] = to16<BF16>(sum);
  }
}

// How a product is launched.
struct BsrForm {
  enum Kernel { kSplit, kWaves, kGroups } kernel;  // wavefronts take steps in turn, tiles by a wavefront, by workgroups of four
  bool wide;     // tiles of 256 features, else of 128 (kSplit by bsr_split_kernel: of kSplitF)
  bool ranked;   // block rows in order of their length
  bool by_rows;  // block rows dealt to XCDs
  int direct = 0;  // operands in registers, so many wavefronts to a tile (16-row slices: kWaves too may have several, and
                   // kGroups with two of them has two tiles of 128 features to a workgroup)
  bool single = false;  // the direct kernels with one step of a wavefront on its way
};

inline int slice_rows(int blk, BsrForm::Kernel kernel) {
  return blk % 32 != 0 ? 16 : kernel == BsrForm::kGroups && blk % 64 == 0 ? 64 : 32;
}

// floats: fp32 results
BsrForm bsr_form(int64_t cus, int mb, int nb, int blk, int feat, int64_t nnzb, bool floats) {
  const int unit = slice_rows(blk, BsrForm::kSplit);
  const int64_t unit_slices = (int64_t)mb * (blk / unit);
  const int64_t steps = nnzb * (blk / 16) / 2 / mb;  // of a slice, 32 columns each, on average
  const bool wavefronts = feat < (1 << 25) && blk <= 4096;  // offsets of a load in 32 bits
  const int64_t split = 8 * stir::ceil_div(unit_slices * stir::ceil_div(feat, kSplitF), 8);
  const int64_t tiles = unit_slices * stir::ceil_div(feat, kTileF);
  auto x_tile_bytes = [&](int width) { return (int64_t)nb * blk * 2 * width; };
  // Of the rows of X that a tile of 256 features reads: what an L2 holds beside A, an L2, far more; of A: the last level.
  constexpr int64_t kMuchX = 3 << 20, kBeyondL2 = 4000000, kFarX = 6000000, kLastLevel = 256 << 20;
  if (unit == 32 && wavefronts) {
    // Tiles of 64 features, by eight wavefronts through LDS, where rows are long and tiles of 128 leave CUs without one or,
    // hardly more than the CUs, with twice as much as the next: 35 x 437 blocks, 97 steps, 96 features 14.6 us, 16.9 with 128;
    // 42 x 285, 70 steps, 64 10.6, 11.3; 93 x 431, 106 steps, 320 (279 tiles) 26.0, 29.6; but 136 x 333, 67 steps, 256 (272, and
    // 544 of 64) 24.1, 20.8.  A little sooner where 128 waste half of a load: 8 x 35 of 128, 35 steps, 192 features 9.4, 10.1.
    // Of 64 features alone from 20 steps on: 77 x 115 of 128, 21 steps 13.3, 14.6, 24 x 99 of 64, 29 steps 8.6, 9.5; and from 32
    // steps on in two turns: 189 x 56 of 128, 154 steps (756) 58.5, 76.4 (260 drawn shapes 0.87 of the time, none above 1.04).
    // Three quarters of a turn where the last 64 are half empty, 62 x 196 of 32, 66 steps, 224 features (248) 12.1, 11.6; all of it from
    // 100 steps on: 17 x 150 of 96, 275 steps, 224 features 35.5, 42.8 (1000 drawn shapes 0.91, none above 1.03).
    const bool half = feat % kTileF != 0 && feat % kTileF <= kSplitF;
    const bool ragged = feat % kSplitF != 0 && (steps < 100 || feat <= kTileF);
    if ((steps >= 40 && (split * 4 <= (ragged ? 3 : 4) * cus || (tiles > cus && split <= 2 * cus))) ||
        (steps >= 32 && half && split <= cus) || (steps >= 20 && feat <= kSplitF && split <= (steps < 32 ? 2 : 4) * cus))
      return {BsrForm::kSplit, false, false, false};
    // Steps in turn as long as that leaves a CU little more than two workgroups of four wavefronts, or four of two.  Means over
    // 5000 drawn shapes, four wavefronts to a tile / two: up to 1.5 tiles a CU 0.7 to 0.95, 1.5 to 2.25 0.92 to 1.0 (the latter for 4
    // to 8 steps: 107 x 48 blocks, 544 features 8.3 / 7.3), 2.25 to 2.75 1.0 to 1.14; two / one: up to 3.25 0.6 to 0.97, 3.25 to 4
    // 0.85 to 0.98, 4 to 5 0.91 to 1.17.  Several wavefronts store the results sooner, so two also where fp32 results are most of the
    // work (up to 3 steps 0.96; 252 x 36, 3 steps, 320 features 7.4 / 8.9), but not for 16-bit ones (1.05; 62 x 35, 2 steps, 2048
    // features 7.3 / 6.2).  With far more X than the L2s hold one passes two sooner, 37 x 441, 102 steps, 2848 features (3.3 tiles) 59
    // / 69.  Eight where a CU has one tile and many steps: 131 x 322, 78 steps, 128 features 14.9, four 16.2.
    const bool few = steps < 4, apart = blk % 64 != 0;  // apart: no workgroup of 64 rows
    if (tiles <= cus && steps >= 24) return {BsrForm::kSplit, false, false, false, 8};
    const int four = apart ? (steps < 8 ? 8 : 9) : few ? 6 : steps < 48 ? 9 : 11;
    if (tiles * 4 <= four * cus) return {BsrForm::kSplit, false, false, false, 4};
    // (64 rows that share X, by a workgroup below, pass two wavefronts in turn where rows are long and CUs have more than three
    // tiles: blocks of 64, 672 features, 46 steps (804 tiles) 31 / 37, 928, 31 steps (817) 23 / 26, of 128, 2304, 92 steps (792) 50 /
    // 57; but of 64, 2240, 30 steps (755) 23.0 / 19.7; and with few steps.  Four pass two from 48 steps on up to 2.75 tiles, 0.93 of
    // the time over 3200 drawn shapes: 22 x 126 of 128, 136 steps, 864 features, fp32 results 66 / 74.  Up to 24 steps two keep 3 to
    // 3.25 tiles of blocks of 64 where there is X enough, 0.99; over little of it the workgroups take 0.95, and of 128 dealt to XCDs
    // 0.97: 51 x 7 of 128, 21 steps, 416 features, fp32 results 13.2 / 17.1)
    const int two = few && !(apart && floats)           ? 0
                    : apart                             ? (x_tile_bytes(kWaveF) <= kFarX ? 16 : 13)
                    : steps >= 48   ? 0
                                    : (blk < 128 && steps < 24 && x_tile_bytes(kWaveF) > 1000000 ? 13 : 12);
    if (tiles * 4 <= two * cus) return {BsrForm::kSplit, false, false, false, 2};
  } else if (unit == 32) {
    // The split form wins as long as its workgroups are resident at once, two per CU, and up to twice as many where block rows
    // have enough steps to pay for the second turn.
    if (split <= 2 * cus || (split <= 4 * cus && steps >= 32)) return {BsrForm::kSplit, false, false, false};
  }
  const int64_t wide_tiles = stir::ceil_div(feat, kWaveF), waste = wide_tiles * kWaveF - feat;
  // Slices in order of their length (row_of_rank) where that makes up for finding the row, which costs as much as 2 or 3
  // steps: with the rows of X of a feature tile (x_bytes) more than an XCD's L2 holds beside A, since what runs side by
  // side then reads the same of them; and with long block rows, since the longest do not come last.  Not with few
  // workgroups or wavefronts, which are resident at once in any order.  In order of length / as they come, us:
  //   wavefronts of 32 x 256, 2048 block rows, 512 columns of blocks (8.4 MB of X in a tile), 1024 features: 3 steps 80 / 62,
  //   10 steps 141 / 148, 16 184 / 218, 32 270 / 389; 305 columns (5 MB) 16 steps 156 / 154, 32 254 / 279; 256 features, 512
  //   columns, 16 steps 63 / 54;
  //   four wavefronts, blocks of 64: 1024 rows, 256 columns, 1024 features 12 steps 141 / 119, 24 208 / 209, 48 345 / 387;
  //   128 features a tile: 256 rows, 512 features 12 steps 24.5 / 22.3, 1024 rows, 24 steps 126 / 132, 48 224 / 246; lengths
  //   that differ by a factor of ten, 500 rows, 152 columns, 512 features 33 steps 78 / 113.
  // Among those that come as they are, wavefronts of 128 features, whose X an L2 still holds, pass those of 256 then (10
  // steps of the first 127 us).
  auto rank_pays = [&](int64_t x_bytes, int64_t tiles, int64_t count, int per_cu) {
    return x_tile_bytes(std::min(feat, kWaveF)) > kMuchX && count >= per_cu * cus &&
           (steps >= 28 || (steps >= 16 && tiles >= 2 && x_bytes > kBeyondL2));
  };
  if (unit == 16) {
    // Offsets of a load in 32 bits: bsr16_direct_kernel and bsr16_wave_kernel allow for more than the others.
    if (feat >= (1 << 27) || blk >= (1 << 15)) return {BsrForm::kSplit, false, false, false};
    if (!wavefronts) return {BsrForm::kGroups, feat >= kWaveF, false, false, feat >= kWaveF ? 2 : 4};
    // Below, "128" are tiles of 128 features by so many wavefronts, "two of 128" the two tiles of a workgroup by two wavefronts
    // each, "256" tiles of 256 by one wavefront (or four); us.
    const bool several = blk > 16;
    const int64_t narrow_tiles = stir::ceil_div(feat, kTileF), waves = unit_slices * wide_tiles;
    const int64_t x_bytes = x_tile_bytes(kWaveF), x_narrow = x_tile_bytes(kTileF);
    const bool even = narrow_tiles % 2 == 0, fits = waves >= 8 * cus && waste * 8 <= feat;
    // Long rows and hardly more tiles than CUs, eight wavefronts with 64 features through LDS / 128 by four / by eight: 29 x 148
    // blocks of 80, 46 steps, 160 features 14.4 / 15.4 / 15.2, 100 x 592 of 16, 19 steps, 320 8.9 / 9.6 / -; and where 128 waste half
    // of a load also up to eight of 64 to a CU: 64 features, 51 steps (402) 13.3 / 13.8 / 13.4, 192, 107 steps (1926) 58.8 / 65.0 / 62.9.
    const bool half = feat % kTileF != 0 && feat % kTileF <= kSplitF;
    if (tiles > cus && ((half && steps >= (feat <= kSplitF ? 32 : 64) && split <= 8 * cus) ||
                        (steps >= 40 && split <= 2 * cus) || (steps >= 18 && tiles * 4 <= 5 * cus && split <= 2 * cus)))
      return {BsrForm::kSplit, false, false, false};
    // 128 by four / by eight: 80 steps, 96 features (154 tiles) 16.5 / 13.0, 33 steps (136) 8.5 / 7.6, 15 steps (220) 5.6 / 5.6; 60
    // steps (399) 15.7 / 15.4, 22 steps (996) 14.8 / 16.0.
    // Of blocks of several slices with much X, 64 by eight through LDS also where 128 have no more than a turn, from 100 steps on: 3 x
    // 68 of 144, 196 steps, 416 features 24.3, 28.5 (1300 drawn shapes of 80 and more 0.91 of the time).
    if (blk >= 80 && feat > kTileF && steps >= 100 && x_bytes > kBeyondL2 && split <= cus) return {BsrForm::kSplit, false, false, false};
    if (tiles <= cus && steps >= 20) return {BsrForm::kSplit, false, false, false, 8};
    // Much X and long rows, blocks of several slices, which read the same X: 256 by four in order of length.  Of the time by one
    // wavefront (ranked), 28 steps and more, blocks of 80 and up 0.89 to 0.95, as they come 0.93 to 0.97, 128 by four 0.96 to 1.0; of
    // 48, 0.90 with more than 9 MB of X, 0.98 from 36 steps on.  With less of both 1.02, as they come 1.01, 128 by four 0.97 (388 x
    // 309, 28 steps, 1408 features 176 / 164 / 148).  And one feature tile gives the order nothing to share: 128 by four 0.81 to 0.95
    // of the time in order with 28 to 35 steps, 0.89 to 1.02 with more (763 x 273 of 48, 30 steps 79 / 62).
    if (several && x_bytes > kMuchX && feat > kTileF && steps >= 28 && waste * 8 <= feat && waves >= 6 * cus) {
      const bool order = wide_tiles > 1 && (blk > 48 || steps >= 36 || x_bytes > 9000000);
      return {BsrForm::kWaves, order, order, false, 4};
    }
    // Much X else: in order of length, by one wavefront, 128 or 256 by what the last tile of 256 wastes.  128 by four as they come / 128
    // ranked / 256 ranked: blocks of 16, 1024 columns (8.4 MB), 51 steps, 1024 features 205 / 188 / 163, 24 steps 105 / 104 / 94,
    // 4096 features 1204 / 736 / 618; 829 columns, 49 steps, 1632 features (12.75 tiles of 128) 200 / 170 / 184.
    // With far more X than an L2 holds and many tiles 128 from 20 steps on and 256 only from 44: 799 columns, 24 steps, 1632 features 167
    // / 145 / 163, 993, 22 steps, 3744 108 / 101 / 115, 872, 32 steps, 3168 231 / 206 / 234, 905, 32 steps, 3680, fp32 results 256 / 223 /
    // 250, 31 drawn shapes of 28 to 44 steps 0.96 of the time of 256; less of it, 722 columns, 25 steps, 2752 174 / 176 / 173, 575, 16 steps, 2784
    // 39 / 42 / 39.  From 16 steps on 256 with few tiles, where the order gives little: 1024 columns, 24 steps, 1024 features 100 / 99 /
    // 90, but 490, 17 steps, 512 34 / 40 / 40.
    // Blocks of several slices, with what such tiles of 256 would waste or too few of them, from 36 steps on; 128 by four as they come
    // are 0.89 to 0.95 of the time below (600 drawn shapes, 4 to 40 MB of X; none above 1.11), 0.92 to 1.02 above: 78 x 108 of 112, 26
    // steps, 832 features 83 ranked, 72.
    const bool wide_ranked = fits && (even || waste * 16 <= feat);
    if (x_bytes > kMuchX && feat > kTileF && steps >= (several ? 36 : 16) && !(several && fits)) {
      const int wide_from = x_bytes > kFarX && wide_tiles > 4 ? 44 : 28;
      if (wide_ranked && (steps >= wide_from || (wide_tiles >= 2 && wide_tiles <= 4 && x_bytes > kBeyondL2)))
        return {BsrForm::kWaves, true, true, false, 1};
      const bool long_enough = !wide_ranked && (steps >= 28 || x_narrow > kBeyondL2);
      if (unit_slices * narrow_tiles >= (fits ? 8 : 10) * cus && (long_enough || (steps >= 20 && x_bytes > kFarX)))
        return {BsrForm::kWaves, false, true, false, 1};
    }
    // Long rows, far more X than an L2 holds and a turn of wavefronts: by one, which stay closer together in X, with one step on its
    // way each where there are more of them; 128 by four / by one with two steps / with one: 95 x 793, 26 steps, 1856 features
    // (1425 tiles) 24.8 / 22.1 / 23.7, 80 x 818, 23 steps, 2848 (1840) 34.5 / 30.9 / 28.6, 70 x 896, 40 steps, 2848 (1610) 48.4 / 40.6 /
    // 37.8, 183 x 840, 64 steps, 1568 (2379) 84.5 / 83.5 / 80.6; but 4.35 tiles to a CU, 90 steps, 320 features 50.5 / 52.3 / 61.5.
    // With many feature tiles from 15 steps and 5 MB on, 0.93 of the time of 128 by four over 2300 drawn shapes: 100 x 902, 18 steps,
    // 2912 features (2300) 29.7 / 36.6, 79 x 657, 20 steps, 3616 (2291) 29.9 / 36.6, 44 x 626, 26 steps, 4064 (1408) 24.8 / 30.7.
    const bool far = (steps >= 20 && x_bytes > kFarX) || (steps >= 15 && x_bytes > 5000000 && wide_tiles > 4);
    if (!several && far && tiles * 10 >= 46 * cus && tiles < 10 * cus)
      return {BsrForm::kWaves, false, false, false, 1, tiles >= 6 * cus};
    // Blocks of several slices else.  A, which every tile reads, more than the last level holds, 128 by four / 256 by four / by one:
    // 3000 x 68 of 80, 20 steps, 800 features 1317 / 1009 / 1067.  Wide tiles and enough of them: from 16 steps on 256 by four, 0.92
    // to 1.0 of the time by one (blocks of 48 with much X 128 by four, 0.965 of that: 269 x 331, 25 steps, 1248 features, fp32 results
    // 109 / 118); with 5 to 15 steps two of 128, 0.91 to 0.97 of the time of 256 by one whatever X (1100 x 341 of 48, 10
    // steps, 1024 features 256 by one / by four / two of 128 142 / 135 / 118); with fewer 128 by one (below), 0.92.  Far more X than
    // an L2 holds and less than 16 steps, 128 by four / two of 128: 1214 x 659 of 80, 10 steps, 416 features 138 / 130, with more steps
    // 0.84 / 1.
    if (several && feat > kTileF && (nnzb * blk * blk * 2 > kLastLevel || (fits && steps >= 16 && (x_bytes > kMuchX ? blk > 48 : even))))
      return {BsrForm::kWaves, true, false, false, 4};
    if (several && feat >= kWaveF && steps < 16 && (x_bytes > 15000000 || (fits && steps >= 5)))
      return {BsrForm::kGroups, true, false, false, 2};
    // X in an L2, 128 by one / by four / two of 128 / 256: 342 x 83 of 16, 4 steps, 1728 features 14.8 / 17.2 / 16.2 / 16.7; 420
    // columns, 10 steps, 512 24.5 / 24.5 / - / 23.3; 300, 12 steps, 1024 47.8 / 47.2 / - / 43.7; 73, 8 steps, 3904 67 / 73 / 65 /
    // 63; 65, 7 steps, 224 features (1254 tiles) 8.7 / 9.0 / 8.4 / 9.3; 92, 8 steps, 160 (1498) 11.1 / 11.5 / 9.1 / 9.9.
    if (steps <= 4 && tiles >= 6 * cus && x_bytes <= 2500000) return {BsrForm::kWaves, false, false, false, 1};
    if (!several && fits && even && x_bytes <= 3500000) return {BsrForm::kWaves, true, false, false, 1};
    if (feat > kTileF && x_bytes <= 2500000 && tiles * 4 >= (even ? 19 : 48) * cus && steps < 20)
      return {BsrForm::kGroups, true, false, false, 2};
    // 128 by one / by four: 5 steps, 1696 features (1442 tiles) 9.4 / 9.8, 3 steps (1140) 9.1 / 7.6; 6 steps, 1024 columns (8000)
    // 37.2 / 37.1; of 48, 11 steps, 320 features (33 k) 230 / 208, of 80, 8 steps, 800 (105 k) 468 / 473.
    if ((steps <= 5 && tiles >= 5 * cus) || (steps <= 11 && tiles >= 40 * cus)) return {BsrForm::kWaves, false, false, false, 1};
    // Many steps, by four / by eight: 202 columns of 80, 105 steps, 896 features (2135 tiles) 108.5 / 105.4, 68 steps, 96 features
    // (842) 28.2 / 27.3; but 94 steps, 3776 (3450) 132 / 135.
    return {tiles < 8 * cus ? BsrForm::kSplit : BsrForm::kWaves, false, false, false, steps >= 64 && tiles < 9 * cus ? 8 : 4};
  }
  const int rs = slice_rows(blk, BsrForm::kGroups) / 32;
  const int64_t slices = (int64_t)mb * (blk / (32 * rs));
  // Two 32-wide accumulators per wavefront once the feature axis is wide enough to still yield workgroups for the chip,
  // 1.6 per CU (us with one / two): 22 x 246 blocks of 64, 2752 features (242 workgroups of two) 56 / 63, 45 x 45 of 128,
  // 1024 (360) 20.6 / 21.6, 60 x 100 of 64, 2048 (480) 26.0 / 24.5, 70 x 60
  // (560) 34.4 / 29.6, 98 x 90, 2432 (980) 45.8 / 38.6.  One prefetched step is enough: measured on MI355X, deeper
  // register rings (2-6 steps) change nothing, the kernel is not bound by latency.
  const int nt = feat >= 1024 && slices * stir::ceil_div(feat, 2 * kTileF) * 5 >= 8 * cus ? 2 : 1;
  // Slices of 32 rows, a wavefront to a tile.  256 features to a wavefront take X through the L1s at twice the length of a load
  // and A half as often; 128 have more wavefronts, and less X in a tile.  us with 128 / 256: 77 x 65 blocks, 7 steps, 1312
  // features (462 wavefronts of 256) 10.1 / 11.3, 152 x 56, 8 steps, 1056 (760) 13.2 / 12.1, 403 x 191, 40 steps, 512 (806) 42.5
  // / 36.8, 307 x 92, 21 steps, 2496 (3070) 73 / 65; a last tile mostly empty 344 x 57, 6 steps, 288 features 10.1 / 11.6; with
  // much X 117 x 257, 20 steps, 2176 (1053, 4.2 MB) 31.6 / 32.5, 109 x 259, 29 steps, 2208 (981) 40.1 / 35.4, 87 x 423, 55
  // steps, 2784 (957, 6.9 MB) 78 / 69.  Blocks of several slices, which read the same X, with much of it: 256 up to twice
  // what an L2 holds, or by workgroups: 400 x 170 of 96 (8.4 MB), 16 steps, 512 features 50 ranked, 60 with 256 as they come,
  // 65 with 128, 64 by workgroups; 1300 x 325 (16 MB), 8 steps, 1504 features 310, 352, 429, 280.
  // Long rows, more X than an L2 holds and a turn of wavefronts: 128 with one step on their way each and four to a SIMD stay closer
  // together in X; 128 / 128 with one step / 256 (6 to 8.2 MB of X in 256): 80 x 501, 61 steps, 2720 features (1760 wavefronts of 128)
  // 88 / 74 / 87, 53 x 495, 45 steps, 3712 (1537) 52 / 50.5 / 59, 60 x 500, 101 steps, 2720 (1320) 96 / 86 / 88; but 40 x 500, 46
  // steps, 3712 (1160) 41.6 / 43.2 / 47, and with many more 139 x 437, 24
  // steps, 3040 (3336) 73 / 71 / 67.
  // Up to four steps a row 128: the results are most of it, and leave sooner (381 x 87, 3 steps, 1536 features 15.2 / - / 15.7, fp32
  // results 19.9 / - / 22.5).
  if (rs == 1 && wavefronts) {
    const bool one = blk == 32;
    const int64_t waves = slices * wide_tiles, x_bytes = x_tile_bytes(std::min(feat, kWaveF));
    const bool crowd = one && steps >= 20 && x_bytes > kMuchX && tiles >= 5 * cus && tiles * 2 <= 17 * cus;
    if (crowd) return {BsrForm::kWaves, false, false, false, 1, true};
    const bool ranked = waste * 3 <= feat && rank_pays(x_bytes, wide_tiles, waves, steps >= 64 && wide_tiles >= 4 ? 3 : 5);
    const bool wide = ranked || (x_bytes <= kMuchX ? waste * 3 <= feat && waves * 10 >= 27 * cus && steps > 4
                                 : !one            ? waste * 8 <= feat && x_bytes <= 2 * kBeyondL2 && waves >= 8 * cus
                                 : steps >= 24     ? waste * 4 <= feat && waves >= 3 * cus
                                                   : waste * 8 <= feat && x_bytes <= kBeyondL2 && waves >= 5 * cus);
    if (wide) return {BsrForm::kWaves, true, ranked, false};
    if (one || x_bytes <= kMuchX) return {BsrForm::kWaves, false, false, false, 1};
  }
  const int64_t f_tiles = stir::ceil_div(feat, kTileF * nt);
  // 16384 x 16384, 10 %, 4096 features: 64 x 64 blocks 424 -> 352 us in ranked order, 128 x 128 345 -> 324
  const bool ranked = rs == 2 && rank_pays(x_tile_bytes(std::min(feat, kTileF * nt)), f_tiles, slices * f_tiles, 3);
  // Blocks of 128 rows and more: block rows dealt to XCDs (decode_tile_by_rows).  Measured at
  // 16384^2, 10 %, 4096 features: 128 x 128 blocks 387 -> 365 us; 64 x 64 blocks (one slice per
  // block row, so only A is shared) 443 -> 514 us: there the feature tile per XCD, which keeps an
  // XCD on one slice of X, is worth more.
  // Few block rows do not go round eight XCDs: 12 block rows (40 x 128 columns, 3008 features) 30.8 us, 26.3 in the
  // other order; 20 (of 20, 4096) 33.4, 29.1; 45 (of 45, 1024) 21.6, 24.1.
  const bool rows_go_round = 8 * stir::ceil_div((int64_t)mb, 8) * 7 <= 8 * (int64_t)mb;
  return {BsrForm::kGroups, nt == 2, ranked, rs == 2 && blk >= 128 && f_tiles >= 2 && rows_go_round};
}

}  // namespace

static int bsr_launch(int32_t dtype, int32_t out_dtype, int32_t mb, int32_t nb, int32_t blk, int32_t feat,
                      int64_t nnzb, const void* d_A, const void* d_X, void* d_Y, const int32_t* d_indptr,
                      const int32_t* d_indices, const int32_t* d_row_ids, void* stream) {
  STIR_REQUIRE(dtype == STIR_F16 || dtype == STIR_BF16, "bsr_spmm: dtype must be STIR_F16 or STIR_BF16");
  STIR_REQUIRE(out_dtype == dtype || out_dtype == STIR_F32, "bsr_spmm: out_dtype must equal dtype or be STIR_F32");
  STIR_REQUIRE(mb >= 0 && nb >= 0 && nnzb >= 0, "bsr_spmm: bad sizes mb=%d nb=%d", mb, nb);
  STIR_REQUIRE(blk > 0 && blk % 16 == 0, "bsr_spmm: blk=%d must be a multiple of 16", blk);
  STIR_REQUIRE(feat > 0 && feat % 32 == 0, "bsr_spmm: feat=%d must be a multiple of 32", feat);
  if (mb == 0) return 0;
  STIR_REQUIRE(d_X && d_Y && d_indptr && (nnzb == 0 || (d_A && d_indices)), "bsr_spmm: null pointer argument");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint16_t* A = static_cast<const uint16_t*>(d_A);
  const uint16_t* X = static_cast<const uint16_t*>(d_X);
  const BsrForm form = bsr_form(stir::compute_units(), mb, nb, blk, feat, nnzb, out_dtype == STIR_F32);
  const int unit = slice_rows(blk, form.kernel), sub = blk / unit;
  const int f_tiles = (int)stir::ceil_div(feat, form.kernel == BsrForm::kSplit && !form.direct ? kSplitF : form.wide ? kWaveF : kTileF);
  const int64_t slices = (int64_t)mb * sub;
  auto eights = [](int64_t n) { return 8 * stir::ceil_div(n, 8); };  // see decode_tile, decode_ranked
  const int64_t blocks = form.by_rows  ? eights(mb) * sub * f_tiles
                         : form.ranked ? eights((int64_t)mb * f_tiles) * sub
                                       : eights(slices * f_tiles);
  STIR_REQUIRE(blocks < (int64_t(1) << 31), "bsr_spmm: too many tiles for one launch");
  const dim3 grid((unsigned)blocks);
  const int ranked = form.ranked, by_rows = form.by_rows;
#define STIR_BSR_GO(KERNEL, THREADS, ...)                                                                      \
  hipLaunchKernelGGL(KERNEL, grid, dim3(THREADS), 0, st, blk, feat, slices, f_tiles, ##__VA_ARGS__, A, X, d_Y, \
                     d_indptr, d_indices, d_row_ids)
#define STIR_ARGS(...) __VA_ARGS__
#define STIR_BSR_16(ARGS, WAVES)                                                                               \
  do {                                                                                                         \
    if (blk == 16) STIR_BSR_GO((bsr16_direct_kernel<STIR_ARGS ARGS, true>), (WAVES) * kWave, ranked);          \
    else STIR_BSR_GO((bsr16_direct_kernel<STIR_ARGS ARGS, false>), (WAVES) * kWave, ranked);                   \
  } while (0)
#define STIR_BSR(BF, OUT)                                                                                      \
  do {                                                                                                         \
    if (form.direct && unit == 16) {                                                                           \
      if (form.kernel == BsrForm::kGroups && form.direct == 2) STIR_BSR_16((BF, OUT, 2, 2), 4);                \
      else if (form.wide && blk == 16) STIR_BSR_GO((bsr16_wave_kernel<BF, OUT, true>), kWave, ranked);         \
      else if (form.wide) STIR_BSR_GO((bsr16_wave_kernel<BF, OUT, false>), 4 * kWave, ranked);                 \
      else if (form.single && blk == 16)                                                                       \
        STIR_BSR_GO((bsr16_direct_kernel<BF, OUT, 1, 1, true, 1>), kWave, ranked);                             \
      else if (form.direct == 1) STIR_BSR_16((BF, OUT, 1, 1), 1);                                              \
      else if (form.direct == 4) STIR_BSR_16((BF, OUT, 4, 1), 4);                                              \
      else STIR_BSR_16((BF, OUT, 8, 1), 8);                                                                    \
    } else if (form.direct) {                                                                                  \
      if (form.single) STIR_BSR_GO((bsr_direct_kernel<BF, OUT, 1, 1>), kWave);                                 \
      else if (form.direct == 1) STIR_BSR_GO((bsr_direct_kernel<BF, OUT, 1>), kWave);                          \
      else if (form.direct == 8) STIR_BSR_GO((bsr_direct_kernel<BF, OUT, 8>), 8 * kWave);                      \
      else if (form.direct == 4) STIR_BSR_GO((bsr_direct_kernel<BF, OUT, 4>), 4 * kWave);                      \
      else STIR_BSR_GO((bsr_direct_kernel<BF, OUT, 2>), 2 * kWave);                                            \
    } else if (form.kernel == BsrForm::kSplit) {                                                               \
      if (unit == 16) STIR_BSR_GO((bsr_split_kernel<BF, OUT, 16>), kWave * kSplitWaves);                       \
      else STIR_BSR_GO((bsr_split_kernel<BF, OUT, 32>), kWave * kSplitWaves);                                  \
    } else if (form.kernel == BsrForm::kWaves) {                                                               \
      STIR_BSR_GO((bsr_wave_kernel<BF, OUT>), kWave, ranked);                                                  \
    } else if (unit == 64) {                                                                                   \
      if (form.wide) STIR_BSR_GO((bsr_spmm_kernel<BF, OUT, 2, 2>), 256, by_rows, ranked);                      \
      else STIR_BSR_GO((bsr_spmm_kernel<BF, OUT, 1, 2>), 256, by_rows, ranked);                                \
    } else {                                                                                                   \
      if (form.wide) STIR_BSR_GO((bsr_spmm_kernel<BF, OUT, 2, 1>), 256, by_rows, ranked);                      \
      else STIR_BSR_GO((bsr_spmm_kernel<BF, OUT, 1, 1>), 256, by_rows, ranked);                                \
    }                                                                                                          \
  } while (0)
  if (dtype == STIR_BF16) {
    if (out_dtype == STIR_F32) STIR_BSR(true, 1); else STIR_BSR(true, 0);
  } else {
    if (out_dtype == STIR_F32) STIR_BSR(false, 1); else STIR_BSR(false, 0);
  }
#undef STIR_BSR
#undef STIR_BSR_16
#undef STIR_ARGS
#undef STIR_BSR_GO
  STIR_LAUNCH_CHECK();
  return 0;
}

extern "C" {

// The form of a product on a device of so many compute units: kernel, then 4 for 256 features a tile, 8 for block rows
// in order of their length, 16 for block rows dealt to XCDs, 32 times BsrForm::direct, 512 for BsrForm::single; -1 for what no
// product is.  For the tests, which say what they cover.
int stir_bsr_form(int32_t cus, int32_t mb, int32_t nb, int32_t blk, int32_t feat, int64_t nnzb, int32_t floats) {
  if (cus <= 0 || mb <= 0 || nb < 0 || nnzb < 0 || blk <= 0 || blk % 16 != 0 || feat <= 0) return -1;
  const BsrForm f = bsr_form(cus, mb, nb, blk, feat, nnzb, floats != 0);
  return f.kernel + 4 * f.wide + 8 * f.ranked + 16 * f.by_rows + 32 * f.direct + 512 * f.single;
}

int stir_bsr_spmm(int32_t dtype, int32_t out_dtype, int32_t mb, int32_t nb, int32_t blk, int32_t feat,
                  int64_t nnzb, const void* d_A, const void* d_X, void* d_Y, const int32_t* d_indptr,
                  const int32_t* d_indices, void* stream) {
  return bsr_launch(dtype, out_dtype, mb, nb, blk, feat, nnzb, d_A, d_X, d_Y, d_indptr, d_indices, nullptr,
                    stream);
}

int stir_dbsr_spmm(int32_t dtype, int32_t out_dtype, int32_t nnz_rows, int32_t nb, int32_t blk,
                   int32_t feat, int64_t nnzb, const void* d_A, const void* d_X, void* d_Y,
                   const int32_t* d_row_ids, const int32_t* d_indptr, const int32_t* d_indices,
                   void* stream) {
  STIR_REQUIRE(nnz_rows == 0 || d_row_ids, "dbsr_spmm: row ids are null");
  return bsr_launch(dtype, out_dtype, nnz_rows, nb, blk, feat, nnzb, d_A, d_X, d_Y, d_indptr, d_indices,
                    d_row_ids, stream);
}

}  // extern "C"
