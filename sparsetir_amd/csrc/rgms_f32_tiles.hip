// Destination-tiled fp32 RGMS declared in rgms_f32_tiles.h: index construction and the kernels.
//
// Index (once per plan): every slot of the ELL3D buckets -- or every stored column of the CSF
// arrays -- is an edge with the key (destination row / 128, relation, destination row % 128).  One
// stable radix sort orders the edges by key; runs of equal key are the (relation, row) pairs, cut
// into pieces of at most EMAX = 32 / KS edges (a second key: key << 20 | position in the run /
// EMAX, run-length encoded).  The pairs of one (tile, relation) run are cut into batches of at
// most 16 pairs and at most EMAX places, listed per tile.  The places of a batch are columns of four: the
// edges of a pair stand in them one below the other, as chains of at most four.
// An edge record holds the source row, the address of the edge's weight (weights are read at
// every launch) and its part in a chain; a pair is one word: row inside the tile, chains, first chain.
//
// Kernel: one workgroup per unit -- a tile, or a piece of one; each wavefront takes an equal stretch of the unit's
// batches, which are in order of their relations, and all of them sum into one partial tile in LDS, in turn.  W is
// read when the relation changes: with batches dealt out one by one it was read for each, 12 KB at 64 -> 32, and
// half the time went there (2 M edges, 65 relations, us per call: 32 -> 32 73 / 63, 64 -> 32 132 / 107, 32 -> 64 107 / 97;
// 342 k edges, 130 relations, hardly two batches of each in a tile: 29.5 / 28.9, 42 / 40, 38 / 37).  Per batch:
//   1. the rows of X of the batch's edges are gathered eight rows (128 bytes each) per load instruction,
//      a column of places per lane group, which weights and adds up its chains in registers and writes
//      each to a row of a tile of LDS;
//   2. lane (i = l % 16, q = l / 16) adds up the chains of pair i, mostly one: inputs 8q .. 8q+7
//      (+32 per further 32 inputs) of S[i, :] = sum over the edges e of pair i of w_e X[src_e, :];
//   3. P = S @ W[rel]^T on v_mfma_f32_16x16x32_bf16, S and W split into three bf16 terms each: a lane's
//      eight inputs are its operand as they stand;
//   4. row i of P is added to row (destination row % 128) of the partial tile with a
//      plain LDS read-modify-write: the pairs of a batch end in different rows or in pieces of
//      one row that this lane order adds one after the other, and the wavefronts take turns (LDS float
//      atomics run at a third of a lane per clock and compute unit on this chip, slower than atomics in
//      memory).
// A batch is a chain of dependent loads (batch record -> edge records -> rows of X and weights), each step
// of it requested one batch ahead of the next.
//
// Bound by the vector unit: 200 instructions per batch, what a unit costs besides included, busy 57 % of the
// kernel's clocks, the matrix cores 13 % (100 k nodes, 65 relations, 2 M edges, 32 -> 32: 117 k batches, 68 us, 75
// per call; 122 before, when each wavefront had a partial tile of 64 rows to itself -- 146 k batches -- and three
// wavefronts per SIMD in the place of four waited on v_mfma_f32_16x16x4_f32, during which the vector unit stands
// still).
// At the end the partial tile is added to the tile's rows of Y, each element once,
// or -- for a unit that is a piece of a tile -- goes to the plan's memory for partial tiles, with
// device-coherent stores.  Such a unit then counts itself in (a counter per cut tile); the one
// that counts last reads the partial tiles of all, coherently, adds them in unit order into Y and
// sets the counter back to zero: no second launch, no fence that writes back or invalidates a
// whole L2, and the same bits whichever unit comes last.
#include "rgms_f32_tiles.h"

#include <algorithm>
#include <type_traits>

#include <hipcub/hipcub.hpp>

namespace stir {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3), aligned(4)));

constexpr int kTileRows = 128;
constexpr int kTileShift = 7;
constexpr int kBatch = 16;    // pairs per matrix-core product
constexpr int kChain = 4;     // edges of a pair that a lane group adds up one after the other
constexpr int kSubBits = 20;  // pieces of one (relation, row) run in the second sort key

struct alignas(16) BatchF32 {
  uint32_t place_begin;  // first place of its edges
  uint32_t counts;       // pairs (at most kBatch) | most chains of a pair << 8 | places (at most EMAX) << 16
  int32_t rel;
  int32_t pad;
};

struct alignas(16) UnitF32 {
  int32_t tile;
  int32_t batch_begin, batch_end;
  int32_t partial;  // -1: the unit is a whole tile and adds to Y; else its place among the partial tiles
  // of a unit that is a piece of a tile: the first partial tile of the tile, its pieces, and its
  // number among the cut tiles (its counter)
  int32_t first_partial, pieces, cut_tile, pad;
};

struct alignas(16) DevBucketF32 {
  const float* A;
  const int32_t* rows;
  const int32_t* cols;
  const int32_t* mids;
  int64_t slot_begin;  // first slot of the bucket in the numbering over all buckets
  int32_t rb, cb;
};

struct CsfArrays {
  const float* A;
  const int32_t* indptr_i;
  const int32_t* indices_i;
  const int32_t* indptr_j;
  const int32_t* indices_j;
  int64_t nnz_i;
};

struct EdgeF32 {  // 12 bytes
  uint32_t src;   // row of X; kUnused: no edge
  uint32_t w_lo;  // address of the edge's weight,
  uint32_t w_hi;  // 48 bits of it | chain << 16: the row of the chain tile the sum goes to after this edge (the
                  // row behind the row of zeros unless the edge ends a chain) | 256 when the edge before it in
                  // the column belongs to the same chain
};
constexpr uint32_t kBehindX = 0xffff0000u;  // X is shorter: no row begins here, and 16 bytes per lane do not wrap
constexpr uint32_t kUnused = (1u << 28) - 1;  // rows of X are fewer: X has less than 2^32 bytes
// pair word: row in the tile | chains << 8 | byte offset of the first chain's row in the chain tile << 16;
// 16 words per batch, for a place without a pair the row behind the tile and the row of zeros
__host__ __device__ constexpr uint32_t chain_row_bytes(int emax) { return emax == 32 ? 36 * 4 : 68 * 4; }

__device__ __forceinline__ int bucket_of(const DevBucketF32* __restrict__ tab, int nb, int64_t q) {
  int lo = 0, hi = nb - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (tab[mid].slot_begin <= q) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// last index i in [0, count] with ptr[i] <= q, minus nothing: the row of position q when ptr is a
// row-pointer array of count rows (count + 1 entries)
__device__ __forceinline__ int64_t row_of(const int32_t* __restrict__ ptr, int64_t count, int64_t q) {
  int64_t lo = 0, hi = count;  // answer in [0, count - 1] for well-formed input
  while (lo < hi) {
    const int64_t mid = (lo + hi + 1) >> 1;
    if ((int64_t)ptr[mid] <= q) lo = mid; else hi = mid - 1;
  }
  return min(lo, count - 1);
}

// destination row, relation, source row and weight address of edge q
template <bool CSF>
__device__ __forceinline__ void edge_of(const DevBucketF32* __restrict__ tab, int nb, const CsfArrays& csf,
                                        int num_rels, int64_t q, int& dest, int& rel, int& src, const float*& w) {
  if constexpr (CSF) {
    const int64_t p = row_of(csf.indptr_j, csf.nnz_i, q);
    dest = csf.indices_i[p];
    rel = (int)row_of(csf.indptr_i, num_rels, p);
    src = csf.indices_j[q];
    w = csf.A + q;
  } else {
    const DevBucketF32 bk = tab[bucket_of(tab, nb, q)];
    const int64_t local = q - bk.slot_begin;
    const int64_t gs = (int64_t)bk.rb * bk.cb;
    const int64_t g = local / gs;
    const int r = (int)((local - g * gs) / bk.cb);
    dest = bk.rows[g * bk.rb + r];
    rel = bk.mids[g];
    src = bk.cols[local];
    w = bk.A + local;
  }
}

template <bool CSF>
__global__ __launch_bounds__(256) void f32_edge_keys_kernel(const DevBucketF32* __restrict__ tab, int nb, CsfArrays csf,
                                                            int64_t slots, int m, int n, int num_rels,
                                                            uint64_t* __restrict__ keys, int32_t* __restrict__ vals,
                                                            int32_t* __restrict__ bad) {
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (q >= slots) return;
  int dest, rel, src;
  const float* w;
  edge_of<CSF>(tab, nb, csf, num_rels, q, dest, rel, src, w);
  if ((unsigned)dest >= (unsigned)m || (unsigned)rel >= (unsigned)num_rels) {
    *bad = 1;
    dest = rel = 0;
  }
  if ((unsigned)src >= (unsigned)n) *bad = 2;
  keys[q] = ((((uint64_t)(dest >> kTileShift)) * num_rels + rel) << kTileShift) | (uint64_t)(dest & (kTileRows - 1));
  vals[q] = (int32_t)q;
}

// Places without an edge: nothing is fetched for them but a weight that exists.
__global__ __launch_bounds__(256) void f32_clear_places_kernel(EdgeF32* __restrict__ places, int64_t count, int emax,
                                                               const float* w, uint32_t* __restrict__ pinfo,
                                                               int64_t words) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const uint64_t at = reinterpret_cast<uintptr_t>(w);
  if (p < count) places[p] = EdgeF32{kUnused, (uint32_t)at, (uint32_t)(at >> 32) | ((uint32_t)(emax + 1) << 16)};
  if (p < words) pinfo[p] = (uint32_t)kTileRows | ((uint32_t)emax * chain_row_bytes(emax) << 16);
}

// Sorted edge i, number t of its pair, goes to the pair's place number t: the last pair whose first
// edge is not behind i.
template <bool CSF>
__global__ __launch_bounds__(256) void f32_edge_records_kernel(const DevBucketF32* __restrict__ tab, int nb,
                                                               CsfArrays csf, int64_t slots, int num_rels, int emax,
                                                               const int32_t* __restrict__ vals,
                                                               const int32_t* __restrict__ pair_first,
                                                               const int32_t* __restrict__ pair_edges,
                                                               const int64_t* __restrict__ pair_place, int64_t pairs,
                                                               EdgeF32* __restrict__ places) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= slots) return;
  int64_t lo = 0, hi = pairs - 1;
  while (lo < hi) {
    const int64_t mid = (lo + hi + 1) >> 1;
    if ((int64_t)pair_first[mid] <= i) lo = mid; else hi = mid - 1;
  }
  const int t = (int)(i - pair_first[lo]);
  int dest, rel, src;
  const float* w;
  edge_of<CSF>(tab, nb, csf, num_rels, vals[i], dest, rel, src, w);
  const uint64_t at = reinterpret_cast<uintptr_t>(w);
  const int64_t place = pair_place[lo];  // place << 8 | first chain
  const bool last = t == pair_edges[lo] - 1 || t % kChain == kChain - 1;
  const uint32_t chain = (last ? (uint32_t)(place & 255) + t / kChain : emax + 1) | (t % kChain ? 256u : 0u);
  places[(place >> 8) + t] = EdgeF32{(uint32_t)src, (uint32_t)at, (uint32_t)(at >> 32) | (chain << 16)};
}

// key2[i] = key[i] << kSubBits | (position of sorted edge i in its run of equal key) / emax; `first`
// holds the first sorted edge of every run.  flags[0] = 3 when a run has more pieces than fit.
__global__ __launch_bounds__(256) void f32_subkeys_kernel(const uint64_t* __restrict__ keys,
                                                          const int32_t* __restrict__ first, int64_t runs, int64_t slots,
                                                          int emax, uint64_t* __restrict__ key2, int32_t* __restrict__ flags) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= slots) return;
  int64_t lo = 0, hi = runs - 1;  // last run whose first edge is not behind i
  while (lo < hi) {
    const int64_t mid = (lo + hi + 1) >> 1;
    if ((int64_t)first[mid] <= i) lo = mid; else hi = mid - 1;
  }
  int64_t piece = (i - first[lo]) / emax;
  if (piece >= (int64_t(1) << kSubBits)) {
    flags[0] = 3;
    piece = (int64_t(1) << kSubBits) - 1;
  }
  key2[i] = (keys[i] << kSubBits) | (uint64_t)piece;
}

// the (tile, relation) part of a pair's second key
__global__ __launch_bounds__(256) void f32_shift_keys_kernel(const uint64_t* __restrict__ in, int64_t count,
                                                             uint64_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < count) out[i] = in[i] >> (kSubBits + kTileShift);
}

// Run i is a (tile, relation) run of run_pairs[i] pairs starting at pair run_first_pair[i]: its
// pairs, in order, fill batches of at most kBatch pairs and emax places.  The places are columns of kChain,
// one column per lane group: a pair of up to kChain edges lies inside a column, a longer one (at most emax
// edges, f32_subkeys_kernel) begins a column and goes on in the next.  Counts the batches (FILL = false) or
// writes them, the pairs' words and first places (FILL = true).
template <bool FILL>
__global__ __launch_bounds__(256) void f32_batches_kernel(const uint64_t* __restrict__ run_keys,
                                                          const int32_t* __restrict__ run_pairs,
                                                          const int32_t* __restrict__ run_first_pair,
                                                          const int32_t* __restrict__ run_first_batch, int64_t runs,
                                                          int num_rels, int emax, const uint64_t* __restrict__ pair_keys,
                                                          const int32_t* __restrict__ pair_edges,
                                                          int32_t* __restrict__ run_batches,
                                                          int64_t* __restrict__ run_places,
                                                          const int64_t* __restrict__ run_first_place,
                                                          BatchF32* __restrict__ batches, uint32_t* __restrict__ pinfo,
                                                          int64_t* __restrict__ pair_place) {
  const int lane = threadIdx.x & 63;
  const int64_t i = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (i >= runs) return;
  const int np = run_pairs[i], fp = run_first_pair[i];
  const int rel = (int)(run_keys[i] % (uint64_t)num_rels);
  int64_t base = FILL ? run_first_place[i] : 0;  // first place of the batch in hand
  int64_t number = FILL ? run_first_batch[i] : 0;
  int nb = 0, pairs = 0, place = 0, chains = 0, most = 0;
  auto close = [&]() {
    if (FILL && lane == 0)
      batches[number] = BatchF32{(uint32_t)base, (uint32_t)pairs | ((uint32_t)most << 8) | ((uint32_t)place << 16), rel, 0};
    base += place, ++number, ++nb;
    pairs = place = chains = most = 0;
  };
  // 64 pairs at a time, one per lane: the wavefront goes through them together (one thread per run would wait
  // for memory at every pair), lane k keeps what came out for pair k
  for (int j0 = 0; j0 < np; j0 += 64) {
    const int count = min(64, np - j0);
    const int mine = lane < count ? min(pair_edges[fp + j0 + lane], emax) : 0;
    int my_pair = 0, my_place = 0, my_chain = 0;
    int64_t my_number = 0, my_base = 0;
    for (int k = 0; k < count; ++k) {
      const int c = __builtin_amdgcn_readlane(mine, k);
      int at = place;
      if (at % kChain + c > kChain) at = (at + kChain - 1) / kChain * kChain;
      if (pairs > 0 && (pairs == kBatch || at + c > emax)) close(), at = 0;
      if (FILL && lane == k) my_pair = pairs, my_place = at, my_chain = chains, my_number = number, my_base = base;
      const int own = (c + kChain - 1) / kChain;
      place = at + c, chains += own, most = max(most, own), ++pairs;
    }
    if (FILL && lane < count) {
      const int j = fp + j0 + lane;
      const uint32_t dl = (uint32_t)((pair_keys[j] >> kSubBits) & (kTileRows - 1));
      pinfo[my_number * kBatch + my_pair] =
          dl | ((uint32_t)((mine + kChain - 1) / kChain) << 8) | ((uint32_t)my_chain * chain_row_bytes(emax) << 16);
      pair_place[j] = ((my_base + my_place) << 8) | my_chain;
    }
  }
  close();
  if (!FILL && lane == 0) run_batches[i] = nb, run_places[i] = base;
}

// begin[t] = first batch of tile t (t = tiles gives the batch count): the first run whose key
// (tile * num_rels + relation) is not below t * num_rels
__global__ __launch_bounds__(256) void f32_tile_batches_kernel(const uint64_t* __restrict__ run_keys,
                                                               const int32_t* __restrict__ run_first_batch, int64_t runs,
                                                               int64_t total_batches, int64_t tiles, int num_rels,
                                                               int64_t* __restrict__ begin) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t > tiles) return;
  const uint64_t target = (uint64_t)t * num_rels;
  int64_t lo = 0, hi = runs;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (run_keys[mid] < target) lo = mid + 1; else hi = mid;
  }
  begin[t] = lo < runs ? run_first_batch[lo] : total_batches;
}

typedef __attribute__((address_space(1))) const float GlobalF32;  // a global-memory load, not a flat one

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// Eight floats as sums of three bf16 each: v = t[0] + t[1] + t[2], exactly as long as nothing underflows or
// overflows (each term is what the ones before it leave, rounded to nearest: 8 + 8 + 8 bits of a 24-bit significand).
// So that nothing underflows, whatever fp32 numbers come in, both factors of the product are taken times kScale: the
// last bit of the smallest subnormal number is a normal bf16 then, and the sums come out times kScale^2.  What
// overflows on the way (sums and weights from 2^104 on, products from 2^80, infinities) leaves an infinity or NaN in
// the partial tile, and the unit is done again without terms (exact_unit).
constexpr float kScale = 0x1p24f;
__device__ __forceinline__ void split3(const float (&v)[8], bf16x8 (&t)[3]) {
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    f32x2 r = {v[j], v[j + 1]};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const bf16x2 h = __builtin_convertvector(r, bf16x2);
      t[k][j] = h[0], t[k][j + 1] = h[1];
      if (k < 2) {
        const uint32_t both = __builtin_bit_cast(uint32_t, h);
        r[0] -= __uint_as_float(both << 16), r[1] -= __uint_as_float(both & 0xffff0000u);
      }
    }
  }
}

// W[rel][16 nt + i][32 s + 8 q .. + 7] -> Wp[((rel * NT + nt) * KS + s) * 3 + term][lane (i, q)]: the B
// operands of a batch, split into three bf16 terms, as 16-byte words in lane order, so that the kernel's loads
// of W are contiguous (a lane of the multiply owns one row of W per output tile: read in place, the 64
// lanes of a load would touch 16 different lines four times over).  Zero beyond feat_in and
// feat_out.  One thread per lane of a fragment.
__global__ __launch_bounds__(256) void f32_pack_w_kernel(const float* __restrict__ W, bf16x8* __restrict__ Wp,
                                                         int64_t fragments, int nt_count, int ks_count, int fin, int fout) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= fragments) return;
  const int lane = (int)(t & 63), i = lane & 15, q = lane >> 4;
  const int64_t f = t >> 6;
  const int s = (int)(f % ks_count);
  const int nt = (int)(f / ks_count % nt_count);
  const int64_t rel = f / ks_count / nt_count;
  const int out = 16 * nt + i;
  float v[8];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int k = 32 * s + 8 * q + 4 * c;  // fin is a multiple of 4
    float4 w = make_float4(0.f, 0.f, 0.f, 0.f);
    if (out < fout && k < fin) w = *reinterpret_cast<const float4*>(W + (rel * fout + out) * fin + k);
    v[4 * c] = kScale * w.x, v[4 * c + 1] = kScale * w.y, v[4 * c + 2] = kScale * w.z, v[4 * c + 3] = kScale * w.w;
  }
  bf16x8 term[3];
  split3(v, term);
#pragma unroll
  for (int k = 0; k < 3; ++k) Wp[(f * 3 + k) * 64 + lane] = term[k];
}

// The value of lane K of the lane's own four, which the compiler makes an operand of the instruction that takes it.
// Broadcasts over eight lanes, as two instructions of their own, were a sixth of the loop's vector instructions
// (2 M edges, 65 relations, us per call: 32 -> 8 52 / 50, 32 -> 32 63 / 61, 64 -> 32 107 / 104, 32 -> 64 97 / 95).
template <int K>
__device__ __forceinline__ uint32_t of_four(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, K * 0x55, 0xf, 0xf, true);
}

template <class F>
__device__ __forceinline__ void static_for_chain(F f) {
  f(std::integral_constant<int, 0>());
  f(std::integral_constant<int, 1>());
  f(std::integral_constant<int, 2>());
  f(std::integral_constant<int, 3>());
}

// KS: feat_in <= 32 * KS; NT: feat_out <= 16 * NT.
//
// Two lane layouts.  Gathering: a row of X (or its first 32 KS floats) is spread over CPR = 8 KS
// neighbouring lanes, four floats each, so that a load instruction reads 64 / CPR whole rows and
// the texture addresser sees whole lines per quad of lanes; the four load instructions of a batch
// cover its EMAX = 32 / KS edges in order.  Multiplying: lane (i = l % 16, q = l / 16) holds
// inputs 8q .. 8q+7 of pair i.  The rows change layout through an EMAX x 32 KS tile of LDS per
// wavefront: written once per edge, read once per edge by the lanes of the edge's pair.
//
// The loads of the batch loop are unconditional, so that the loop body has no branch around a load:
// edge records are clamped to ones that exist, and a row of X that no edge asks for is read behind the
// end of the buffer, which returns zeros and fetches nothing.  Offsets into X and the edge records are
// 32-bit byte offsets (the launch checks that they fit).
template <int KS, int NT>
struct TileShape {
  // as many wavefronts as registers and LDS allow per compute unit: 16, and 8 above 32 inputs and outputs (4 workgroups,
  // 2 above 32 outputs).  Twelve there left ten registers of W in memory, and waiting for them was waiting for
  // everything in flight (2 M edges, 65 relations, 64 -> 64: 291 / 166 us; 342 k edges, 8 relations: 63 / 43).
  static constexpr int kWaves = KS == 1 && NT == 4 ? 8 : 4;
  static constexpr int kPerSimd = KS == 2 && NT == 4 ? 2 : 4;
};

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef __attribute__((address_space(3))) float LdsF32;
typedef __attribute__((address_space(3))) int LdsInt;

// All of a unit once more into its partial tile, with fp32 products.  A function of its own: in the kernel it took
// registers from the loop, as a branch inside or behind it (110 k nodes, 130 relations, 2 M edges, 64 -> 64: 333 us,
// 422 and 458 with it).  A unit that comes here takes about six times as long.
template <int KS, int NT>
__device__ __attribute__((noinline)) void exact_unit(int b_begin, int b_end, int fin, int fout, const BatchF32* batches,
                                                     const uint32_t* pinfo, const EdgeF32* edges, const float* W,
                                                     const float* X, LdsF32* yt, LdsF32* et, LdsInt* turn) {
  constexpr int WAVES = TileShape<KS, NT>::kWaves, THREADS = 64 * WAVES, FO = 16 * NT, CPR = 8 * KS, EMAX = 32 / KS;
  constexpr int SS = 32 * KS + 4;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, q = lane >> 4, g = lane / CPR, gc = lane % CPR;
  for (int e = tid; e < kTileRows * FO; e += THREADS) yt[e] = 0.f;
  if (tid == 0) *turn = b_begin;
  __syncthreads();
#pragma unroll 1
  for (int b = b_begin + wave; b < b_end; b += WAVES) {
    const BatchF32 bt = batches[b];
    const int places = (int)((bt.counts >> 16) & 255u);
    // the places of a lane group's column, one after the other
    f32x4 run = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int k = 0; k < kChain; ++k) {
      const int place = g * kChain + k;
      uint32_t chain = (uint32_t)(EMAX + 1);
      f32x4 x = {0.f, 0.f, 0.f, 0.f};
      float w = 0.f;
      if (place < places) {
        const EdgeF32 rec = edges[(int64_t)bt.place_begin + place];
        chain = rec.w_hi >> 16;
        if (rec.src != kUnused) {
          w = *reinterpret_cast<GlobalF32*>((uintptr_t)rec.w_lo | ((uintptr_t)(rec.w_hi & 0xffffu) << 32));
          if (4 * gc < fin) x = *reinterpret_cast<const f32x4u*>(X + (int64_t)rec.src * fin + 4 * gc);
        }
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) run[c] = k == 0 ? w * x[c] : fmaf(w, x[c], chain >= 256 ? run[c] : 0.f);
      LdsF32* row = et + (chain & 255) * SS + 4 * gc;
#pragma unroll
      for (int c = 0; c < 4; ++c) row[c] = run[c];
    }
    const uint32_t pair = pinfo[(int64_t)b * kBatch + i];
    const LdsF32* first = et + 8 * q + (pair >> 16) / 4;
    const int chains = (int)((pair >> 8) & 255u);
    const float* wrel = W + (int64_t)bt.rel * fout * fin;
    f32x4 acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int j = 0; j < 8 * KS; ++j) {  // product number j of four inputs takes input 8 q + j of each lane
      const int k = 32 * (j >> 3) + 8 * q + (j & 7), at = 32 * (j >> 3) + (j & 7);
      float x = first[at];
      for (int t = 1; t < chains; ++t) x += first[t * SS + at];
      x = k < fin ? x : 0.f;  // what lies beyond feat_in is no input
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int out = 16 * nt + i;
        acc[nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, out < fout && k < fin ? wrel[out * fin + k] : 0.f, acc[nt], 0, 0, 0);
      }
    }
    while (__hip_atomic_load(turn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != b) __builtin_amdgcn_s_sleep(1);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      LdsF32* row = yt + (pinfo[(int64_t)b * kBatch + 4 * q + v] & 255u) * FO + NT * i;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) row[nt] += acc[nt][v];
    }
    asm volatile("" ::: "memory");
    __hip_atomic_store(turn, b + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  __syncthreads();
}

template <int KS, int NT>
__global__ __launch_bounds__((64 * TileShape<KS, NT>::kWaves))
__attribute__((amdgpu_waves_per_eu(TileShape<KS, NT>::kPerSimd, TileShape<KS, NT>::kPerSimd)))
void rgms_f32_tile_kernel(int m, int fin, int fout, int total_batches, uint32_t x_bytes,
                          const UnitF32* __restrict__ units, const BatchF32* __restrict__ batches,
                          const uint32_t* __restrict__ pinfo, const EdgeF32* __restrict__ edges,
                          const bf16x8* __restrict__ Wp, const float* __restrict__ W,
                          const float* __restrict__ X, float* __restrict__ Y, float* partials, uint32_t* arrived) {
  constexpr int WAVES = TileShape<KS, NT>::kWaves;
  constexpr int THREADS = 64 * WAVES;
  constexpr int FO = 16 * NT;      // floats per row of the partial tile
  constexpr int CPR = 8 * KS;      // lanes (16-byte chunks) per gathered row
  constexpr int RPI = 64 / CPR;    // rows per load instruction
  constexpr int EMAX = 32 / KS;    // places per batch
  constexpr int SS = 32 * KS + 4;  // floats per row of the chain tile: 16 lanes reading 32 bytes each hit 64 banks
  static_assert(EMAX == RPI * kChain, "a lane group has a column of places");
  static_assert(NT == 1 || NT == 2 || NT == 4, "a lane's outputs are one word of the partial tile");
  __shared__ __attribute__((aligned(16))) float yt[(kTileRows + 1) * FO];
  // a row per chain; row EMAX stays zero, row EMAX + 1 takes what ends no chain
  __shared__ __attribute__((aligned(16))) float etile[WAVES][(EMAX + 2) * SS - 4];
  __shared__ int turn, last_of_tile;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, q = lane >> 4;      // multiplying
  const int gc = lane % CPR;                   // gathering
  const UnitF32 u = units[blockIdx.x];
  float* et = etile[wave];
  for (int e = tid; e < kTileRows * FO; e += THREADS) yt[e] = 0.f;
  for (int e = lane; e < SS; e += 64) et[EMAX * SS + e] = 0.f;
  if (tid == 0) turn = 0;
  // a stretch of batches for each wavefront, its k-th one in turn k * WAVES + wave
  const int fewest = (u.batch_end - u.batch_begin) / WAVES, more = (u.batch_end - u.batch_begin) % WAVES;
  int b = u.batch_begin + wave * fewest + min(wave, more);
  const int b_end = b + fewest + (wave < more ? 1 : 0);
  int my_turn = wave;
  const bool chunk_live = 4 * gc < fin;  // fin is a multiple of 4: chunks are whole
  const uint32_t row_bytes = 4u * (uint32_t)fin;
  const __amdgpu_buffer_rsrc_t Xr =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(X), 0, x_bytes, 0x00027000);

  struct Batch {  // the same in every lane
    uint32_t place_begin;
    int npairs, most, places, rel;
  };
  // A vector load although every lane wants the same 16 bytes: a scalar load in flight makes every wait for
  // LDS a wait for memory (both count in lgkmcnt, and scalar loads return in any order).
  int no_scalar = 0;
  asm("" : "+v"(no_scalar));
  auto raw_batch = [&](int bi) { return batches[min(bi, total_batches - 1) + no_scalar]; };
  auto scalars = [&](const BatchF32& t, int bi) {  // a batch beyond the unit's last one: no pairs
    Batch r;
    const uint32_t c = bi < b_end ? __builtin_amdgcn_readfirstlane(t.counts) : 0u;
    r.place_begin = __builtin_amdgcn_readfirstlane(t.place_begin);
    r.npairs = (int)(c & 255u), r.most = (int)((c >> 8) & 255u), r.places = (int)((c >> 16) & 255u);
    r.rel = __builtin_amdgcn_readfirstlane(t.rel);
    return r;
  };
  // Each four lanes hold the four places of their lane group's column, and a lane gets at them by DPP.
  const int my_place = lane / CPR * kChain + (lane & (kChain - 1));
  auto load_record = [&](const Batch& bt) {
    return *reinterpret_cast<const u32x3*>(edges + (int64_t)bt.place_begin + min(my_place, max(bt.places - 1, 0)));
  };
  struct Rows {
    f32x4 x[kChain];  // place k of the lane group's column
    float w;          // of the lane's own place
    uint32_t chain;   // of the lane's own place
  };
  const uint32_t no_chunk = chunk_live ? 0u : 0xfffffff0u;
  auto load_rows = [&](const u32x3& rec, int places) {  // rec: {src, w_lo, w_hi} of EdgeF32
    Rows r;
    r.w = *reinterpret_cast<GlobalF32*>((uintptr_t)rec.y | ((uintptr_t)(rec.z & 0xffffu) << 32));
    const bool live = my_place < places;
    r.chain = live ? rec.z >> 16 : (uint32_t)(EMAX + 1);
    // no edge or no such inputs: behind the end of X, which reads as zeros
    const uint32_t off = live && rec.x != kUnused ? rec.x * row_bytes : kBehindX;
    static_for_chain([&](auto K) {
      const uint32_t at = of_four<decltype(K)::value>(off) + 16u * gc;
      r.x[K] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(Xr, at | no_chunk, 0, 0));
    });
    return r;
  };
  // lane (i, q): the word of pair i, and, i < 4, the word of pair 4 q + i
  auto load_pair = [&](int bi) { return pinfo[(int64_t)min(bi, total_batches - 1) * kBatch + i]; };
  auto load_row = [&](int bi) { return pinfo[(int64_t)min(bi, total_batches - 1) * kBatch + (4 * q + (i & 3))]; };
  bf16x8 wq[NT][KS][3];  // W operands of the batch, three terms each
  auto load_w = [&](int rel) {
    const bf16x8* wrel = Wp + (int64_t)rel * (NT * KS * 3 * 64) + lane;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int k = 0; k < 3; ++k) wq[nt][s][k] = wrel[((nt * KS + s) * 3 + k) * 64];
  };

  // The pipeline: at batch j the record of batch j + 3 is requested, the edge records of j + 2, the rows of
  // X, weights, pair words and W operands of j + 1.  One set of registers: what a batch holds is used up
  // before the next one's is requested into it, and the other wavefronts of the SIMD cover the rest.  All but the
  // pair words behind the products, where fewer registers are in use, and W last, so that only what needs W waits
  // for it (requests before the products: 3 to 5 % slower above 32 outputs, else the same).
  Batch bt0 = scalars(raw_batch(b), b), bt1 = scalars(raw_batch(b + 1), b + 1);
  BatchF32 raw = raw_batch(b + 2);
  Rows rw = load_rows(load_record(bt0), bt0.places);
  u32x3 rec = load_record(bt1);
  uint32_t pw = load_pair(b), pr = load_row(b);
  load_w(bt0.rel);
  __syncthreads();

  while (bt0.npairs > 0) {  // the same for every lane
    // 1. the chains of this batch: a lane group adds up its column of weighted rows, and writes a row of the
    // chain tile wherever a chain ends
    f32x4 run = {0.f, 0.f, 0.f, 0.f};
    const uint32_t own = __float_as_uint(kScale * rw.w);
    const uint32_t keep = (uint32_t)__builtin_amdgcn_sbfe((int)rw.chain, 8, 1);  // all bits: the sum goes on
    const uint32_t to = 4u * __umul24(rw.chain & 255, SS);
    static_for_chain([&](auto K) {
      constexpr int k = decltype(K)::value;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float w = __uint_as_float(of_four<k>(own));
        if constexpr (k == 0)
          run[c] = w * rw.x[K][c];
        else
          run[c] = fmaf(w, rw.x[K][c], __uint_as_float(of_four<k>(keep) & __float_as_uint(run[c])));
      }
      *reinterpret_cast<f32x4*>(reinterpret_cast<char*>(et + 4 * gc) + of_four<k>(to)) = run;
    });
    // 2. the sums of the pairs, multiplying layout: lane (i, q) adds the chains of pair i, mostly one; a lane
    // whose pair has fewer than the batch's longest reads the tile's row of zeros meanwhile
    const int my_count = (int)((pw >> 8) & 255u);
    const uint32_t next_pw = load_pair(b + 1), next_pr = load_row(b + 1);
    const char* first = reinterpret_cast<const char*>(et + 8 * q) + (pw >> 16);
    float sum[KS][8];
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const float4 v = reinterpret_cast<const float4*>(first)[8 * s + c];
        sum[s][4 * c] = v.x, sum[s][4 * c + 1] = v.y, sum[s][4 * c + 2] = v.z, sum[s][4 * c + 3] = v.w;
      }
#pragma unroll 1
    for (int t = 1; t < bt0.most; ++t) {  // the same for every lane
      const char* row = t < my_count ? first + t * (4 * SS) : reinterpret_cast<const char*>(et + EMAX * SS + 8 * q);
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const float4 v = reinterpret_cast<const float4*>(row)[8 * s + c];
          sum[s][4 * c] += v.x, sum[s][4 * c + 1] += v.y, sum[s][4 * c + 2] += v.z, sum[s][4 * c + 3] += v.w;
        }
    }
    // 3. times W[rel]^T, on the bf16 matrix cores: both factors are three terms, and of the nine products the
    // six above 2^-24 of the whole are added, small ones first.  v_mfma_f32_16x16x4_f32 would keep the vector
    // unit waiting for its 32 clocks (measured: the two add up, a bf16 product of twice the size costs it 9),
    // and this loop needs the vector unit most of the time.
    f32x4 acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      bf16x8 a[3];
      split3(sum[s], a);
      constexpr int kTerms[6][2] = {{0, 2}, {2, 0}, {1, 1}, {0, 1}, {1, 0}, {0, 0}};
#pragma unroll
      for (int p = 0; p < 6; ++p)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[kTerms[p][0]], wq[nt][s][kTerms[p][1]], acc[nt], 0, 0, 0);
    }
    // requests for the batches to come
    rw = load_rows(rec, bt1.places);
    const Batch bt2 = scalars(raw, b + 2);
    rec = load_record(bt2);
    raw = raw_batch(b + 3);
    if (bt1.rel != bt0.rel) load_w(bt1.rel);
    // 4. acc[nt][v]: pair 4 q + v of the batch, output 16 nt + i, which lives at float NT i + nt of
    // its row of the partial tile: a lane's NT outputs are neighbours, one read and one write.
    // The pairs of a batch end in different rows (a row cut into pieces has at most its last,
    // shorter piece in a batch with other pairs: a full piece fills a batch), so no two lanes
    // update the same float; the wavefronts take turns.  (LDS instructions of a wavefront execute in
    // order: the turn goes on after the tile is written.)
    while (__hip_atomic_load(&turn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != my_turn) __builtin_amdgcn_s_sleep(1);
    asm volatile("" ::: "memory");
    struct alignas(4 * NT) Outs {
      float v[NT];
    };
    Outs *at[4], sums[4];
    const uint32_t row = 4 * FO * (pr & 255);
    static_for_chain([&](auto V) {
      at[V] = reinterpret_cast<Outs*>(reinterpret_cast<char*>(yt + NT * i) + of_four<decltype(V)::value>(row));
    });
#pragma unroll
    for (int v = 0; v < 4; ++v) sums[v] = *at[v];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) sums[v].v[nt] += acc[nt][v];
      *at[v] = sums[v];
    }
    asm volatile("" ::: "memory");
    __hip_atomic_store(&turn, my_turn + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    pw = next_pw, pr = next_pr;
    ++b, my_turn += WAVES;
    bt0 = bt1, bt1 = bt2;
  }

  __syncthreads();
  // a unit in which something overflowed is done again, with fp32 products
  float unscale = 1.f / (kScale * kScale), all_finite = 0.f;  // all_finite: or NaN
  for (int e = tid; e < kTileRows * FO / 4; e += THREADS) {
    const float4 v = reinterpret_cast<const float4*>(yt)[e];
    all_finite = fmaf(v.x, 0.f, all_finite), all_finite = fmaf(v.y, 0.f, all_finite);
    all_finite = fmaf(v.z, 0.f, all_finite), all_finite = fmaf(v.w, 0.f, all_finite);
  }
  if (__syncthreads_or(!(all_finite == 0.f))) {
    exact_unit<KS, NT>(u.batch_begin, u.batch_end, fin, fout, batches, pinfo, edges, W, X, (LdsF32*)yt, (LdsF32*)et, (LdsInt*)&turn);
    unscale = 1.f;
  }
  // The tile's rows of Y are one stretch of memory.  A thread requests all it is about to add to before it
  // waits for any of it: one element at a time this end of a unit took 13 round trips to memory.
  const int64_t row0 = (int64_t)u.tile * kTileRows;
  const int64_t stride = (int64_t)kTileRows * fout;
  const int count = (int)min((int64_t)kTileRows, m - row0) * fout;
  float* Yt = Y + row0 * fout;
  constexpr int AHEAD = 8;
  const uint32_t inverse = (uint32_t)((0x100000000ull + fout - 1) / fout);  // exact quotients for these e
  auto sum_at = [&](int e) {
    const int r = fout > 1 ? (int)__umulhi((uint32_t)e, inverse) : e, c = e - r * fout;
    return unscale * yt[r * FO + NT * (c & 15) + (c >> 4)];
  };
  if (u.partial < 0) {
    for (int e0 = tid; e0 < count; e0 += AHEAD * THREADS) {
      float old[AHEAD];
#pragma unroll
      for (int k = 0; k < AHEAD; ++k) old[k] = Yt[min(e0 + k * THREADS, count - 1)];
#pragma unroll
      for (int k = 0; k < AHEAD; ++k)
        if (e0 + k * THREADS < count) Yt[e0 + k * THREADS] = old[k] + sum_at(e0 + k * THREADS);
    }
    return;
  }
  for (int e = tid; e < count; e += THREADS)
    __hip_atomic_store(partials + u.partial * stride + e, sum_at(e), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // A piece of a tile.  Every wavefront waits until its stores have arrived, then one thread
  // counts the unit in; the unit that counts last finds the partial tiles of all the others in
  // memory (stores and loads of partial tiles pass the L2 of their XCD).
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    uint32_t* counter = arrived + u.cut_tile;
    const uint32_t before = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const bool last = before + 1 == (uint32_t)u.pieces;
    if (last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
    last_of_tile = last;
  }
  __syncthreads();
  if (!last_of_tile) return;
  const float* all = partials + u.first_partial * stride;
  for (int e0 = tid; e0 < count; e0 += AHEAD * THREADS) {
    float old[AHEAD], sum[AHEAD];
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) old[k] = Yt[min(e0 + k * THREADS, count - 1)], sum[k] = 0.f;
    for (int p0 = 0; p0 < u.pieces; p0 += 4) {  // the pieces add up in their order
      float v[4][AHEAD];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int k = 0; k < AHEAD; ++k)
          v[j][k] = __hip_atomic_load(all + min(p0 + j, u.pieces - 1) * stride + min(e0 + k * THREADS, count - 1),
                                      __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) sum[k] += p0 + j < u.pieces ? v[j][k] : 0.f;
    }
#pragma unroll
    for (int k = 0; k < AHEAD; ++k)
      if (e0 + k * THREADS < count) Yt[e0 + k * THREADS] = old[k] + sum[k];
  }
}

// Device memory for the duration of an index build, in one piece: an allocation and its release take
// 50 to 150 us each, and 20 of them took longer than the build itself (first call of a plan with 2 M edges: 3.8 -> 1.4 ms).
struct Scratch {
  char* base = nullptr;
  size_t size = 0, used = 0;
  ~Scratch() {
    if (base) (void)hipFree(base);
  }
  static size_t rounded(size_t bytes) { return (std::max<size_t>(bytes, 1) + 255) / 256 * 256; }
  int reserve(size_t bytes) {
    STIR_HIP(hipMalloc(reinterpret_cast<void**>(&base), bytes));
    size = bytes;
    return 0;
  }
  template <typename T>
  int get(T** out, size_t count) {
    const size_t bytes = rounded(count * sizeof(T));
    STIR_REQUIRE(used + bytes <= size, "rgms_f32: scratch of the index build is too small");
    *out = reinterpret_cast<T*>(base + used);
    used += bytes;
    return 0;
  }
};

}  // namespace

namespace {
int build_index(F32TileIndex& idx, const F32Source& src, int32_t m, int32_t n, int32_t num_rels, int32_t emax,
                hipStream_t stream);
}

bool f32_tiles_serves(int32_t feat_in, int32_t feat_out) {
  return feat_in > 0 && feat_in % 4 == 0 && feat_in <= 64 && feat_out > 0 && feat_out <= 64;
}

bool f32_tiles_fits(int32_t n, int32_t feat_in, int64_t edges) {
  return (int64_t)n * feat_in * 4 <= (int64_t)kBehindX && edges < (int64_t(1) << 31);
}

void f32_tiles_free(F32TileIndex& idx) {
  if (idx.d_batches) (void)hipFree(idx.d_batches);
  for (F32Units& u : idx.units) {
    if (u.d_units) (void)hipFree(u.d_units);
  }
  idx = F32TileIndex();
}

int f32_tiles_prepare(F32TileIndex& idx, const F32Source& src, int32_t m, int32_t n, int32_t num_rels,
                      int32_t feat_in, hipStream_t stream) {
  const int32_t emax = feat_in <= 32 ? 32 : 16;
  if (idx.m == m && idx.n == n && idx.num_rels == num_rels && idx.emax == emax) return 0;
  f32_tiles_free(idx);
  F32TileIndex built;
  const int rc = build_index(built, src, m, n, num_rels, emax, stream);
  if (rc != 0) {
    f32_tiles_free(built);  // nothing half-made stays behind
    return rc;
  }
  idx = built;
  return 0;
}

namespace {
// The units of a launch: whole tiles, or pieces of tiles of at most `cap` batches, longest first.  As many as
// run at the same time: 4 workgroups per compute unit, 2 when feat_out is above 32 (wide), so that each takes
// an equal part of the whole.  Fewer when there are few tiles -- most of them would be cut, and the last
// piece of a tile adds up what all of them wrote (24 k nodes, 65 relations, 299 k edges: 26.8 us with 768
// units, 30.0 with 1024, 36.8 uncut) -- and no pieces so short that filling the pipeline and the partial
// tile cost more than they bring.  Wide launches with many tiles: two rounds (110 k nodes, 130
// relations, 2 M edges, 64 -> 64: 334 us with 1024 units, 371 with 860 whole tiles).
int make_units(F32Units& out, const std::vector<int64_t>& tile_begin, bool wide, int32_t feat_out, size_t wpack_bytes,
               hipStream_t stream) {
  const int64_t tiles = (int64_t)tile_begin.size() - 1, cus = compute_units();
  STIR_REQUIRE(cus > 0, "rgms_f32: no device");
  const int64_t target = tiles > 2 * cus ? 4 * cus : (wide ? 2 : 3) * cus;
  auto count_with = [&](int64_t cap) {
    int64_t count = 0;
    for (int64_t t = 0; t < tiles; ++t) count += ceil_div(tile_begin[(size_t)t + 1] - tile_begin[(size_t)t], cap);
    return count;
  };
  int64_t cap = wide ? 48 : 24, top = std::max(tile_begin[(size_t)tiles], cap);
  while (cap < top) {  // the shortest pieces that are not too many
    const int64_t mid = (cap + top) / 2;
    if (count_with(mid) <= target) top = mid; else cap = mid + 1;
  }
  std::vector<UnitF32> units;
  int64_t partial_tiles = 0, cut_tiles = 0;
  for (int64_t t = 0; t < tiles; ++t) {
    const int64_t lo = tile_begin[(size_t)t], hi = tile_begin[(size_t)t + 1];
    if (hi <= lo) continue;
    if (hi - lo <= cap) {
      units.push_back(UnitF32{(int32_t)t, (int32_t)lo, (int32_t)hi, -1, 0, 0, 0, 0});
      continue;
    }
    const int64_t pieces = ceil_div(hi - lo, cap);
    STIR_REQUIRE(partial_tiles + pieces < (int64_t(1) << 31), "rgms_f32: too many partial tiles");
    for (int64_t p = 0; p < pieces; ++p)
      units.push_back(UnitF32{(int32_t)t, (int32_t)(lo + (hi - lo) * p / pieces), (int32_t)(lo + (hi - lo) * (p + 1) / pieces),
                              (int32_t)(partial_tiles + p), (int32_t)partial_tiles, (int32_t)pieces,
                              (int32_t)cut_tiles, 0});
    partial_tiles += pieces, ++cut_tiles;
  }
  std::stable_sort(units.begin(), units.end(), [](const UnitF32& a, const UnitF32& b) {
    return a.batch_end - a.batch_begin > b.batch_end - b.batch_begin;
  });
  out.count = (int64_t)units.size(), out.partial_tiles = partial_tiles;
  // one allocation: the units, the counters of the cut tiles (zero between launches), W in operand order, the
  // partial tiles
  const size_t unit_bytes = sizeof(UnitF32) * units.size();
  std::vector<char> image(Scratch::rounded(unit_bytes + sizeof(uint32_t) * (size_t)cut_tiles));
  std::copy_n(reinterpret_cast<const char*>(units.data()), unit_bytes, image.data());
  const size_t partial_bytes = sizeof(float) * (size_t)partial_tiles * kTileRows * (size_t)feat_out;
  STIR_HIP(hipMalloc(&out.d_units, image.size() + Scratch::rounded(wpack_bytes) + partial_bytes));
  char* base = static_cast<char*>(out.d_units);
  out.d_arrived = base + unit_bytes;
  out.d_wpack = base + image.size();
  out.d_partials = base + image.size() + Scratch::rounded(wpack_bytes);
  out.wpack_bytes = wpack_bytes, out.feat_out = feat_out;
  STIR_HIP(hipMemcpyAsync(out.d_units, image.data(), image.size(), hipMemcpyHostToDevice, stream));
  STIR_HIP(hipStreamSynchronize(stream));  // there before a launch on any stream
  return 0;
}

int build_index(F32TileIndex& idx, const F32Source& src, int32_t m, int32_t n, int32_t num_rels, int32_t emax,
                hipStream_t stream) {
  STIR_REQUIRE(m > 0 && n > 0 && num_rels > 0, "rgms_f32: m, n and num_rels must be positive");
  // edges and their numbering
  std::vector<DevBucketF32> tab;
  int64_t slots = 0;
  if (src.csf) {
    slots = src.nnz_j;
  } else {
    for (const F32Bucket& b : src.buckets) {
      if (b.groups == 0) continue;
      tab.push_back(DevBucketF32{b.A, b.rows, b.cols, b.mids, slots, b.rb, b.cb});
      slots += b.groups * b.rb * b.cb;
    }
  }
  STIR_REQUIRE(slots < (int64_t(1) << 31), "rgms_f32: %lld slots exceed 32-bit edge numbers", (long long)slots);
  const int64_t tiles = ceil_div(m, kTileRows);
  STIR_REQUIRE(tiles < (int64_t(1) << 31), "rgms_f32: too many tiles");
  int key_bits = kTileShift;
  while (key_bits < 64 && ((uint64_t)tiles * num_rels) >> (key_bits - kTileShift)) ++key_bits;
  STIR_REQUIRE(key_bits + kSubBits <= 64, "rgms_f32: sort keys exceed 64 bits");
  idx.m = m, idx.n = n, idx.num_rels = num_rels, idx.emax = emax;
  idx.edges = slots, idx.tiles = tiles;
  if (slots == 0) return 0;  // no units: the launch returns at once
  size_t sort_bytes = 0, rle_bytes = 0, scan_bytes = 0;
  STIR_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, (uint64_t*)nullptr, (uint64_t*)nullptr,
                                              (int32_t*)nullptr, (int32_t*)nullptr, (int)slots, 0,
                                              key_bits, stream));
  STIR_HIP(hipcub::DeviceRunLengthEncode::Encode(nullptr, rle_bytes, (uint64_t*)nullptr, (uint64_t*)nullptr, (int32_t*)nullptr,
                                                 (int32_t*)nullptr, (int)slots,
                                                 stream));
  STIR_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, scan_bytes, (int32_t*)nullptr, (int32_t*)nullptr, (int)slots + 1, stream));
  size_t scan3_bytes = 0;
  STIR_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, scan3_bytes, (int64_t*)nullptr, (int64_t*)nullptr, (int)slots + 1, stream));
  const size_t cub_bytes = std::max(std::max(sort_bytes, rle_bytes), std::max(scan_bytes, scan3_bytes));
  const size_t rows = (size_t)slots + 1;
  Scratch tmp;
  if (tmp.reserve(Scratch::rounded(sizeof(DevBucketF32) * tab.size()) + 6 * Scratch::rounded(8 * rows) +
                  7 * Scratch::rounded(4 * rows) + Scratch::rounded(8) + Scratch::rounded(8 * (size_t)(tiles + 1)) +
                  Scratch::rounded(cub_bytes)))
    return -1;
  char* cub_tmp = nullptr;
  if (tmp.get(&cub_tmp, cub_bytes)) return -1;
  DevBucketF32* d_tab = nullptr;
  if (!tab.empty()) {
    if (tmp.get(&d_tab, tab.size())) return -1;
    STIR_HIP(hipMemcpyAsync(d_tab, tab.data(), sizeof(DevBucketF32) * tab.size(), hipMemcpyHostToDevice, stream));
  }
  const CsfArrays csf = {src.A, src.indptr_i, src.indices_i, src.indptr_j, src.indices_j, src.nnz_i};
  uint64_t *keys_in = nullptr, *keys_out = nullptr, *unique = nullptr;
  int32_t *vals_in = nullptr, *vals_out = nullptr, *counts = nullptr, *first = nullptr, *flags = nullptr;
  int64_t* tile_begin = nullptr;
  if (tmp.get(&keys_in, slots) || tmp.get(&keys_out, slots) || tmp.get(&unique, slots) || tmp.get(&vals_in, slots) ||
      tmp.get(&vals_out, slots) || tmp.get(&counts, slots) || tmp.get(&first, slots) || tmp.get(&flags, 2) ||
      tmp.get(&tile_begin, tiles + 1))
    return -1;
  STIR_HIP(hipMemsetAsync(flags, 0, sizeof(int32_t) * 2, stream));
  const dim3 grid((unsigned)ceil_div(slots, 256)), block(256);
  const int nb = (int)tab.size();
  if (src.csf)
    hipLaunchKernelGGL(f32_edge_keys_kernel<true>, grid, block, 0, stream, d_tab, nb, csf, slots, m, n, num_rels,
                       keys_in, vals_in, flags);
  else
    hipLaunchKernelGGL(f32_edge_keys_kernel<false>, grid, block, 0, stream, d_tab, nb, csf, slots, m, n, num_rels,
                       keys_in, vals_in, flags);
  STIR_LAUNCH_CHECK();
  size_t bytes = sort_bytes;
  STIR_HIP(hipcub::DeviceRadixSort::SortPairs(cub_tmp, bytes, keys_in, keys_out, vals_in, vals_out, (int)slots, 0,
                                              key_bits, stream));
  // runs of equal key, cut into pieces of at most emax edges by a second key
  bytes = rle_bytes;
  STIR_HIP(hipcub::DeviceRunLengthEncode::Encode(cub_tmp, bytes, keys_out, unique, counts, flags + 1, (int)slots,
                                                 stream));
  int32_t host_flags[2] = {0, 0};
  STIR_HIP(hipMemcpyAsync(host_flags, flags, sizeof(host_flags), hipMemcpyDeviceToHost, stream));
  STIR_HIP(hipStreamSynchronize(stream));
  if (host_flags[0] != 0)
    return fail(host_flags[0] == 1 ? "rgms_f32: a row id or relation id lies outside [0, m) / [0, num_rels)"
                                   : "rgms_f32: a column id lies outside [0, n)");
  const int64_t key_runs = host_flags[1];
  bytes = scan_bytes;
  STIR_HIP(hipcub::DeviceScan::ExclusiveSum(cub_tmp, bytes, counts, first, (int)key_runs, stream));
  hipLaunchKernelGGL(f32_subkeys_kernel, grid, block, 0, stream, keys_out, first, key_runs, slots, (int)emax, keys_in,
                     flags);
  STIR_LAUNCH_CHECK();
  bytes = rle_bytes;
  STIR_HIP(hipcub::DeviceRunLengthEncode::Encode(cub_tmp, bytes, keys_in, unique, counts, flags + 1, (int)slots,
                                                 stream));
  STIR_HIP(hipMemcpyAsync(host_flags, flags, sizeof(host_flags), hipMemcpyDeviceToHost, stream));
  STIR_HIP(hipStreamSynchronize(stream));
  STIR_REQUIRE(host_flags[0] == 0, "rgms_f32: a (relation, row) pair has too many edges for the tiled kernel");
  const int64_t pairs = host_flags[1];
  idx.pairs = pairs;
  bytes = scan_bytes;
  STIR_HIP(hipcub::DeviceScan::ExclusiveSum(cub_tmp, bytes, counts, first, (int)pairs, stream));
  // the (tile, relation) runs of pairs.  keys_out and vals_in are free again; keys_in is
  // once the run-length encoding above has read it (same stream)
  uint64_t* run_of_pair = keys_out;
  uint64_t* run_keys = keys_in;
  int32_t *run_pairs = vals_in, *run_first_pair = nullptr;
  int32_t *run_batches = nullptr, *run_first_batch = nullptr;
  int64_t *pair_place = nullptr, *run_places = nullptr, *run_first_place = nullptr;
  if (tmp.get(&run_batches, pairs + 1) || tmp.get(&run_first_batch, pairs + 1) || tmp.get(&run_first_pair, pairs + 1) ||
      tmp.get(&pair_place, pairs) || tmp.get(&run_places, pairs + 1) || tmp.get(&run_first_place, pairs + 1))
    return -1;
  hipLaunchKernelGGL(f32_shift_keys_kernel, dim3((unsigned)ceil_div(pairs, 256)), block, 0, stream, unique, pairs,
                     run_of_pair);
  STIR_LAUNCH_CHECK();
  size_t rle2 = 0, scan2 = 0;
  STIR_HIP(hipcub::DeviceRunLengthEncode::Encode(nullptr, rle2, run_of_pair, run_keys, run_pairs, flags + 1, (int)pairs,
                                                 stream));
  STIR_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, scan2, run_pairs, run_first_pair, (int)pairs + 1, stream));
  STIR_REQUIRE(std::max(rle2, scan2) <= cub_bytes, "rgms_f32: scratch of the index build is too small");
  bytes = rle2;
  STIR_HIP(hipcub::DeviceRunLengthEncode::Encode(cub_tmp, bytes, run_of_pair, run_keys, run_pairs, flags + 1, (int)pairs,
                                                 stream));
  STIR_HIP(hipMemcpyAsync(host_flags, flags, sizeof(host_flags), hipMemcpyDeviceToHost, stream));
  STIR_HIP(hipStreamSynchronize(stream));
  const int64_t runs = host_flags[1];
  bytes = scan2;
  STIR_HIP(hipcub::DeviceScan::ExclusiveSum(cub_tmp, bytes, run_pairs, run_first_pair, (int)runs, stream));
  const dim3 run_grid((unsigned)ceil_div(runs, 4));
  hipLaunchKernelGGL(f32_batches_kernel<false>, run_grid, block, 0, stream, run_keys, run_pairs, run_first_pair,
                     (const int32_t*)nullptr, runs, num_rels, (int)emax, unique, counts, run_batches, run_places,
                     (const int64_t*)nullptr, (BatchF32*)nullptr, (uint32_t*)nullptr, (int64_t*)nullptr);
  STIR_LAUNCH_CHECK();
  // one entry more than runs: the last one is the batch count (run_batches[runs] is not read as an addend)
  STIR_HIP(hipMemsetAsync(run_batches + runs, 0, sizeof(int32_t), stream));
  bytes = scan2;
  STIR_HIP(hipcub::DeviceScan::ExclusiveSum(cub_tmp, bytes, run_batches, run_first_batch, (int)runs + 1, stream));
  STIR_HIP(hipMemsetAsync(run_places + runs, 0, sizeof(int64_t), stream));
  size_t scan3 = 0;
  STIR_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, scan3, run_places, run_first_place, (int)runs + 1, stream));
  STIR_REQUIRE(scan3 <= cub_bytes, "rgms_f32: scratch of the index build is too small");
  STIR_HIP(hipcub::DeviceScan::ExclusiveSum(cub_tmp, scan3, run_places, run_first_place, (int)runs + 1, stream));
  int32_t total_batches = 0;
  int64_t places = 0;
  STIR_HIP(hipMemcpyAsync(&places, run_first_place + runs, sizeof(int64_t), hipMemcpyDeviceToHost, stream));
  STIR_HIP(hipMemcpyAsync(&total_batches, run_first_batch + runs, sizeof(int32_t), hipMemcpyDeviceToHost, stream));
  STIR_HIP(hipStreamSynchronize(stream));
  idx.batches = total_batches;
  const int64_t words = (int64_t)total_batches * kBatch;
  STIR_REQUIRE(places < (int64_t(1) << 32), "rgms_f32: too many edges");
  const size_t batch_bytes = Scratch::rounded(sizeof(BatchF32) * (size_t)total_batches);
  const size_t word_bytes = Scratch::rounded(sizeof(uint32_t) * (size_t)words);
  STIR_HIP(hipMalloc(&idx.d_batches, batch_bytes + word_bytes + Scratch::rounded(sizeof(EdgeF32) * (size_t)places)));
  idx.d_pairs = static_cast<char*>(idx.d_batches) + batch_bytes;
  idx.d_edges = static_cast<char*>(idx.d_batches) + batch_bytes + word_bytes;
  EdgeF32* d_places = static_cast<EdgeF32*>(idx.d_edges);
  const float* some_weight = src.csf ? src.A : tab[0].A;
  hipLaunchKernelGGL(f32_clear_places_kernel, dim3((unsigned)ceil_div(std::max(places, words), 256)), block, 0, stream,
                     d_places, places, (int)emax, some_weight, static_cast<uint32_t*>(idx.d_pairs), words);
  STIR_LAUNCH_CHECK();
  hipLaunchKernelGGL(f32_batches_kernel<true>, run_grid, block, 0, stream, run_keys, run_pairs, run_first_pair,
                     run_first_batch, runs, num_rels, (int)emax, unique, counts, (int32_t*)nullptr,
                     (int64_t*)nullptr, run_first_place, static_cast<BatchF32*>(idx.d_batches), static_cast<uint32_t*>(idx.d_pairs), pair_place);
  STIR_LAUNCH_CHECK();
  if (src.csf)
    hipLaunchKernelGGL(f32_edge_records_kernel<true>, grid, block, 0, stream, d_tab, nb, csf, slots, num_rels,
                       (int)emax, vals_out, first, counts, pair_place, pairs, d_places);
  else
    hipLaunchKernelGGL(f32_edge_records_kernel<false>, grid, block, 0, stream, d_tab, nb, csf, slots, num_rels,
                       (int)emax, vals_out, first, counts, pair_place, pairs, d_places);
  STIR_LAUNCH_CHECK();
  hipLaunchKernelGGL(f32_tile_batches_kernel, dim3((unsigned)ceil_div(tiles + 1, 256)), block, 0, stream, run_keys,
                     run_first_batch, runs, (int64_t)total_batches, tiles, num_rels, tile_begin);
  STIR_LAUNCH_CHECK();
  idx.tile_begin.resize((size_t)tiles + 1);
  STIR_HIP(hipMemcpyAsync(idx.tile_begin.data(), tile_begin, sizeof(int64_t) * idx.tile_begin.size(),
                          hipMemcpyDeviceToHost, stream));
  STIR_HIP(hipStreamSynchronize(stream));  // also: the scratch arrays go away
  return 0;
}
}  // namespace

int f32_tiles_launch(F32TileIndex& idx, int32_t feat_in, int32_t feat_out, const float* d_W, const float* d_X,
                     float* d_Y, hipStream_t stream) {
  STIR_REQUIRE(f32_tiles_serves(feat_in, feat_out), "rgms_f32: feature sizes %d -> %d are not served by the tiled kernel",
               feat_in, feat_out);
  STIR_REQUIRE(idx.emax == (feat_in <= 32 ? 32 : 16), "rgms_f32: the edge index was built for another feat_in");
  if (idx.edges == 0) return 0;
  // the kernel's 32-bit byte offsets
  STIR_REQUIRE(f32_tiles_fits(idx.n, feat_in, idx.edges),
               "rgms_f32: the tiled kernel addresses X and its index with 32-bit offsets");
  const int ks = feat_in <= 32 ? 1 : 2, nt = feat_out <= 16 ? 1 : feat_out <= 32 ? 2 : 4;
  // W in operand order, rewritten by every launch (W may change between launches)
  const int64_t fragments = (int64_t)idx.num_rels * nt * ks * 64;
  const size_t wpack_bytes = 3 * sizeof(bf16x8) * (size_t)fragments;
  const bool wide = feat_out > 32;
  F32Units& u = idx.units[wide];
  if (!u.d_units || wpack_bytes > u.wpack_bytes || feat_out > u.feat_out) {
    if (u.d_units) STIR_HIP(hipFree(u.d_units));
    u = F32Units();
    if (make_units(u, idx.tile_begin, wide, feat_out, wpack_bytes, stream)) return -1;
  }
  if (u.count == 0) return 0;
  STIR_REQUIRE(u.count < (int64_t(1) << 31), "rgms_f32: too many units for one launch");
  bf16x8* wp = static_cast<bf16x8*>(u.d_wpack);
  hipLaunchKernelGGL(f32_pack_w_kernel, dim3((unsigned)ceil_div(fragments, 256)), dim3(256), 0, stream, d_W, wp, fragments, nt, ks,
                     feat_in, feat_out);
  STIR_LAUNCH_CHECK();
  const dim3 grid((unsigned)u.count);  // longest units first: they go to whichever slot is free
  const UnitF32* units = static_cast<const UnitF32*>(u.d_units);
  const BatchF32* bts = static_cast<const BatchF32*>(idx.d_batches);
  const uint32_t* pinfo = static_cast<const uint32_t*>(idx.d_pairs);
  const EdgeF32* edges = static_cast<const EdgeF32*>(idx.d_edges);
  float* partials = static_cast<float*>(u.d_partials);
#define STIR_F32_TILE(KS, NT)                                                                                   \
  hipLaunchKernelGGL((rgms_f32_tile_kernel<KS, NT>), grid, dim3((64 * TileShape<KS, NT>::kWaves)), 0, stream, idx.m, \
                     feat_in, feat_out, (int)idx.batches, (uint32_t)((int64_t)idx.n * feat_in * 4), units, bts,  \
                     pinfo, edges, wp, d_W, d_X, d_Y, partials, static_cast<uint32_t*>(u.d_arrived))
  switch (ks * 10 + nt) {
    case 11: STIR_F32_TILE(1, 1); break;
    case 12: STIR_F32_TILE(1, 2); break;
    case 14: STIR_F32_TILE(1, 4); break;
    case 21: STIR_F32_TILE(2, 1); break;
    case 22: STIR_F32_TILE(2, 2); break;
    default: STIR_F32_TILE(2, 4); break;
  }
#undef STIR_F32_TILE
  STIR_LAUNCH_CHECK();
  return 0;
}

}  // namespace stir
