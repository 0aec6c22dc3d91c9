// CSR SpMM fp32 in one launch whose workgroups do equal work whatever the row lengths.
//
// The rows and the nonzeros are one list -- every row's mark, followed by its nonzeros -- and a workgroup
// takes `items` consecutive entries of it.  Inside, every lane group takes an equal stretch of the
// nonzeros, eight rows of B in flight, and writes a row of C when it meets the row's last nonzero; what
// is left of a row at either end of a stretch meets in LDS.  A row cut by the end of a workgroup leaves
// partial rows in memory; the workgroup that finishes last among those of the row -- a counter in device
// memory, set back to zero by that workgroup -- adds them up in order.  So C is written once, without
// atomics, and the same bits every time.
//
// Bound by the gather of rows of B (1.17 M nonzeros, 47 features: 36 us, 10 TB/s of the 128-byte lines
// that its rows touch).  With a launch over rows and a second one for what is long among them (spmm.hip) the
// same product pays a second launch, a search of every piece for long rows that mostly are not there, and
// wavefronts whose rows differ in length (51 us).
#include <algorithm>

#include "coherent.h"
#include "common.h"
#include "lane_group.h"
#include "../../include/sparsetir_amd.h"

namespace {

using stir::chunk_offset;
using stir::fma4;
using stir::kWave;
using stir::ld4;

constexpr int kBlock = 256;
// Workgroups per compute unit and the nonzeros that each then has room for in LDS (REP = 2: rows of more than 256
// features in one piece, whose partial sums take 8 KB more).
constexpr int resident(int rep) { return rep == 1 ? 7 : 6; }
constexpr int slots(int rep) { return rep == 1 ? 1152 : 832; }
// A row of at most this many nonzeros is not cut: it is left whole to the workgroup that has its mark, and may lie
// behind the workgroup's entries.
constexpr int kWhole = 128;
constexpr int max_items(int rep) { return slots(rep) - kWhole; }
constexpr int kFlight = 8;      // rows of B requested at a time by a lane group

// Last row r with indptr[r] + r <= q: q is a place in the list (indptr[0] added) and indptr[r] + r that of
// the row's mark (q >= indptr[0], m >= 1).  The whole wavefront looks, 64 places at a time; four times as
// many make the chain of round trips no shorter at these sizes and keep the texture addresser busy for
// 0.6 us a workgroup (64 cache lines per load).
__device__ __forceinline__ int last_mark(const int32_t* __restrict__ indptr, int m, int64_t q, int lane) {
  int lo = 0, hi = m - 1;
  while (hi > lo) {
    const int64_t span = hi - lo;
    const int base = lo;
    const int pos = base + (int)((span * (lane + 1) + kWave - 1) / kWave);  // in (lo, hi], ascending
    const int cnt = __popcll(__ballot((int64_t)indptr[pos] + pos <= q));
    if (cnt) lo = base + (int)((span * cnt + kWave - 1) / kWave);
    if (cnt < kWave) hi = base + (int)((span * (cnt + 1) + kWave - 1) / kWave) - 1;
  }
  return lo;
}

__device__ __forceinline__ void add4(float4& a, const float4& b) { a.x += b.x, a.y += b.y, a.z += b.z, a.w += b.w; }

__device__ __forceinline__ void store4(float* q, const float4& v) {
  __builtin_nontemporal_store(v.x, q);
  __builtin_nontemporal_store(v.y, q + 1);
  __builtin_nontemporal_store(v.z, q + 2);
  __builtin_nontemporal_store(v.w, q + 3);
}

// C[row] += acc by the only lane group that adds to the row in this launch.  All of the row is read before any of
// it is written: of a width that is no multiple of four, two chunks share features.
template <int G, int REP>
__device__ __forceinline__ void add_row(float* row, int feat, int gl, const float4 (&acc)[REP]) {
  float4 old[REP];
#pragma unroll
  for (int r = 0; r < REP; ++r) {
    const int c0 = gl * 4 + r * G * 4;
    if (c0 < feat) old[r] = ld4(row + chunk_offset(c0, feat));
  }
#pragma unroll
  for (int r = 0; r < REP; ++r) {
    const int c0 = gl * 4 + r * G * 4;
    if (c0 >= feat) continue;
    add4(old[r], acc[r]);
    float* q = row + chunk_offset(c0, feat);
    q[0] = old[r].x, q[1] = old[r].y, q[2] = old[r].z, q[3] = old[r].w;
  }
}

// MERGED: the merged rows of a hyb plan (spmm.hip).  A holds addresses of the values, slots of value 0 (padding)
// fetch no row of B, and the product is added to C: what a workgroup has of a row that it shares with others goes
// there by atomics, so there are no partial rows to be added up.
template <int G, int REP, bool MERGED = false>
__global__ __launch_bounds__(kBlock, resident(REP)) void csr_balanced_kernel(int m, int stride, int slices, int64_t nnz,
                                                                             int items, const float* __restrict__ A,
                                                                             const float* __restrict__ B,
                                                                             float* __restrict__ C,
                                                                             const int32_t* __restrict__ indptr,
                                                                             const int32_t* __restrict__ indices,
                                                                             uint32_t* __restrict__ counters,
                                                                             float* __restrict__ partials) {
  constexpr int NG = kBlock / G;
  constexpr int CH = kFlight / REP;
  constexpr int kPad = 4 * G * REP;  // floats of a partial row
  constexpr int kSlots = slots(REP);
  __shared__ int2 nz[kSlots];     // column, value
  __shared__ int ends[kSlots];    // row + 1 at the row's last nonzero, else 0
  __shared__ float4 head[NG * G * REP], tail[NG * G * REP];
  __shared__ int open_all[NG];
  __shared__ int row_at[2], nz_at[2], cut[2];
  __shared__ int last[2];
  // all of the above, and what an allocation is rounded up to, in a share of the compute unit's 160 KB
  static_assert((kSlots * 12 + 2 * NG * G * REP * 16 + NG * 4 + 32 + 1279) / 1280 * 1280 * resident(REP) <= 160 * 1024,
                "fewer workgroups per compute unit than the number of workgroups is chosen for");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int base = indptr[0];
  const int64_t total = m + min(nnz, (int64_t)indptr[m]) - base;
  int feat = stride;
  int64_t wg = blockIdx.x;
  if (slices > 1) {  // see slice_block
    const int64_t wgs = (m + nnz + items - 1) / items;
    int slice;
    stir::slice_block(blockIdx.x, slices, wgs, slice, wg);
    const int f0 = slice * kPad;
    B += f0, C += f0, feat -= f0;
    if (!MERGED) counters += slice * wgs, partials += slice * wgs * 2 * kPad;
  }
  const int64_t d0 = wg * items, d1 = min(total, d0 + items);
  if (d0 >= total) return;
  if (wave < 2) {
    const int64_t d = wave ? d1 : d0;
    int i = 0, j = base, c = 0;
    if (d > 0) {
      const int r = last_mark(indptr, m, d - 1 + base, lane);
      const int s = indptr[r], e = indptr[r + 1];
      i = r + 1, j = (int)(d - i + base);
      if (e > j) {
        c = e - s > kWhole;
        if (c) c = s < j; else j = e;
      }
    }
    if (lane == 0) row_at[wave] = i, nz_at[wave] = j, cut[wave] = c;
  }
  for (int t = tid; t < kSlots; t += kBlock) ends[t] = 0;
  __syncthreads();
  // rows [i0, i1) have their marks here, the nonzeros [j0, j1) belong to them and, cut_before, to row i0 - 1
  const int i0 = __builtin_amdgcn_readfirstlane(row_at[0]), i1 = __builtin_amdgcn_readfirstlane(row_at[1]);
  const int j0 = __builtin_amdgcn_readfirstlane(nz_at[0]), j1 = __builtin_amdgcn_readfirstlane(nz_at[1]);
  const bool cut_before = __builtin_amdgcn_readfirstlane(cut[0]), cut_after = __builtin_amdgcn_readfirstlane(cut[1]);
  const int cnt = j1 - j0;
  for (int t = tid; t < cnt; t += kBlock) {
    float value;
    if constexpr (MERGED)
      value = *reinterpret_cast<const float* const*>(A)[j0 + t];
    else
      value = __builtin_nontemporal_load(A + j0 + t);
    nz[t] = make_int2(__builtin_nontemporal_load(indices + j0 + t), __float_as_int(value));
  }
  const int first = max(i0 - 1, 0);
  for (int r0 = first; r0 < i1; r0 += kBlock) {
    const int r = r0 + tid;
    int s = 0, e = 0;
    if (r < i1) s = indptr[r], e = indptr[r + 1];
    if (e > j0 && e > s && e <= j1) ends[e - 1 - j0] = r + 1;
    if constexpr (MERGED) continue;
    uint64_t empty = __ballot(r >= i0 && r < i1 && s == e);
    while (empty) {
      const int k = __ffsll((long long)empty) - 1;
      empty &= empty - 1;
      float* row = C + (int64_t)(r0 + wave * kWave + k) * stride;
      for (int f = lane; f < min(feat, kPad); f += kWave) __builtin_nontemporal_store(0.f, row + f);
    }
  }
  __syncthreads();

  const int grp = tid / G, gl = tid % G;
  const int per = max(CH, (cnt + NG - 1) / NG);
  const int a = min(cnt, grp * per), b = min(cnt, a + per);
  const bool mid = a < b ? (a > 0 ? ends[a - 1] == 0 : cut_before) : true;  // begins inside a row
  bool flushed = false;
  int head_row = 0;
  float4 acc[REP];
#pragma unroll
  for (int r = 0; r < REP; ++r) acc[r] = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int k0 = 0; k0 < per; k0 += CH) {
    float4 x[CH][REP];
    float v[CH];
    int f[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int p = a + k0 + u;
      bool live = p < b;
      const int2 q = nz[min(p, kSlots - 1)];
      f[u] = live ? ends[min(p, kSlots - 1)] : 0;
      v[u] = live ? __int_as_float(q.y) : 0.f;
      if constexpr (MERGED) live = live && v[u] != 0.f;
      const float* bp = B + (int64_t)q.x * stride;
#pragma unroll
      for (int r = 0; r < REP; ++r) {
        const int c0 = gl * 4 + r * G * 4;
        x[u][r] = live && c0 < feat ? ld4(bp + chunk_offset(c0, feat)) : make_float4(0.f, 0.f, 0.f, 0.f);
      }
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) {
#pragma unroll
      for (int r = 0; r < REP; ++r) fma4(acc[r], v[u], x[u][r]);
      if (f[u]) {
        const bool keep = mid && !flushed;
        float* row = C + (int64_t)(f[u] - 1) * stride;
#pragma unroll
        for (int r = 0; r < REP; ++r) {
          const int c0 = gl * 4 + r * G * 4;
          if (keep)
            head[(grp * REP + r) * G + gl] = acc[r];
          else if (!MERGED && c0 < feat)
            store4(row + chunk_offset(c0, feat), acc[r]);
        }
        if constexpr (MERGED) {
          if (!keep) add_row<G, REP>(row, feat, gl, acc);
        }
#pragma unroll
        for (int r = 0; r < REP; ++r) acc[r] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (keep) head_row = f[u];
        flushed = true;
      }
    }
  }
#pragma unroll
  for (int r = 0; r < REP; ++r) tail[(grp * REP + r) * G + gl] = acc[r];
  if (gl == 0) open_all[grp] = mid && !flushed;
  __syncthreads();

  // pieces of rows: what the groups before a head left of its row, and of the row the workgroup ends in
  const uint64_t open_groups = __ballot(lane < NG && open_all[lane % NG]);
  const bool through = cut_after && cut_before && i0 == i1;
  const stir::CoherentPiece own(partials + wg * 2 * kPad, 2 * kPad * 4);  // of a row it begins in, of one it ends in
  for (int which = 0; which < 2; ++which) {
    const bool mine = which == 0 ? head_row != 0 : cut_after && grp == NG - 1;
    if (!mine) continue;
    // the row began in group k, -1: in a workgroup before this one
    const uint64_t closed = ~open_groups & ((uint64_t(1) << (which == 0 ? grp : NG - 1) << (which == 0 ? 0 : 1)) - 1);
    const int k = closed ? 63 - __clzll((long long)closed) : -1;
    float4 sum[REP];
#pragma unroll
    for (int r = 0; r < REP; ++r)
      sum[r] = which == 0 ? head[(grp * REP + r) * G + gl] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
    for (int q = max(k, 0); q < (which == 0 ? grp : NG); ++q)
#pragma unroll
      for (int r = 0; r < REP; ++r) add4(sum[r], tail[(q * REP + r) * G + gl]);
    if constexpr (MERGED) {
      if (which == 0 && k >= 0) {
        add_row<G, REP>(C + (int64_t)(head_row - 1) * stride, feat, gl, sum);
        continue;
      }
    }
#pragma unroll
    for (int r = 0; r < REP; ++r) {
      const int c0 = gl * 4 + r * G * 4;
      if constexpr (MERGED) {
        if (c0 >= feat) continue;
        const int over = c0 + 4 - feat;
        const float4 v = over > 0 ? stir::tail_chunk(sum[r], over) : sum[r];
        float* q = C + (int64_t)((which == 0 ? i0 : i1) - 1) * stride + c0;
        const float part[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int f = 0; f < 4; ++f)
          if (c0 + f < feat) __hip_atomic_fetch_add(q + f, part[f], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        continue;
      }
      if (which == 0 && k >= 0) {
        if (c0 < feat) store4(C + (int64_t)(head_row - 1) * stride + chunk_offset(c0, feat), sum[r]);
      } else {
        own.store(which * kPad + c0, sum[r]);
      }
    }
  }
  if constexpr (MERGED) return;
  // a row that goes through the whole workgroup counts as the one it ends in
  const bool has_head = cut_before && !through;
  if (!has_head && !cut_after) return;  // uniform
  // every store above has to have reached memory before the workgroup counts itself in
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid < 2) {
    const bool mine = tid == 0 ? has_head : cut_after;
    int before_last = 0;
    if (mine) {
      const int64_t r = tid == 0 ? i0 - 1 : i1 - 1;
      const int64_t b0 = (indptr[r] - base + r + 1) / items, b1 = (indptr[r + 1] - base + r) / items;
      before_last = __hip_atomic_fetch_add(counters + b0, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)(b1 - b0);
      if (before_last) __hip_atomic_store(counters + b0, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    last[tid] = before_last;
  }
  __syncthreads();
  for (int which = 0; which < 2; ++which) {
    if (!last[which]) continue;  // uniform
    const int r = which == 0 ? i0 - 1 : i1 - 1;
    const int64_t b0 = ((int64_t)indptr[r] - base + r + 1) / items, b1 = ((int64_t)indptr[r + 1] - base + r) / items;
    const int count = (int)(b1 - b0) + 1, share = (count + NG - 1) / NG;
    float4 sum[REP];
#pragma unroll
    for (int q = 0; q < REP; ++q) sum[q] = make_float4(0.f, 0.f, 0.f, 0.f);
    // Eight partial rows in flight: one at a time a row of 300 k nonzeros, 256 features ended on a chain of 150 round
    // trips to memory (120 -> 65 us in all).  A row's workgroups leave less than 2^32 bytes.
    const stir::CoherentPiece all(partials + b0 * 2 * kPad, (uint32_t)count * 2 * kPad * 4);
    const int k1 = min(count, (grp + 1) * share);
    for (int k0 = grp * share; k0 < k1; k0 += 8) {
#pragma unroll
      for (int q = 0; q < REP; ++q) {
        float4 y[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int k = min(k0 + u, k1 - 1);  // the last piece is the head of its workgroup, the others are tails
          y[u] = all.load((2 * k + (k == count - 1 ? 0 : 1)) * kPad + gl * 4 + q * G * 4);
        }
        __builtin_amdgcn_sched_barrier(0);  // all eight, then the sums
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (k0 + u < k1) add4(sum[q], y[u]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < REP; ++q) tail[(grp * REP + q) * G + gl] = sum[q];
    __syncthreads();
    if (grp == 0) {
      const int used = min(NG, count);
      for (int k = 1; k < used; ++k)
#pragma unroll
        for (int q = 0; q < REP; ++q) add4(sum[q], tail[(k * REP + q) * G + gl]);
#pragma unroll
      for (int q = 0; q < REP; ++q) {
        const int c0 = gl * 4 + q * G * 4;
        if (c0 < feat) store4(C + (int64_t)r * stride + chunk_offset(c0, feat), sum[q]);
      }
    }
  }
}

// Lane groups as wide as feat, or of 64 features and several feature slices (slice_block): an XCD's L2 holds
// more rows of B a slice wide, which pays for looking for the entries once per slice from 1.5e8 multiplications
// on, as long as slices begin on 256-byte boundaries and B is not far beyond what the last level holds.
// In one piece / in slices, uniform and skewed columns, us:
//   25 k rows, 1 M nonzeros, 256 features 136 / 87, 84 / 81 (300 k nonzeros 49 / 40, 31 / 38);
//   60 k, 720 k, 256: 118 / 97, 71 / 72 (128: 58 / 54, 36 / 39); 150 k, 1.2 M, 192: 154 / 142, 102 / 90;
//   300 k, 7.8 M, 128: 573 / 563, 434 / 377; the same, 256 (307 MB): 1161 / 1167, 1016 / 797;
//   600 k, 6 M, 256 (614 MB): 932 / 1012, 786 / 757.
// The upper end of the products is that of the measurements (and bounds the workspace).
int slice_class(int32_t n, int32_t feat, int64_t nnz) {
  const int whole = stir::vector_class(feat);
  const int64_t work = nnz * feat;
  const bool cut = whole > 2 && feat % 64 == 0 && work >= 150000000 && work <= 2500000000 &&
                   (int64_t)n * feat * 4 <= 320000000;
  return cut ? 2 : whole;
}

// In one piece, as many workgroups as are resident at once, so that all end together: seven per compute unit (rows of
// more than 256 features: six) where that leaves them a few hundred entries each, else five.  us with 4 / 5 / 6 / 7 / 8
// per compute unit, and with 512 entries each:
//   169 k rows, 1.17 M nonzeros, 64 features 35.2 / 35.3 / 33.0 / 32.2 / 36.2, 35.6; 47: 39.3 / 39.4 / 37.1 / 36.1 / 39.8, 39.7;
//   108 k, 1.2 M, 64: 33.4 / 33.3 / 31.8 / 31.4 / 35.2, 34.4; 17 k, 288 k, 12: 10.3 / 10.1 / 10.6 / 11.3 / 13.7, 10.2;
//   54 k, 521 k, 100: 27.6 / 28.1 / 27.8 / 28.1 / 30.8, 29.2; 9 k, 146 k, 64: 10.3 / 9.8 / 10.1 / 10.4 / 12.9, 10.3.
// In slices of features 768 entries: their workgroups take several turns anyhow, each looks for its entries once per
// slice, and the less of a slice of B comes from memory the more that counts.  512 / 768 / 1024, uniform and skewed
// columns:
//   169 k, 1.17 M, 192: 140 / 146 / 147, 92 / 89 / 90; 256: 188 / 189 / 189, 145 / 142 / 142; merged rows of two
//   partitions 213 / 216 / 223, 172 / 166 / 167; 100 k, 2 M, 256: 279 / 282 / 284, 173 / 168 / 167; 50 k, 2 M, 192: 181 /
//   183 / 184, 112 / 104 / 102; 400 k, 5 M, 192: 579 / 588 / 592 (896 entries), 385 / 374 / 372; 25 k, 1 M, 256: 88 / 86 /
//   85, 80 / 76 / 75; 10 k, 300 k, 512: 50 / 48 / 45 (896), 50 / 48 / 46, with five per compute unit and slice 59, 58.
// Six of the wide ones: with room for 1152 nonzeros only five fit, and a sixth each was a turn of its own (uniform /
// skewed columns, 1152 and 832 nonzeros): 60 k rows, 1 M nonzeros, 260 features 178 / 129, 172 / 114; 100 k, 1.4 M, 300
// 283 / 204, 281 / 193; merged rows 100 k, 700 k, 300 184 / 139, 176 / 116; 30 k, 500 k, 400 140 / 101, 139 / 87.  Five
// that ask for five: the same for CSR, but merged rows 100 k, 700 k, 300 177 / 126, 500 278 / 213 against 285 / 192.
// Up to 32 features no fewer than 256 entries, eight for each of 32 or more lane groups (us with 64 / 256 as the fewest,
// 512 entries each): 16 k rows, 121 k nonzeros, 8 features 9.7 / 8.7, 9.2; 10 k, 100 k, 32: 9.3 / 8.7, 8.7; 12 k, 200 k,
// 16: 9.7 / 9.3, 9.5; but 9 k, 115 k, 84 12.1 / 13.6, 12.2; 9 k, 60 k, 128 11.1 / 13.4, 11.0.
// The other way (us, against some 1100 workgroups of 32 k entries): 100 k rows, 1.5 M nonzeros of uniform columns, 128
// features 111.4, 109.3 (skewed: 69.6, 73.0); 60 k, 400 k, 32 11.4, 9.7; 50 k, 350 k, 20 11.1, 9.8 and 32 10.7, 9.2; 8 k,
// 150 k, 500 43.4, 41.4.  Up to 32 features a few entries more or less to a lane group move single sizes by 15 % either
// way (40 k, 300 k, 28 10.2, 10.9; 60 k, 400 k, 12 8.1, 9.4); the mean over 10 sizes each of 12 to 48 features is 2 % less.
// More than one turn of the largest workgroups (beyond_a_turn), 512 / 768 / 1024 entries, uniform and skewed columns: a
// last turn that is nearly empty costs wide rows more, finding the entries narrow ones.
//   170 k rows, 2 M nonzeros, 8 features 34.3 / 32.1 / 30.9, 32.2 / 30.2 / 29.0; 600 k, 20 M, 4: 265 / 245 / 240,
//   249 / 213 / 197; 170 k, 1.7 M (1.02 turns), 32: 41.6 / 40.9 / 43.5, 32.5 / 30.8 / 31.8; 1.9 M: 44.5 / 43.7 / 45.2,
//   34.6 / 31.8 / 32.9; 2.7 M: 55.9 / 55.8 / 55.5, 44.1 / 41.1 / 38.7; 500 k, 12 M, 32: 234 / 235 / 236, 169 / 153 / 150;
//   170 k, 2 M, 64: 81.2 / 83.3 / 84.2, 52.7 / 53.0 / 54.3; 3.5 M: 129.7 / 132.3 / 135.5, 81.5 / 80.6 / 79.5; 50 k, 2.6 M,
//   47: 74.7 / 74.0 / 75.2, 56.7 / 54.5 / 53.4; 300 k, 4.5 M, 64: 174 / 178 / 177, 112 / 111 / 112;
//   170 k, 2 M, 150: 221 / 224 / 226, 145 / 149 / 153; 2.8 M, 100: 209 / 214 / 216, 132.5 / 134.8 / 135.2.
// Turns made equal (two of 560 to 1024 entries each) lie between: 2.4 M, 64 95.7 against 95.2 with 512; 2.4 M, 32 37.4
// against 36.3 with 1024.
int64_t beyond_a_turn(int c, int64_t entries, int64_t turn) {
  if (c == 0) return 1024;
  if (c == 1) return 4 * entries <= 5 * turn ? 768 : 1024;
  return c == 2 && entries <= 2 * turn ? 768 : 512;
}

int entries_per_workgroup(int32_t m, int32_t n, int32_t feat, int64_t nnz) {
  const int c = slice_class(n, feat, nnz), slices = (int)stir::ceil_div(feat, 16 << c), rep = c == 5 ? 2 : 1;
  constexpr int64_t kUnits = 256;  // compute units
  const int64_t entries = m + nnz, most = max_items(rep);
  int64_t per_unit = resident(rep);
  if (slices > 1) return 768;
  const int64_t turn = kUnits * per_unit * most;
  if (entries > turn) return (int)beyond_a_turn(c, entries, turn);
  if (entries < kUnits * per_unit * 400) per_unit = 5;
  const int64_t items = stir::ceil_div(entries, kUnits * per_unit);
  const int64_t fewest = c <= 1 ? 256 : 64;
  return (int)(std::max(fewest, std::min(items, most)) + 3) / 4 * 4;
}

int64_t workgroups(int32_t m, int32_t n, int32_t feat, int64_t nnz) {
  return stir::ceil_div(m + nnz, entries_per_workgroup(m, n, feat, nnz));
}

// Below, the search for its entries costs a workgroup more than it gains (4096 rows, 65 k nonzeros, 32
// features: 8.6 us against 6.9); above, if not in slices, two launches over rows read B as fast and leave no
// partial rows (2.4 M rows, 61.9 M nonzeros, 128 features: 5.49 ms against 4.98).  Between (old / new, us):
// 6 k rows, 90 k nonzeros, 128 features 15.5 / 10.0; 24 k, 360 k, 33: 19.4 / 13.1; 50 k, 450 k, 8: 24.3 / 11.6;
// 169 k, 1.17 M, 47: 50.7 / 38.2; 115 k, 2.3 M, 64: 92 / 85; 100 k, 1.5 M, 128: 121 / 117.
bool balanced(int32_t m, int32_t n, int32_t feat, int64_t nnz) {
  const int c = stir::vector_class(feat);
  if (c < 0 || (nnz * feat >= 500000000 && slice_class(n, feat, nnz) == c)) return false;
  return m >= 8192 || nnz * feat >= 3000000;
}

template <bool MERGED>
int launch(int c, int64_t grid, int slices, int items, int32_t m, int32_t feat, int64_t nnz, const float* d_A,
           const float* d_B, float* d_C, const int32_t* d_indptr, const int32_t* d_indices, uint32_t* counters,
           float* partials, hipStream_t st) {
#define STIR_BALANCED(G, REP)                                                                                        \
  hipLaunchKernelGGL((csr_balanced_kernel<G, REP, MERGED>), dim3((unsigned)grid), dim3(kBlock), 0, st, m, feat,       \
                     slices, nnz, items, d_A, d_B, d_C, d_indptr, d_indices, counters, partials)
  switch (c) {
    case 0: STIR_BALANCED(4, 1); break;
    case 1: STIR_BALANCED(8, 1); break;
    case 2: STIR_BALANCED(16, 1); break;
    case 3: STIR_BALANCED(32, 1); break;
    case 4: STIR_BALANCED(64, 1); break;
    default: STIR_BALANCED(64, 2); break;
  }
#undef STIR_BALANCED
  STIR_LAUNCH_CHECK();
  return 0;
}

}  // namespace

namespace stir {

bool merged_balanced(int32_t m, int32_t n, int32_t feat, int64_t slots) { return balanced(m, n, feat, slots); }

int launch_merged_balanced(int32_t m, int32_t n, int32_t feat, int64_t slots, const float* const* d_vals,
                           const float* d_B, float* d_C, const int32_t* d_slot_ptr, const int32_t* d_cols,
                           hipStream_t st) {
  const int c = slice_class(n, feat, slots), slices = (int)ceil_div(feat, 16 << c);
  const int64_t grid = slice_grid(slices, workgroups(m, n, feat, slots));
  STIR_REQUIRE(grid < (int64_t(1) << 31), "hyb_spmm: %lld workgroups exceed one launch", (long long)grid);
  return launch<true>(c, grid, slices, entries_per_workgroup(m, n, feat, slots), m, feat, slots,
                      reinterpret_cast<const float*>(d_vals), d_B, d_C, d_slot_ptr, d_cols, nullptr, nullptr, st);
}

}  // namespace stir

extern "C" {

// the counters, one per workgroup; behind them two partial rows per workgroup
size_t stir_csr_spmm_workspace_clear_bytes(int32_t m, int32_t n, int32_t feat, int64_t nnz) {
  if (m < 0 || n < 0 || feat <= 0 || nnz < 0 || !balanced(m, n, feat, nnz)) return 0;
  const size_t parts = size_t(workgroups(m, n, feat, nnz)) * stir::ceil_div(feat, 16 << slice_class(n, feat, nnz));
  return (parts * 4 + 15) / 16 * 16;
}

size_t stir_csr_spmm_workspace_bytes(int32_t m, int32_t n, int32_t feat, int64_t nnz) {
  if (m < 0 || n < 0 || feat <= 0 || nnz < 0 || !balanced(m, n, feat, nnz)) return 0;
  const int c = slice_class(n, feat, nnz);
  const size_t parts = size_t(workgroups(m, n, feat, nnz)) * stir::ceil_div(feat, 16 << c);
  return stir_csr_spmm_workspace_clear_bytes(m, n, feat, nnz) + parts * 2 * (size_t(16) << c) * 4;
}

int stir_csr_spmm_f32_workspace(int32_t m, int32_t n, int32_t feat, int64_t nnz, const float* d_A, const float* d_B,
                                float* d_C, const int32_t* d_indptr, const int32_t* d_indices, void* d_workspace,
                                void* stream) {
  STIR_REQUIRE(m >= 0 && n >= 0 && feat > 0 && nnz >= 0, "csr_spmm: bad sizes m=%d n=%d feat=%d", m, n, feat);
  if (m == 0 || !balanced(m, n, feat, nnz))
    return stir_csr_spmm_f32(m, n, feat, nnz, d_A, d_B, d_C, d_indptr, d_indices, stream);
  STIR_REQUIRE(d_B && d_C && d_indptr && d_workspace && (nnz == 0 || (d_A && d_indices)),
               "csr_spmm: null pointer argument");
  const int64_t wgs = workgroups(m, n, feat, nnz);
  const int c = slice_class(n, feat, nnz), slices = (int)stir::ceil_div(feat, 16 << c);
  const int64_t grid = stir::slice_grid(slices, wgs);
  STIR_REQUIRE(grid < (int64_t(1) << 31), "csr_spmm: %lld workgroups exceed one launch", (long long)grid);
  const int items = entries_per_workgroup(m, n, feat, nnz);
  uint32_t* counters = static_cast<uint32_t*>(d_workspace);
  float* partials = reinterpret_cast<float*>(static_cast<char*>(d_workspace) +
                                             stir_csr_spmm_workspace_clear_bytes(m, n, feat, nnz));
  return launch<false>(c, grid, slices, items, m, feat, nnz, d_A, d_B, d_C, d_indptr, d_indices, counters, partials,
                       static_cast<hipStream_t>(stream));
}

}  // extern "C"
