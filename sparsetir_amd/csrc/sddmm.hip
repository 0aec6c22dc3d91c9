// SDDMM for gfx950, fp32: C[e] = <A[mid[e], :], B[indices[e], :]> for every nonzero e, and the
// row-lookup preprocess mid[e] = upper_bound(indptr, e) - 1.
//
// A wavefront owns 64 consecutive nonzeros.  Their mid / indices entries are fetched with one
// coalesced load each (lane l holds nonzero l).  The feature rows are spread over lane groups
// of G lanes (float4 per lane), so 64/G nonzeros are in flight per step; each dot product is
// finished with an all-reduce inside the lane group (DPP for distances below 16), and lane j
// of a group keeps the result of the group's j-th nonzero, so the 64 results leave with one
// coalesced store.
#include "common.h"
#include "row_lookup.h"
#include "../../include/sparsetir_amd.h"

namespace {

using stir::kWave;

template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}

// Sum over the G lanes of a lane group; every lane of the group gets the total.
template <int G>
__device__ __forceinline__ float group_allreduce(float p) {
  if constexpr (G >= 2) p += dpp_move<0xB1>(p);   // quad_perm [1,0,3,2]
  if constexpr (G >= 4) p += dpp_move<0x4E>(p);   // quad_perm [2,3,0,1]
  if constexpr (G >= 8) p += dpp_move<0x141>(p);  // row_half_mirror
  if constexpr (G >= 16) p += dpp_move<0x140>(p); // row_mirror
  if constexpr (G >= 32) p += __shfl_xor(p, 16, kWave);
  if constexpr (G >= 64) p += __shfl_xor(p, 32, kWave);
  return p;
}

// a row whose width is no multiple of four starts at any float: 16-byte loads need 4-byte alignment only
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ float4 ld4(const float* p) {
  const f32x4u v = *reinterpret_cast<const f32x4u*>(p);
  return make_float4(v[0], v[1], v[2], v[3]);
}

// TAIL: feat is no multiple of 4.  The row's last chunk of four features is then loaded from feat - 4
// on (it must not reach past the end of the array), and the features it shares with the chunk before
// it are left out of the product.
template <int G, int REP, bool TAIL>
__global__ __launch_bounds__(256) void sddmm_kernel(int64_t nnz, int feat, const float* __restrict__ A,
                                                    const float* __restrict__ B, float* __restrict__ C,
                                                    const int32_t* __restrict__ indices,
                                                    const int32_t* __restrict__ mid,
                                                    const float* __restrict__ scale) {
  constexpr int CH = (G < 4 ? G : 4);  // nonzeros in flight per lane group (2 row loads each)
  const int lane = threadIdx.x & 63;
  const int64_t tile = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int64_t e0 = tile * kWave;
  if (e0 >= nnz) return;
  const int g = lane / G, gl = lane % G;
  const int64_t e = e0 + lane;
  // streamed once: non-temporal, so they do not displace feature rows in the caches
  const int my_row = e < nnz ? __builtin_nontemporal_load(mid + e) : 0;
  const int my_col = e < nnz ? __builtin_nontemporal_load(indices + e) : 0;
  float out = 0.f;
#pragma unroll
  for (int c = 0; c < G; c += CH) {
    float4 a[CH][REP], b[CH][REP];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int sl = g * G + c + u;
      const int r = __shfl(my_row, sl, kWave);
      const int col = __shfl(my_col, sl, kWave);
      const float* ap = A + (int64_t)r * feat;
      const float* bp = B + (int64_t)col * feat;
#pragma unroll
      for (int q = 0; q < REP; ++q) {
        // feat below 4*G*REP: the lanes beyond feat / 4 hold padding
        const int c0 = gl * 4 + q * G * 4, at = TAIL ? min(c0, feat - 4) : c0;
        a[u][q] = c0 < feat ? ld4(ap + at) : make_float4(0.f, 0.f, 0.f, 0.f);
        b[u][q] = c0 < feat ? ld4(bp + at) : make_float4(0.f, 0.f, 0.f, 0.f);
        if constexpr (TAIL) {
          const int over = c0 - at;  // features of the chunk that belong to the one before
          a[u][q].x = over > 0 ? 0.f : a[u][q].x, b[u][q].x = over > 0 ? 0.f : b[u][q].x;
          a[u][q].y = over > 1 ? 0.f : a[u][q].y, b[u][q].y = over > 1 ? 0.f : b[u][q].y;
          a[u][q].z = over > 2 ? 0.f : a[u][q].z, b[u][q].z = over > 2 ? 0.f : b[u][q].z;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      float p = 0.f;
#pragma unroll
      for (int q = 0; q < REP; ++q) {
        p = fmaf(a[u][q].x, b[u][q].x, p);
        p = fmaf(a[u][q].y, b[u][q].y, p);
        p = fmaf(a[u][q].z, b[u][q].z, p);
        p = fmaf(a[u][q].w, b[u][q].w, p);
      }
      p = group_allreduce<G>(p);
      if (gl == c + u) out = p;
    }
  }
  if (e < nnz) __builtin_nontemporal_store(scale ? out * __builtin_nontemporal_load(scale + e) : out, C + e);
}

// Rows narrower than one float4 or wider than two per lane: one wavefront per 64 nonzeros, lanes
// stride over the features.
__global__ __launch_bounds__(256) void sddmm_generic_kernel(int64_t nnz, int feat, const float* __restrict__ A,
                                                            const float* __restrict__ B, float* __restrict__ C,
                                                            const int32_t* __restrict__ indices,
                                                            const int32_t* __restrict__ mid,
                                                            const float* __restrict__ scale) {
  const int lane = threadIdx.x & 63;
  const int64_t tile = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int64_t e0 = tile * kWave;
  if (e0 >= nnz) return;
  const int cnt = (int)min((int64_t)kWave, nnz - e0);
  float out = 0.f;
  for (int j = 0; j < cnt; ++j) {
    const float* ap = A + (int64_t)mid[e0 + j] * feat;
    const float* bp = B + (int64_t)indices[e0 + j] * feat;
    float p = 0.f;
    for (int f = lane; f < feat; f += kWave) p = fmaf(ap[f], bp[f], p);
    p = group_allreduce<64>(p);
    if (lane == j) out = p;
  }
  if (lane < cnt) C[e0 + lane] = scale ? out * scale[e0 + lane] : out;
}

// Row lookup mid[e] = upper_bound(indptr, e) - 1, 512 consecutive nonzeros per wavefront.
constexpr int kMidPerLane = 8;

__global__ __launch_bounds__(256) void sddmm_preproc_kernel(int m, int64_t nnz,
                                                            const int32_t* __restrict__ indptr,
                                                            int32_t* __restrict__ mid) {
  __shared__ int32_t win_all[4][stir::kRowLookupWindow];
  const int lane = threadIdx.x & 63;
  const int64_t e0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * (kWave * kMidPerLane);
  if (e0 >= nnz) return;
  const int64_t e_last = min(nnz, e0 + kWave * kMidPerLane) - 1;
  stir::for_each_nonzero_row<kMidPerLane>(indptr, m, e0, e_last, win_all[threadIdx.x >> 6], lane,
                                          [&](int64_t e, int row, int, bool live) {
                                            if (live) mid[e] = row;
                                          });
}

}  // namespace

extern "C" {

int stir_sddmm_preproc(int32_t m, int64_t nnz, const int32_t* d_indptr, int32_t* d_mid,
                       void* stream) {
  STIR_REQUIRE(m >= 0 && nnz >= 0, "sddmm_preproc: bad sizes m=%d nnz=%lld", m, (long long)nnz);
  if (nnz == 0) return 0;
  STIR_REQUIRE(d_indptr && d_mid, "sddmm_preproc: null pointer argument");
  const int64_t blocks = stir::ceil_div(nnz, 4 * kWave * kMidPerLane);
  STIR_REQUIRE(blocks < (int64_t(1) << 31), "sddmm_preproc: nnz=%lld exceeds one launch", (long long)nnz);
  hipLaunchKernelGGL(sddmm_preproc_kernel, dim3((unsigned)blocks), dim3(256), 0,
                     static_cast<hipStream_t>(stream), m, nnz, d_indptr, d_mid);
  STIR_LAUNCH_CHECK();
  return 0;
}

static int sddmm_launch(int32_t m, int32_t n, int32_t feat, int64_t nnz, const float* d_A, const float* d_B,
                        float* d_C, const int32_t* d_indices, const int32_t* d_mid, const float* d_scale,
                        void* stream) {
  STIR_REQUIRE(m >= 0 && n >= 0 && feat > 0 && nnz >= 0, "sddmm: bad sizes m=%d n=%d feat=%d", m, n, feat);
  if (nnz == 0) return 0;
  STIR_REQUIRE(d_A && d_B && d_C && d_indices && d_mid, "sddmm: null pointer argument");
  const int64_t blocks = stir::ceil_div(stir::ceil_div(nnz, kWave), 4);
  STIR_REQUIRE(blocks < (int64_t(1) << 31), "sddmm: nnz=%lld exceeds one launch", (long long)nnz);
  hipStream_t st = static_cast<hipStream_t>(stream);
  dim3 grid((unsigned)blocks), block(256);
#define STIR_SDDMM(G, REP)                                                                             \
  if (feat % 4 == 0)                                                                                   \
    hipLaunchKernelGGL((sddmm_kernel<G, REP, false>), grid, block, 0, st, nnz, feat, d_A, d_B, d_C, d_indices, d_mid, \
                       d_scale);                                                                       \
  else                                                                                                 \
    hipLaunchKernelGGL((sddmm_kernel<G, REP, true>), grid, block, 0, st, nnz, feat, d_A, d_B, d_C, d_indices, d_mid, \
                       d_scale)
  // the smallest lane group that covers the feature width
  int cls = -1;
  if (feat >= 4 && feat <= 512)
    for (cls = 0; (16 << cls) < feat; ++cls) {
    }
  switch (cls) {
    case 0: STIR_SDDMM(4, 1); break;
    case 1: STIR_SDDMM(8, 1); break;
    case 2: STIR_SDDMM(16, 1); break;
    case 3: STIR_SDDMM(32, 1); break;
    case 4: STIR_SDDMM(64, 1); break;
    case 5: STIR_SDDMM(64, 2); break;
    default:
      hipLaunchKernelGGL(sddmm_generic_kernel, grid, block, 0, st, nnz, feat, d_A, d_B, d_C, d_indices, d_mid,
                         d_scale);
  }
#undef STIR_SDDMM
  STIR_LAUNCH_CHECK();
  return 0;
}

int stir_sddmm_f32(int32_t m, int32_t n, int32_t feat, int64_t nnz, const float* d_A,
                   const float* d_B, float* d_C, const int32_t* d_indptr,
                   const int32_t* d_indices, const int32_t* d_mid, void* stream) {
  (void)d_indptr;  // part of the reference's argument list; rows come from mid
  return sddmm_launch(m, n, feat, nnz, d_A, d_B, d_C, d_indices, d_mid, nullptr, stream);
}

int stir_sddmm_scaled_f32(int32_t m, int32_t n, int32_t feat, int64_t nnz, const float* d_A,
                          const float* d_B, float* d_C, const int32_t* d_indptr,
                          const int32_t* d_indices, const int32_t* d_mid, const float* d_edge_values,
                          void* stream) {
  (void)d_indptr;
  STIR_REQUIRE(nnz == 0 || d_edge_values, "sddmm_scaled: edge values are null");
  return sddmm_launch(m, n, feat, nnz, d_A, d_B, d_C, d_indices, d_mid, d_edge_values, stream);
}

}  // extern "C"
