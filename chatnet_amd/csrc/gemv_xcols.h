// gemv_xcols.h — a few columns of x (2 to 7) against the same rows of a type
// multiplied in fp32 (fine_type), instantiated by the gemv_*.hip files.
//
// The columns' fp32 records (stage_fp32's) lie in LDS together and every group of
// 16 weights, unpacked once, meets all of them: one pass over W, where one launch
// per column reads and unpacks it again each time.  Bound by the fma per weight and
// column and by the LDS reads of x, which two rows share (per library call, calls back
// to back): Q5_0 11008 x 4096 at 3
// columns 13.8 us, at 7 26.9; a packing pass and a GEMV per column took 103 and 200,
// the matrix-core product of x in 23-bit digits 14.9 and 21.7.  Rows whose columns do
// not fit in LDS together run in groups: 4096 x 11008 at 7 columns 41.7 us.  Error
// against float64 1.1e-7, as the single column's.
#pragma once
#include "gemv_quant.h"

namespace {

// A unit of RPW rows against the records of ncols columns, cstride floats apart.
template <int QT, int RPW, int NC>
__device__ __forceinline__ void dot_unit_cols(const uint32_t (*w)[QTraits<QT>::NDW], const float* rec, int cstride, int h,
                                              int ncols, float (&acc)[NC][RPW]) {
  constexpr int G = QTraits<QT>::UNIT / 16;
#pragma unroll
  for (int g = 0; g < G; g++) {
    uint32_t q[RPW][4];
    float a[RPW], b[RPW];
#pragma unroll
    for (int i = 0; i < RPW; i++) unit_group<QT>(w[i], h, g, q[i], a[i], b[i]);
#pragma unroll
    for (int c = 0; c < NC; c++)
      if (c < ncols) {
        const float* r = rec + c * cstride;
        float4 x[4];
#pragma unroll
        for (int k = 0; k < 4; k++) x[k] = *reinterpret_cast<const float4*>(r + 16 * g + 4 * k);
        const float sx = group_min<QT>() ? r[16 * G + g] : 0.f;
#pragma unroll
        for (int i = 0; i < RPW; i++) {
          if constexpr (group_min<QT>()) acc[c][i] = fmaf(b[i], sx, acc[c][i]);
          acc[c][i] = fmaf(a[i], group_dot(q[i], x), acc[c][i]);
        }
      }
  }
}

template <int QT, int NC, int LPR, int NU>
__global__ __launch_bounds__(512) void gemv_xcols_kernel(GemvArgs a, int ncols) {
  using T = QTraits<QT>;
  constexpr int BS = 512, NWV = BS / CN_WAVE, RPW = 2, RW = RPW * (CN_WAVE / LPR);
  extern __shared__ float smem[];
  const int K = a.K, M = a.n_vrows;
  const int nunits = K / T::UNIT, groups = K >> 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int sub = lane / LPR, li = lane % LPR;
  const int n_iters = (M + RW - 1) / RW;
  const size_t bpr = (size_t)(K / T::BLOCK) * T::BLOCK_BYTES;
  const int wstride = gridDim.x * NWV, cstride = nunits * xf_unit_dw<QT>();
  int it = blockIdx.x * NWV + wave;

  uint32_t w[RPW][NU][T::NDW];
  issue_loads<QT, RPW, LPR, NU, GEMV_EPI_STORE>(a, it, sub, li, nunits, bpr, w);
  for (int t = threadIdx.x; t < ncols * groups; t += BS) {
    const int c = t / groups, g = t - c * groups;
    float v[16];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const float4 f = *reinterpret_cast<const float4*>(a.x + (size_t)c * K + 16 * g + 4 * k);
      v[4 * k] = f.x; v[4 * k + 1] = f.y; v[4 * k + 2] = f.z; v[4 * k + 3] = f.w;
    }
    store_group_fp32<QT>(v, g, smem + c * cstride);
  }
  __syncthreads();
  while (it < n_iters) {
    float acc[NC][RPW];
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
      for (int i = 0; i < RPW; i++) acc[c][i] = 0.f;
#pragma unroll
    for (int n = 0; n < NU; n++) {
      const int u = li + LPR * n;
      if (u < nunits) {
        uint32_t wu[RPW][T::NDW];
#pragma unroll
        for (int i = 0; i < RPW; i++)
#pragma unroll
          for (int k = 0; k < T::NDW; k++) wu[i][k] = w[i][n][k];
        dot_unit_cols<QT, RPW, NC>(wu, smem + u * xf_unit_dw<QT>(), cstride, u & 1, ncols, acc);
      }
    }
    const int row0 = it * RW + sub * RPW;
    it += wstride;
    if (it < n_iters) issue_loads<QT, RPW, LPR, NU, GEMV_EPI_STORE>(a, it, sub, li, nunits, bpr, w);
#pragma unroll
    for (int c = 0; c < NC; c++)
      if (c < ncols) {
#pragma unroll
        for (int i = 0; i < RPW; i++) {
#pragma unroll
          for (int off = LPR / 2; off > 0; off >>= 1) acc[c][i] += __shfl_xor(acc[c][i], off, CN_WAVE);
          if (li == 0 && row0 + i < M) a.out[0][(size_t)c * M + row0 + i] = acc[c][i];
        }
      }
  }
}

template <int QT, int NC, int LPR, int NU>
hipError_t launch_xcols_k(const GemvArgs& a, int ncols, int num_cus, hipStream_t st) {
  constexpr int RW = 2 * (CN_WAVE / LPR);
  const size_t smem = (size_t)ncols * (a.K / QTraits<QT>::UNIT) * xf_unit_dw<QT>() * sizeof(float);
  const auto kern = &gemv_xcols_kernel<QT, NC, LPR, NU>;
  if (smem > 64 * 1024) {
    static std::atomic<uint64_t> lds_done{0};
    const hipError_t e = allow_full_lds(reinterpret_cast<const void*>(kern), lds_done);
    if (e != hipSuccess) return e;
  }
  if (smem > (size_t)kCuLdsBytes) return hipErrorInvalidValue;
  const int per_cu = 2 * smem > (size_t)kCuLdsBytes ? 1 : 2;
  const int waves = (a.n_vrows + RW - 1) / RW;
  int grid = (waves + 7) / 8;
  if (grid > per_cu * num_cus) grid = per_cu * num_cus;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(512), smem, st, a, ncols);
  return hipGetLastError();
}

template <int QT, int NC>
hipError_t launch_xcols_nc(const GemvArgs& a, int ncols, int num_cus, hipStream_t st) {
  const int nunits = a.K / QTraits<QT>::UNIT;
  if (nunits <= 16) return launch_xcols_k<QT, NC, 16, 1>(a, ncols, num_cus, st);
  if (nunits <= 32) return launch_xcols_k<QT, NC, 32, 1>(a, ncols, num_cus, st);
  if (nunits <= 64) return launch_xcols_k<QT, NC, 64, 1>(a, ncols, num_cus, st);
  if constexpr (QTraits<QT>::UNIT == 64) {
    if (nunits <= 128) return launch_xcols_k<QT, NC, 64, 2>(a, ncols, num_cus, st);
  }
  // K > 8192: LDS holds four columns at most
  if constexpr (NC > 4) {
    return hipErrorInvalidValue;
  } else if constexpr (QTraits<QT>::UNIT == 128) {
    return launch_xcols_k<QT, NC, 64, 2>(a, ncols, num_cus, st);
  } else {
    if (nunits <= 192) return launch_xcols_k<QT, NC, 64, 3>(a, ncols, num_cus, st);
    return launch_xcols_k<QT, NC, 64, 4>(a, ncols, num_cus, st);
  }
}

template <int QT>
hipError_t launch_xcols(const GemvArgs& a, int ncols, int num_cus, hipStream_t st) {
  if (ncols <= 2) return launch_xcols_nc<QT, 2>(a, ncols, num_cus, st);
  if (ncols <= 4) return launch_xcols_nc<QT, 4>(a, ncols, num_cus, st);
  return launch_xcols_nc<QT, 8>(a, ncols, num_cus, st);
}

}  // namespace
