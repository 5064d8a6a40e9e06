// What the fp32 products share (f32.hip, gemm_f32_split.hip).
#pragma once

#include "common.h"

namespace oamd {

struct GemmF32 {
  const float *X, *W;
  float *Y, *P;          // P: slabs [S][M][N] of S > 1 K slices
  int M, N, K, S;
  int64_t ldx, ldy, xh, yh;   // row strides; head strides of X and Y (one product per head, W [H][N][K])
  const int* gtab;
  const float* rscale;
  GluAct act;
  int vec;               // Y takes 16-B stores
};

__device__ __forceinline__ float glu1(float g, float u, const GluAct& act) {
  return g / (1.f + expf(-g * __builtin_fmaf(act.c, g * g, act.a))) * u;
}

// 4 neighbouring outputs of a row, n valid ones
__device__ __forceinline__ void put4(float* y, const f32x4& v, int n, bool vec) {
  if (n >= 4 && vec) {
    *reinterpret_cast<f32x4*>(y) = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < n) y[e] = v[e];
  }
}

int gemm_f32_split(const GemmF32& a, bool glu, int rows, hipStream_t stream);   // rows of a tile: 64, 128 or 256

int sum_f32_slabs(const float* P, float* Y, int S, int M, int N, int ldy, hipStream_t stream);   // f32.hip

}  // namespace oamd
