// Sums over lanes of the row-streaming products (gemm_rows.hip, gemm_f32_rows.hip).
#pragma once

#include "common.h"

namespace oamd {

template <int CTRL>
__device__ __forceinline__ float from(float v) {   // of the lane that CTRL names, 0 where it is none
  return __uint_as_float(__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), CTRL, 0xf, 0xf, true));
}
constexpr int kNext = 0xb1, kNext2 = 0x4e;   // quad_perm: lane ^ 1, lane ^ 2
constexpr int row_shr(int n) { return 0x110 + n; }   // lane - n of the same 16
constexpr int row_shl(int n) { return 0x100 + n; }   // lane + n
constexpr int kOther8 = 0x128;   // lane ^ 8 of the same 16 (a rotation by 8)

// MT values of every lane -> in the last MT lanes of each 16, lane l: the 16 lanes' sum of value l % MT
template <int MT>
__device__ __forceinline__ float sums16(const float (&v)[MT], int lane) {
  float r;
  if constexpr (MT == 16) {   // halve the values four times, by the lane's bits 0 to 3
    float a[8], b[4], c[2];
    const bool b0 = lane & 1, b1 = lane & 2, b2 = lane & 4, b3 = lane & 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = (b0 ? v[2 * i + 1] : v[2 * i]) + from<kNext>(b0 ? v[2 * i] : v[2 * i + 1]);
#pragma unroll
    for (int i = 0; i < 4; ++i) b[i] = (b1 ? a[2 * i + 1] : a[2 * i]) + from<kNext2>(b1 ? a[2 * i] : a[2 * i + 1]);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float hi = b[2 * i + 1] + from<row_shr(4)>(b[2 * i + 1]), lo = b[2 * i] + from<row_shl(4)>(b[2 * i]);   // every lane takes part in both
      c[i] = b2 ? hi : lo;
    }
    return (b3 ? c[1] : c[0]) + from<kOther8>(b3 ? c[0] : c[1]);
  } else if constexpr (MT == 1) {
    r = v[0] + from<kNext>(v[0]);
    r += from<kNext2>(r);
  } else {
    float h[MT / 2];
    const bool hi = lane & 1;
#pragma unroll
    for (int i = 0; i < MT / 2; ++i) h[i] = (hi ? v[2 * i + 1] : v[2 * i]) + from<kNext>(hi ? v[2 * i] : v[2 * i + 1]);
    const bool hi2 = lane & 2;
    if constexpr (MT == 2) {
      r = h[0] + from<kNext2>(h[0]);
    } else {
      r = (hi2 ? h[1] : h[0]) + from<kNext2>(hi2 ? h[0] : h[1]);
      if constexpr (MT == 8) {   // the last four lanes of eight keep values 4 to 7, and of the values 0 to 3 the lanes before those get theirs
        const float q = (hi2 ? h[3] : h[2]) + from<kNext2>(hi2 ? h[2] : h[3]);
        const float hi4 = q + from<row_shr(4)>(q), lo4 = r + from<row_shl(4)>(r);   // every lane takes part in both
        r = lane & 4 ? hi4 : lo4;
        return r + from<row_shr(8)>(r);
      }
    }
  }
  r += from<row_shr(4)>(r);
  return r + from<row_shr(8)>(r);
}

}  // namespace oamd
