// Shared by the sampler (sample.hip) and the decode step's state advance (norm_act.hip), which takes the best of a row's candidates.
#pragma once
#include "common.h"
#include "kernels.h"

namespace oamd {

// The larger value, of equal ones the smaller index.
__device__ __forceinline__ void argmax_merge(float& bv, int& bi, float v, int i) {
  if (v > bv || (v == bv && i < bi)) { bv = v; bi = i; }
}

// Rows whose token nobody reads (given tokens, the padding rows of a bucket) carry this NaN as their temperature: they get
// token 0 and their logits are not read (256 rows of 128256: 36 us, 5 when all are skipped). Any other NaN is greedy, as ever.
__device__ __forceinline__ bool no_sample(float temperature) { return __float_as_uint(temperature) == kNoSampleBits; }

}  // namespace oamd
