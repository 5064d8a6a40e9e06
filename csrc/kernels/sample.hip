// Token sampler: temperature + Gumbel-max over the
// vocabulary (or one tensor-parallel vocab shard: col_offset + out_val let the
// caller take the max over shards, Gumbel-max being decomposable), greedy when temperature <= 0. Several workgroups
// per row, each on a run of columns, then a merge (few rows leave CUs idle: 1 row of 128256 28 us on one
// workgroup, 7 on 32 and the merge, captured back to back, 5.7 + 4.5 within a decode step; 64 rows 30 -> 13, 15.4 + 5.1);
// each thread keeps a (value, index) pair over a grid-stride of the vocab with
// 16-B loads, then a wave + LDS argmax. The noise is a counter-based hash of
// (seed[row], position[row], column), so a captured hipGraph replays to the
// same tokens and the kernel needs no RNG state on the device.
#include "common.h"
#include "kernels.h"
#include "sample.h"

namespace oamd {

template <typename T>
__device__ __forceinline__ float load_logit(const T* p, int64_t i);
template <>
__device__ __forceinline__ float load_logit<float>(const float* p, int64_t i) { return p[i]; }
template <>
__device__ __forceinline__ float load_logit<bf16_t>(const bf16_t* p, int64_t i) { return bf2f(p[i]); }

// Columns [a, b) vectors of 16 bytes and [sa, sb) of a row to fp32, by the whole workgroup. A step's given rows leave through the sampler, which
// is in their step anyway, and not through a launch of their own behind it, which with its gap cost a step 12 us (one row, 4 layers of 4096: 537 us a
// step and 532).
template <typename T, int NT>
__device__ __forceinline__ void copy_f32(const T* lr, float* yr, int a, int b, int sa, int sb, bool vec) {
  constexpr int VEC = 16 / static_cast<int>(sizeof(T)), UNR = 4;
  const uint4* lv = reinterpret_cast<const uint4*>(lr);
  auto put = [&](const uint4& raw, int v) {
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
    f32x4 o[VEC / 4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if constexpr (sizeof(T) == 2) {
        o[k / 2][2 * (k & 1)] = __uint_as_float(w[k] << 16);
        o[k / 2][2 * (k & 1) + 1] = __uint_as_float(w[k] & 0xffff0000u);
      } else {
        o[0][k] = __uint_as_float(w[k]);
      }
    }
    if (vec) {
#pragma unroll
      for (int k = 0; k < VEC / 4; ++k) *reinterpret_cast<f32x4*>(yr + VEC * v + 4 * k) = o[k];
    } else {
#pragma unroll
      for (int k = 0; k < VEC; ++k) yr[VEC * v + k] = o[k / 4][k & 3];
    }
  };
  int v = a + threadIdx.x;
  for (; v + (UNR - 1) * NT < b; v += UNR * NT) {
    uint4 raw[UNR];
#pragma unroll
    for (int u = 0; u < UNR; ++u) raw[u] = lv[v + u * NT];
#pragma unroll
    for (int u = 0; u < UNR; ++u) put(raw[u], v + u * NT);
  }
  for (; v < b; v += NT) put(lv[v], v);
  for (int i = sa + threadIdx.x; i < sb; i += NT) yr[i] = load_logit<T>(lr, i);
}

// PARTS: workgroup blockIdx.y of gridDim.y, its best (value in base-2 units, column) to part
template <typename T, int NT, bool PARTS>
__global__ void __launch_bounds__(NT) sample_kernel(const T* __restrict__ logits, int64_t stride, int vocab,
                                                      const float* __restrict__ temperature,
                                                      const int64_t* __restrict__ seeds,
                                                      const int64_t* __restrict__ positions,
                                                      int64_t* __restrict__ out_tokens, int64_t col_offset,
                                                      float* __restrict__ out_val, float2* __restrict__ part, GivenRows given) {
  __shared__ float sv[NT / 64];
  __shared__ int si[NT / 64];
  const int row = blockIdx.x;
  const T* lr = logits + row * stride;
  const float temp = temperature[row];
  // 16-B loads over the aligned body of the row (8 bf16 / 4 fp32 per lane), scalar tail: this workgroup's vectors [va, nv) and its
  // share [sa, sb) of the tail, which is the whole row when that is misaligned
  constexpr int VEC = 16 / static_cast<int>(sizeof(T));
  const int all = (reinterpret_cast<uintptr_t>(lr) & 15) == 0 ? vocab / VEC : 0;
  const int py = PARTS ? blockIdx.y : 0, np = PARTS ? gridDim.y : 1;
  const int va = (int)((int64_t)all * py / np), nv = (int)((int64_t)all * (py + 1) / np);
  const int ta = all * VEC, tail = vocab - ta, sa = ta + (int)((int64_t)tail * py / np), sb = ta + (int)((int64_t)tail * (py + 1) / np);
  if (no_sample(temp)) {
    if (given.out != nullptr) {
      float* const to = reinterpret_cast<float*>(given.out[0]);
      const int64_t d = given.dst[row];
      if (to != nullptr && d >= 0 && d < given.out[1])
        copy_f32<T, NT>(lr, to + d * vocab, va, nv, sa, sb, vocab % 4 == 0 && reinterpret_cast<uintptr_t>(to) % 16 == 0);
    }
    if (!PARTS && threadIdx.x == 0) {
      out_tokens[row] = col_offset;
      if (out_val) out_val[row] = 0.f;
    }
    return;
  }
  const bool greedy = !(temp > 0.f);
  // Perturbed values are compared in base 2: x/T - ln(-ln u) = ln2 * (x log2e / T -
  // log2(-log2 u)) - ln(ln2), a monotone map, so the loop pays one FMA and two v_log_f32
  // per column and the winner is mapped back once (out_val stays in natural units).
  constexpr float kLog2e = 1.4426950408889634f, kLn2 = 0.6931471805599453f, kNegLnLn2 = 0.36651292058166435f;
  const float inv_t = greedy ? 1.f : kLog2e / temp;
  const uint64_t key = mix64((static_cast<uint64_t>(seeds[row]) * 0x9E3779B97F4A7C15ULL) ^
                             (static_cast<uint64_t>(positions[row]) << 32));
  const uint32_t k1 = static_cast<uint32_t>(key), k2 = static_cast<uint32_t>(key >> 32);
  const uint32_t c0 = static_cast<uint32_t>(col_offset);
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  auto visit = [&](float x, int i) {
    if (!greedy) {
      const float u = uniform01(hash_col(c0 + static_cast<uint32_t>(i), k1, k2));
      // -log2(u) >= 8.6e-8 exactly; the clamp only guards a hardware log rounding to 0
      x = x * inv_t - __builtin_amdgcn_logf(fmaxf(-__builtin_amdgcn_logf(u), 5.9604645e-8f));
    }
    argmax_merge(bv, bi, x, i);
  };
  // argmax_merge is a total order (value, then smaller index), so the visiting order
  // does not change the result.
  auto visit16 = [&](const uint4& raw, int v) {
    const uint32_t wv[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if constexpr (sizeof(T) == 2) {
        visit(__uint_as_float(wv[k] << 16), VEC * v + 2 * k);
        visit(__uint_as_float(wv[k] & 0xffff0000u), VEC * v + 2 * k + 1);
      } else {
        visit(__uint_as_float(wv[k]), VEC * v + k);
      }
    }
  };
  // UNR row vectors per thread requested before any is consumed: one dependent HBM round
  // trip per UNR vectors instead of per vector (the loop was latency-bound: ~16 trips
  // of 16 B per thread for a 128k vocab row)
  constexpr int UNR = 4;
  const uint4* lv = reinterpret_cast<const uint4*>(lr);
  constexpr int step = NT;
  int v0 = va + threadIdx.x;
  for (; v0 + (UNR - 1) * step < nv; v0 += UNR * step) {
    uint4 raw[UNR];
#pragma unroll
    for (int u = 0; u < UNR; ++u) raw[u] = lv[v0 + u * step];
#pragma unroll
    for (int u = 0; u < UNR; ++u) visit16(raw[u], v0 + u * step);
  }
  for (int v = v0; v < nv; v += step) visit16(lv[v], v);
  for (int i = sa + threadIdx.x; i < sb; i += NT) visit(load_logit<T>(lr, i), i);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(bv, o, kWave);
    const int oi = __shfl_xor(bi, o, kWave);
    argmax_merge(bv, bi, ov, oi);
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) { sv[w] = bv; si[w] = bi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    float v = sv[0];
    int id = si[0];
    for (int j = 1; j < NT / 64; ++j) argmax_merge(v, id, sv[j], si[j]);
    if constexpr (PARTS) {
      part[row * gridDim.y + blockIdx.y] = make_float2(v, __int_as_float(id));
    } else {
      out_tokens[row] = ((id == 0x7fffffff) ? 0 : id) + col_offset;
      if (out_val) out_val[row] = greedy ? v : v * kLn2 + kNegLnLn2;
    }
  }
}

// One wave per row: the best of its parts.
__global__ void __launch_bounds__(256) sample_merge_kernel(const float2* __restrict__ part, int rows, int parts,
                                                           const float* __restrict__ temperature, int64_t* __restrict__ out_tokens,
                                                           int64_t col_offset, float* __restrict__ out_val) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= rows) return;
  float v = -INFINITY;
  int id = 0x7fffffff;
  const bool skip = no_sample(temperature[row]);   // its parts were not written
  if (skip) v = 0.f;
  else if (lane < parts) {
    const float2 p = part[row * parts + lane];
    argmax_merge(v, id, p.x, __float_as_int(p.y));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(v, o, kWave);
    const int oi = __shfl_xor(id, o, kWave);
    argmax_merge(v, id, ov, oi);
  }
  if (lane == 0) {
    out_tokens[row] = ((id == 0x7fffffff) ? 0 : id) + col_offset;
    if (out_val) out_val[row] = temperature[row] > 0.f ? v * 0.6931471805599453f + 0.36651292058166435f : v;
  }
}

// Workgroups per row: up to eight per CU in all, 2048 columns each at least, where they gain more than the merge kernel
// costs (captured, one workgroup against several): 16384 columns 1 row 6.7 us against 5.7, 64 rows 7.3 and 6.6 (12288: 6.1 and
// 6.6); 32000 columns 128 rows 13.7 and 11.0 (20480: 7.9 and 8.2); 100000 columns 192 rows 25.0 and 22.2 (65536: 18.2 and 21.6).
// More rows fill the GPU with one each (128256 columns, 240 rows: 31.7 and 34.5).
int sample_parts(int rows, int vocab) {
  if (rows > 224 || vocab < (rows <= 64 ? 16384 : rows <= 160 ? 28672 : 98304)) return 1;
  return max(1, min(min(32, 2048 / max(rows, 1)), vocab / 2048));
}

int sample_tokens(const void* logits, bool logits_bf16, int64_t stride, int rows, int vocab,
                  const float* temperature, const int64_t* seeds, const int64_t* positions,
                  int64_t* out_tokens, int64_t col_offset, float* out_val, float* part, bool merge, const GivenRows& given, hipStream_t stream) {
  if (rows == 0) return 0;
  const int parts = part ? sample_parts(rows, vocab) : 1;
  float2* pp = reinterpret_cast<float2*>(part);
#define OAMD_SAMPLE(T)                                                                                                              \
  if (parts > 1)                                                                                                                    \
    sample_kernel<T, 256, true><<<dim3(rows, parts), 256, 0, stream>>>(static_cast<const T*>(logits), stride, vocab, temperature,   \
                                                                       seeds, positions, out_tokens, col_offset, out_val, pp, given);      \
  else                                                                                                                              \
    sample_kernel<T, 1024, false><<<rows, 1024, 0, stream>>>(static_cast<const T*>(logits), stride, vocab, temperature, seeds,      \
                                                             positions, out_tokens, col_offset, out_val, nullptr, given)
  if (logits_bf16) {
    OAMD_SAMPLE(bf16_t);
  } else {
    OAMD_SAMPLE(float);
  }
#undef OAMD_SAMPLE
  OAMD_LAUNCH_CHECK();
  if (parts > 1 && merge) {
    sample_merge_kernel<<<(rows + 3) / 4, 256, 0, stream>>>(pp, rows, parts, temperature, out_tokens, col_offset, out_val);
    OAMD_LAUNCH_CHECK();
  }
  return 0;
}

}  // namespace oamd
