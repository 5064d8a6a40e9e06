// RMSNorm (+ fused residual add), SiLU-and-mul, embedding gather.
//
// These are the memory-bound elementwise/normalisation ops of the explanation
// model. All bf16 traffic is 16 B per lane.
#include "common.h"
#include "kernels.h"
#include "sample.h"

namespace oamd {

// One 256-thread block per row. Each thread owns up to MAXV vectors of 8 bf16
// kept in registers between the reduction and the scaling pass, so the row is
// read from HBM exactly once (x, and residual when fused).
// With `xp` set, x is not read: the row is the bf16 rounding of the sum of S
// fp32 split-K slabs xp[s * slab + row * hidden + c] written by gemm_decode —
// the GEMM's reduction pass is folded into this kernel (same numerics: the
// projection output is rounded to bf16 once, then added to the residual).
// SC = compile-time slab count (0: runtime S) so the S slab loads of a vector are
// all issued before the first add (a runtime-trip-count loop waits for each load
// in turn: S dependent L2/HBM round trips per vector).
// Q8: the row goes out as e4m3fn with its scale amax / 448 instead of bf16, as quantize_fp8_rows makes them of the bf16
// row: an fp8 projection's input needs no second pass (64 rows of 8192 from 2 slabs: 7.4 + 4.6 us -> 8.0).
template <int NT, int MAXV, int SC, bool Q8 = false>
__global__ void __launch_bounds__(NT) rmsnorm_kernel(
    const bf16_t* __restrict__ x, bf16_t* __restrict__ residual,
    const bf16_t* __restrict__ w, bf16_t* __restrict__ y, int hidden,
    int64_t x_stride, int64_t r_stride, int64_t y_stride, float eps,
    const float* __restrict__ xp, int S_rt, int64_t slab, uint8_t* __restrict__ q = nullptr, float* __restrict__ sx = nullptr) {
  const int S = SC > 0 ? SC : S_rt;
  __shared__ float scratch[NT / 64];
  const int row = blockIdx.x;
  const int nvec = hidden >> 3;
  const u16x8* xr = reinterpret_cast<const u16x8*>(x + row * x_stride);
  u16x8* rr = residual ? reinterpret_cast<u16x8*>(residual + row * r_stride) : nullptr;
  float v[MAXV][8];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int vi = threadIdx.x + i * NT;
    if (vi < nvec) {
      u16x8 a;
      if (xp) {
        const float* pr = xp + (int64_t)row * hidden + vi * 8;
        f32x4 lo = *reinterpret_cast<const f32x4*>(pr), hi = *reinterpret_cast<const f32x4*>(pr + 4);
        if constexpr (SC > 0) {
          f32x4 pl[SC > 1 ? SC - 1 : 1], ph[SC > 1 ? SC - 1 : 1];
#pragma unroll
          for (int sp = 1; sp < SC; ++sp) {
            pl[sp - 1] = *reinterpret_cast<const f32x4*>(pr + sp * slab);
            ph[sp - 1] = *reinterpret_cast<const f32x4*>(pr + sp * slab + 4);
          }
#pragma unroll
          for (int sp = 1; sp < SC; ++sp) {
            lo += pl[sp - 1];
            hi += ph[sp - 1];
          }
        } else {
#pragma unroll 4
          for (int sp = 1; sp < S; ++sp) {
            lo += *reinterpret_cast<const f32x4*>(pr + sp * slab);
            hi += *reinterpret_cast<const f32x4*>(pr + sp * slab + 4);
          }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          a[j] = f2bf(lo[j]);
          a[4 + j] = f2bf(hi[j]);
        }
      } else {
        a = xr[vi];
      }
      if (rr) {
        u16x8 b = rr[vi];
        u16x8 s;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          // residual stream is bf16: round the sum before normalising it
          s[j] = f2bf(bf2f(a[j]) + bf2f(b[j]));
        }
        rr[vi] = s;
        a = s;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[i][j] = bf2f(a[j]);
        ss += v[i][j] * v[i][j];
      }
    }
  }
  // the weight vectors are requested before the block reduction, so their round trip
  // overlaps the barrier instead of following it
  const u16x8* wr = reinterpret_cast<const u16x8*>(w);
  u16x8 wpre[MAXV];
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int vi = threadIdx.x + i * NT;
    if (vi < nvec) wpre[i] = wr[vi];
  }
  const float tot = block_sum<NT>(ss, scratch);
  const float rs = rsqrtf(tot / static_cast<float>(hidden) + eps);
  if constexpr (Q8) {
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < MAXV; ++i) {
      if (threadIdx.x + i * NT < nvec) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          v[i][j] = bf2f(f2bf(bf2f(f2bf(v[i][j] * rs)) * bf2f(wpre[i][j])));
          amax = fmaxf(amax, fabsf(v[i][j]));
        }
      }
    }
    amax = wave_max(amax);
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = amax;   // block_sum ended in a barrier
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) amax = fmaxf(amax, scratch[i]);
    const float s = amax > 0.f ? amax / 448.f : 1.f;
    const float inv = 1.f / s;
    if (threadIdx.x == 0) sx[row] = s;
    uint2* qr = reinterpret_cast<uint2*>(q + (int64_t)row * hidden);
#pragma unroll
    for (int i = 0; i < MAXV; ++i) {
      const int vi = threadIdx.x + i * NT;
      if (vi < nvec) qr[vi] = pack_fp8x8(v[i], inv);
    }
    return;
  }
  // y_stride < 0: y is written in the fragment-major tiled layout that gemm_xr reads its
  // activations from (common.h xr_tiled_off; one block per row, rows % 16 == 0)
  const bool tiled = y_stride < 0;
  u16x8* yr = reinterpret_cast<u16x8*>(y + (tiled ? 0 : row * y_stride));
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int vi = threadIdx.x + i * NT;
    if (vi < nvec) {
      const u16x8 wv = wpre[i];
      u16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        // HF semantics: normalised value is rounded to bf16, then scaled by w
        o[j] = f2bf(bf2f(f2bf(v[i][j] * rs)) * bf2f(wv[j]));
      }
      if (tiled) {
        *reinterpret_cast<u16x8*>(y + xr_tiled_off(row, vi * 8, gridDim.x)) = o;
      } else {
        yr[vi] = o;
      }
    }
  }
}

template <bool Q8>
static void rmsnorm_launch(const bf16_t* x, bf16_t* residual, const bf16_t* w, bf16_t* y, int rows, int hidden, int64_t x_stride,
                           int64_t r_stride, int64_t y_stride, float eps, const float* xp, int S, uint8_t* q, float* sx,
                           hipStream_t stream) {
  constexpr int NT = 256;
  const int nvec = hidden / 8;
  const int64_t slab = (int64_t)rows * hidden;
  const int sc = xp == nullptr ? 1 : S;
#define OAMD_RMS(NTH, MV, SCC) \
  rmsnorm_kernel<NTH, MV, SCC, Q8><<<rows, NTH, 0, stream>>>(x, residual, w, y, hidden, x_stride, r_stride, y_stride, eps, xp, S, slab, q, sx)
#define OAMD_RMS_S(NTH, MV)                  \
  switch (sc) {                              \
    case 1: OAMD_RMS(NTH, MV, 1); break;     \
    case 2: OAMD_RMS(NTH, MV, 2); break;     \
    case 4: OAMD_RMS(NTH, MV, 4); break;     \
    case 8: OAMD_RMS(NTH, MV, 8); break;     \
    default: OAMD_RMS(NTH, MV, 0); break;    \
  }
  // split-K slab sums of rows up to 4096 wide: 512 threads, one vector each, so a row's
  // slab loads all leave in one round (OAMD_RMS_WIDE=0: 256 threads x 2 vectors)
  static const bool wide = [] { const char* e = getenv("OAMD_RMS_WIDE"); return !(e && e[0] == '0'); }();
  if (wide && xp != nullptr && sc > 1 && nvec > NT && nvec <= 2 * NT) {
    OAMD_RMS_S(2 * NT, 1)
  } else if (nvec <= NT * 2) {
    OAMD_RMS_S(NT, 2)
  } else if (nvec <= NT * 4) {
    OAMD_RMS_S(NT, 4)
  } else {
    OAMD_RMS_S(NT, 8)
  }
#undef OAMD_RMS_S
#undef OAMD_RMS
}

int rmsnorm(const bf16_t* x, bf16_t* residual, const bf16_t* w, bf16_t* y,
            int rows, int hidden, int64_t x_stride, int64_t r_stride,
            int64_t y_stride, float eps, const float* xp, int S, hipStream_t stream) {
  if (rows == 0) return 0;
  rmsnorm_launch<false>(x, residual, w, y, rows, hidden, x_stride, r_stride, y_stride, eps, xp, S, nullptr, nullptr, stream);
  OAMD_LAUNCH_CHECK();
  return 0;
}

int rmsnorm_fp8(const bf16_t* x, bf16_t* residual, const bf16_t* w, uint8_t* q, float* sx, int rows, int hidden, int64_t x_stride,
                int64_t r_stride, float eps, const float* xp, int S, hipStream_t stream) {
  if (rows == 0) return 0;
  rmsnorm_launch<true>(x, residual, w, nullptr, rows, hidden, x_stride, r_stride, 0, eps, xp, S, q, sx, stream);
  OAMD_LAUNCH_CHECK();
  return 0;
}

// out[m, i] = act(gate) * up; grid-stride over 8-element vectors. gate|up
// columns are interleaved in blocks of `block` features (block == inter: the
// plain [gate | up] concatenation): gate of feature i at (i / block) * 2 * block
// + i % block, up `block` columns later.
__global__ void silu_mul_kernel(const bf16_t* __restrict__ gu, bf16_t* __restrict__ out,
                                int64_t rows, int inter, int block, int64_t in_stride, int64_t out_stride, GluAct act) {
  const int vpr = inter >> 3;
  const int64_t total = rows * vpr;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t m = idx / vpr;
    const int c = static_cast<int>(idx - m * vpr) << 3;
    const int gc = (c / block) * 2 * block + c % block;
    const u16x8 g = *reinterpret_cast<const u16x8*>(gu + m * in_stride + gc);
    const u16x8 u = *reinterpret_cast<const u16x8*>(gu + m * in_stride + gc + block);
    u16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float gf = bf2f(g[j]);
      // HF: act(gate) rounded to bf16, then multiplied by up in bf16
      const float s = bf2f(f2bf(glu_gate(gf, act)));
      o[j] = f2bf(s * bf2f(u[j]));
    }
    *reinterpret_cast<u16x8*>(out + m * out_stride + c) = o;
  }
}

int silu_mul(const bf16_t* gu, bf16_t* out, int64_t rows, int inter, int block,
             int64_t in_stride, int64_t out_stride, int glu, hipStream_t stream) {
  if (rows == 0) return 0;
  if (block <= 0 || block % 8 != 0 || inter % block != 0) return -1;
  const int64_t total = rows * (inter / 8);
  const int nt = 256;
  int64_t blocks = (total + nt - 1) / nt;
  if (blocks > 256 * 16) blocks = 256 * 16;
  silu_mul_kernel<<<static_cast<int>(blocks), nt, 0, stream>>>(gu, out, rows, inter, block, in_stride,
                                                               out_stride, glu_act(glu));
  OAMD_LAUNCH_CHECK();
  return 0;
}

// Row gather: out[t, :] = table[ids[t], :]. One block per token, 16 B per lane.
__global__ void embedding_kernel(const int64_t* __restrict__ ids, const bf16_t* __restrict__ table,
                                 bf16_t* __restrict__ out, int hidden, int64_t vocab) {
  const int t = blockIdx.x;
  int64_t id = ids[t];
  if (id < 0 || id >= vocab) id = 0;  // out-of-range ids are clamped, never read OOB
  const u16x8* src = reinterpret_cast<const u16x8*>(table + id * hidden);
  u16x8* dst = reinterpret_cast<u16x8*>(out + (int64_t)t * hidden);
  for (int i = threadIdx.x; i < (hidden >> 3); i += blockDim.x) dst[i] = src[i];
}

int embedding(const int64_t* ids, const bf16_t* table, bf16_t* out, int tokens,
              int hidden, int64_t vocab, hipStream_t stream) {
  if (tokens == 0) return 0;
  embedding_kernel<<<tokens, 256, 0, stream>>>(ids, table, out, hidden, vocab);
  OAMD_LAUNCH_CHECK();
  return 0;
}

// Decode-step bookkeeping of a hipGraph-captured step (engine/llm.py _DecodeGraph), one
// thread per batch row instead of ~15 one-op torch kernels:
//   decode_slots:   slot = page(bt[row], pos / P) * P + pos % P for live rows (ctx > 0), else -1;
//                   spos = pos + 1 (the sampler's stream position)
//   decode_advance: ids = tok; hist[row, step % ms] = tok; live rows pos += 1, ctx += 1; then
//                   (one thread) step += 1. With parts, tok is the best of a row's sampling candidates (sample.hip); with bt, slots
//                   and spos become the next step's, as decode_slots has them.
// The engine writes the first step's slots itself, so a step has one launch behind its sampler instead of two and one in front of it (one row, 4 layers
// of 4096: 538 us a step and 537; 2 rows of 4 layers of 2048 273 and 270).
__device__ __forceinline__ int64_t decode_slot(const int* bt, int r, int64_t p, int ctx, int max_pages, int page_size) {
  int64_t pg = p / page_size;
  pg = pg < max_pages - 1 ? pg : max_pages - 1;
  return ctx > 0 ? (int64_t)bt[(int64_t)r * max_pages + pg] * page_size + p % page_size : -1;
}

__global__ void decode_slots_kernel(const int* __restrict__ bt, const int64_t* __restrict__ pos,
                                    const int* __restrict__ ctx, int64_t* __restrict__ slots,
                                    int64_t* __restrict__ spos, int B, int max_pages, int page_size) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= B) return;
  const int64_t p = pos[r];
  slots[r] = decode_slot(bt, r, p, ctx[r], max_pages, page_size);
  spos[r] = p + 1;
}

__global__ void __launch_bounds__(1024) decode_advance_kernel(const DecodeAdvance a) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  int64_t* const step = a.step;
  if (r < a.B) {
    int c = a.ctx[r];
    int64_t p = a.pos[r], t;
    if (a.parts > 0) {
      float v = -INFINITY;
      int id = 0x7fffffff;
      if (!no_sample(a.temperature[r])) {   // its candidates were not written
        const float2* q = a.part + (int64_t)r * a.parts;
#pragma unroll 8
        for (int i = 0; i < a.parts; ++i) argmax_merge(v, id, q[i].x, __float_as_int(q[i].y));
      }
      t = id == 0x7fffffff ? 0 : id;
    } else {
      t = a.tok[r];
    }
    a.ids[r] = t;
    a.hist[(int64_t)r * a.ms + (int)(step[0] % a.ms)] = t;
    if (c > 0) {
      a.pos[r] = ++p;
      a.ctx[r] = ++c;
    }
    if (a.bt != nullptr) {
      a.slots[r] = decode_slot(a.bt, r, p, c, a.max_pages, a.page_size);
      a.spos[r] = p + 1;
    }
  }
  __syncthreads();
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    // every block read step[0] before block 0's thread 0 bumps it: one block covers all rows
    step[0] += 1;
    if (a.out != nullptr) a.out[0] = 0;
  }
}

int decode_slots(const int* bt, const int64_t* pos, const int* ctx, int64_t* slots, int64_t* spos, int B,
                 int max_pages, int page_size, hipStream_t stream) {
  if (B <= 0) return 0;
  if (B > 1024) return -1;
  decode_slots_kernel<<<1, 1024, 0, stream>>>(bt, pos, ctx, slots, spos, B, max_pages, page_size);
  OAMD_LAUNCH_CHECK();
  return 0;
}

int decode_advance(const DecodeAdvance& a, hipStream_t stream) {
  if (a.B <= 0) return 0;
  if (a.B > 1024) return -1;   // one block: every row reads step before it is bumped
  decode_advance_kernel<<<1, 1024, 0, stream>>>(a);
  OAMD_LAUNCH_CHECK();
  return 0;
}

// out[dst[r]] = fp32 of row r: a decode step's logits, in the caller's order. Bound by memory: one 2-byte read and
// one 4-byte write per element (256 x 128256: 32 us within a decode step, 6.2 TB/s, against 125 for a conversion pass and an indexed copy).
template <typename T>
__global__ void __launch_bounds__(256) scatter_rows_f32_kernel(const T* __restrict__ x, int64_t ld, const int* __restrict__ dst,
                                                               float* __restrict__ out, int n_out, int cols, bool vec) {
  const int d = dst[blockIdx.y];
  if (d < 0 || d >= n_out) return;
  const T* xr = x + blockIdx.y * ld;
  float* yr = out + (int64_t)d * cols;
  const int c = (blockIdx.x * 256 + threadIdx.x) * 8;
  auto val = [&](int i) {
    if constexpr (sizeof(T) == 2) return bf2f(xr[i]);
    else return xr[i];
  };
  if (vec && c + 8 <= cols) {
    f32x4 a, b;
    if constexpr (sizeof(T) == 2) {
      const u16x8 v = *reinterpret_cast<const u16x8*>(xr + c);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        a[e] = bf2f(v[e]);
        b[e] = bf2f(v[4 + e]);
      }
    } else {
      a = *reinterpret_cast<const f32x4*>(xr + c);
      b = *reinterpret_cast<const f32x4*>(xr + c + 4);
    }
    *reinterpret_cast<f32x4*>(yr + c) = a;
    *reinterpret_cast<f32x4*>(yr + c + 4) = b;
  } else {
    for (int i = c; i < min(c + 8, cols); ++i) yr[i] = val(i);
  }
}

int scatter_rows_f32(const void* x, bool bf16, int64_t ld, const int* dst, float* out, int rows, int n_out, int cols,
                     hipStream_t stream) {
  if (rows == 0 || cols == 0) return 0;
  if (rows > 65535) return -1;
  const int64_t e = bf16 ? 2 : 4;
  const bool vec = ld * e % 16 == 0 && cols % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
  const dim3 grid((cols + 2047) / 2048, rows);
  if (bf16) scatter_rows_f32_kernel<<<grid, 256, 0, stream>>>(static_cast<const bf16_t*>(x), ld, dst, out, n_out, cols, vec);
  else scatter_rows_f32_kernel<<<grid, 256, 0, stream>>>(static_cast<const float*>(x), ld, dst, out, n_out, cols, vec);
  OAMD_LAUNCH_CHECK();
  return 0;
}

}  // namespace oamd
