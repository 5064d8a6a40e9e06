// fp32 products of few rows (one to sixteen): Y[M, N] = X[M, K] W[N, K]^T, 32-bit operands, products and sums.
//
// What bounds it: the weights' stream. The 16-row fragments of the matrix unit's kernel (f32.hip) ask for 64 B of each of 16 rows at a time and
// wait for a group of them before the next. Here, as in gemm_rows.hip, a wave reads 1 KB of one row of W a request, past the caches, with two sets of rows
// in flight by turns; X stays in registers and the products are FMAs, at eight rows 18 TB/s of weights by themselves, at sixteen 6.6 to 7.6 with the sums over lanes. A lane's sum is a chain
// of at most 32 products, the rest goes over lanes and waves as a tree.
// us on gemm_f32_skinny_kernel and here (weights from HBM), one row and eight: 16384 x 2048 gated 37 -> 23, 40 -> 26 (5.9 and 5.1 TB/s); 2048 x 8192 26 -> 13,
// 33 -> 16; 32000 x 2048 58 -> 40, 62 -> 45; 28672 x 4096 gated 114 -> 72, 122 -> 75; 128256 x 4096 388 -> 309, 468 -> 325 (6.8 and 6.5); 2048 x 2048
// 7.5 -> 5.7, 9.6 -> 6.6. Sixteen rows, which the vector units bound: 16384 x 2048 gated 41 -> 33, 2048 x 8192 in four slices 37 -> 23, 32000 x 2048 77 -> 63.
#include <type_traits>

#include "common.h"
#include "gemm_f32.h"
#include "kernels.h"
#include "row_sums.h"

namespace oamd {

// A workgroup takes rows of W from f0 to f1 (GLU: of gate and up), its NW waves an equal part each of K; lane l of wave w holds the X values of its 4 columns in
// every 256 of the part. MT: rows of X, J: 256-column pieces of the part, RF: rows of W requested at a time. P: K slice blockIdx.y of gridDim.y into its slab.
template <int MT, int J, int NW, bool GLU>
__global__ void __launch_bounds__(64 * NW) gemm_f32_rows_kernel(const float* __restrict__ X, const float* __restrict__ W, float* __restrict__ Y,
                                                                float* __restrict__ P, int M, int N, int K, int ldy, GluAct act) {
  constexpr int HALVES = GLU ? 2 : 1, RF = J == 1 ? 8 : J == 2 ? 4 : J <= 4 ? 2 : 1;
  extern __shared__ float red[];   // [slot][MT][wave, its 16 lanes]
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int units = N / HALVES;
  const int f0 = (int)((int64_t)units * blockIdx.x / gridDim.x), nf = (int)((int64_t)units * (blockIdx.x + 1) / gridDim.x) - f0;
  const int n = nf * HALVES, Kw = K / gridDim.y / NW, k0 = (blockIdx.y * NW + w) * Kw;
  const bool tail = ((J - 1) * 64 + lane) * 4 < Kw;   // this lane has columns in the last piece
  auto col = [&](int j) { return k0 + (j < J - 1 || tail ? (j * 64 + lane) * 4 : 0); };
  struct Rows { f32x4 v[RF][J]; } even, odd;
  auto load = [&](Rows& r, int s0) {
#pragma unroll
    for (int i = 0; i < RF; ++i) {
      const int s = min(s0 + i, n - 1), f = f0 + s / HALVES;
      const float* p = W + (int64_t)(GLU ? (f >> 6) * 128 + (f & 63) + (s & 1) * 64 : f) * K;
#pragma unroll
      for (int j = 0; j < J; ++j) r.v[i][j] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p + col(j)));
    }
  };
  auto clear = [&](f32x4& v) {   // where the last piece has no columns both operands are 0
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = tail ? v[e] : 0.f;
  };
  f32x4 x[MT][J];   // requested in front of the first rows: their loop waits for none of its own loads
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int j = 0; j < J; ++j) x[m][j] = *reinterpret_cast<const f32x4*>(X + (int64_t)min(m, M - 1) * K + col(j));
  load(even, 0);
  load(odd, RF);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int m = 0; m < MT; ++m) clear(x[m][J - 1]);
  auto mul = [&](Rows& r, int s0) {
    float t[RF];
#pragma unroll
    for (int i = 0; i < RF; ++i) {
      clear(r.v[i][J - 1]);
      float a[MT] = {};
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int m = 0; m < MT; ++m) a[m] = __builtin_fmaf(r.v[i][j][e], x[m][j][e], a[m]);
      t[i] = sums16<MT>(a, lane);
    }
    load(r, s0 + 2 * RF);
    if ((lane & 15) >= 16 - MT)
#pragma unroll
      for (int i = 0; i < RF; ++i) red[((s0 + i) * MT + (lane & (MT - 1))) * 4 * NW + 4 * w + (lane >> 4)] = t[i];
  };
  int s = 0;
  for (; s + RF < n; s += 2 * RF) {
    mul(even, s);
    mul(odd, s + RF);
  }
  if (s < n) mul(even, s);
  __syncthreads();
  auto sum = [&](int slot, int m) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(red + (slot * MT + m) * 4 * NW + 4 * i);
      t += (v[0] + v[1]) + (v[2] + v[3]);
    }
    return t;
  };
  for (int e = threadIdx.x; e < nf * M; e += 64 * NW) {
    const int m = e / nf, f = e % nf;
    if (!GLU && P != nullptr) P[((int64_t)blockIdx.y * M + m) * N + f0 + f] = sum(f, m);
    else Y[(int64_t)m * ldy + f0 + f] = GLU ? glu1(sum(2 * f, m), sum(2 * f + 1, m), act) : sum(f, m);
  }
}

template <int MT, int J, int NW>
static int launch(const float* X, const float* W, float* Y, float* P, int S, int M, int N, int K, int ldy, int glu, int blocks, hipStream_t stream) {
  // four waves where their registers hold X; else eight
  if constexpr (MT * J > 32 || (NW == 8 && 2 * J <= 8 && MT * 2 * J <= 32)) {
    return -1;
  } else {
    constexpr int RF = J == 1 ? 8 : J == 2 ? 4 : 2;
    const int units = glu ? N / 2 : N, most = (units + blocks - 1) / blocks * (glu ? 2 : 1) + RF;   // slots, and what the last rows run over
    const size_t lds = (size_t)most * MT * 16 * NW;
    if (lds > (48 << 10)) return -4;
    if (glu) gemm_f32_rows_kernel<MT, J, NW, true><<<blocks, 64 * NW, lds, stream>>>(X, W, Y, nullptr, M, N, K, ldy, glu_act(glu));
    else gemm_f32_rows_kernel<MT, J, NW, false><<<dim3(blocks, S), 64 * NW, lds, stream>>>(X, W, Y, S > 1 ? P : nullptr, M, N, K, ldy, GluAct{});
    return 0;
  }
}

// waves of a workgroup: as many as hold X's part of M rows in their registers, 0: K is too long
int f32_rows_waves(int M, int K) {
  const int mt = M > 8 ? 16 : M > 4 ? 8 : M > 2 ? 4 : M;
  for (int nw = 4; nw <= 8; nw += 4) {
    const int J = (K / nw + 255) / 256;
    if (K % (4 * nw) == 0 && J <= 8 && mt * J <= 32) return nw;
  }
  return 0;
}

int gemm_f32_rows(const float* X, const float* W, float* Y, float* P, int S, int M, int N, int K, int ldy, int glu, int blocks, hipStream_t stream) {
  if (M < 1 || M > 16 || N < 1 || K < 16 || blocks < 1 || ldy < (glu ? N / 2 : N)) return -1;
  if (S < 1 || S > 8 || K % (16 * S) || (S > 1 && (P == nullptr || glu || N % 4))) return -4;
  if (glu && N % 128) return -2;
  const int nw = f32_rows_waves(M, K / S);
  if (!nw) return -3;
  blocks = min(blocks, glu ? N / 2 : N);
  const int J = (K / S / nw + 255) / 256;
  auto run = [&](auto mt, auto waves) {
    constexpr int MT = decltype(mt)::value, NW = decltype(waves)::value;
    switch (J) {
      case 1: return launch<MT, 1, NW>(X, W, Y, P, S, M, N, K, ldy, glu, blocks, stream);
      case 2: return launch<MT, 2, NW>(X, W, Y, P, S, M, N, K, ldy, glu, blocks, stream);
      case 3: return launch<MT, 3, NW>(X, W, Y, P, S, M, N, K, ldy, glu, blocks, stream);
      case 4: return launch<MT, 4, NW>(X, W, Y, P, S, M, N, K, ldy, glu, blocks, stream);
      case 5: return launch<MT, 5, NW>(X, W, Y, P, S, M, N, K, ldy, glu, blocks, stream);
      case 6: return launch<MT, 6, NW>(X, W, Y, P, S, M, N, K, ldy, glu, blocks, stream);
      case 7: return launch<MT, 7, NW>(X, W, Y, P, S, M, N, K, ldy, glu, blocks, stream);
      default: return launch<MT, 8, NW>(X, W, Y, P, S, M, N, K, ldy, glu, blocks, stream);
    }
  };
  auto rows = [&](auto waves) {
    return M == 1 ? run(std::integral_constant<int, 1>{}, waves) : M == 2 ? run(std::integral_constant<int, 2>{}, waves)
           : M <= 4 ? run(std::integral_constant<int, 4>{}, waves) : M <= 8 ? run(std::integral_constant<int, 8>{}, waves)
                     : run(std::integral_constant<int, 16>{}, waves);
  };
  const int rc = nw == 4 ? rows(std::integral_constant<int, 4>{}) : rows(std::integral_constant<int, 8>{});
  if (rc) return rc;
  OAMD_LAUNCH_CHECK();
  return S > 1 ? sum_f32_slabs(P, Y, S, M, N, ldy, stream) : 0;
}

}  // namespace oamd
