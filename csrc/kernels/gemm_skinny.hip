// Skinny-M GEMM for small decode buckets: Y[M, N] = X[M, K] . W[N, K]^T with
// M <= 32 (most products of up to 8 rows go to gemm_rows.hip, whose rule is the caller's).
//
// At M = 1..32 the step is a pure weight stream (16 GB of bf16 weights per 8B
// decode step): the kernel's only job is to keep enough W bytes in flight to
// run HBM at full rate. Structure (weights straight
// to VGPRs, deep unroll, no LDS round trip):
//   * a block owns one, two or four 16-row tiles of W (skinny_tiles; for the fused SwiGLU gate rows
//     and the matching up rows 64 rows later) and its 4 waves split K;
//   * each wave streams its K range in 32-deep steps: lane l loads 16 B of W
//     row (l & 15) at k = 8 (l >> 4) -- exactly the A-fragment of
//     v_mfma_f32_16x16x32_bf16 -- and the matching 16 B of X rows (l & 15) as
//     the B-fragment (X is tiny and L2-resident); U steps are issued before
//     the first MFMA, so every wave keeps U x 1 KB of W in flight;
//   * the MFMA does the M-way reuse for free (16 output columns = 16 rows of
//     X per instruction; 2 instructions for M in 17..32) -- no cross-lane
//     shuffle reductions as in a VALU GEMV;
//   * the 4 per-wave partial tiles are summed through LDS, then stored as bf16,
//     as fp32 split-K slabs (consumed by rmsnorm / rope_kv), or through the
//     SwiGLU epilogue (HF rounding points, as gemm.hip).
// Split-K across blocks (gridDim.y = S) only adds parallelism for short-N shapes.
#include "common.h"
#include "kernels.h"

namespace oamd {

typedef __bf16 bf16x8s_t __attribute__((ext_vector_type(8)));

namespace sk {
constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
enum { kStore = 0, kPartial = 1, kSilu = 2 };
}  // namespace sk

// NT: 16-row W tiles of a block (for SwiGLU in pairs of gate and up rows), MT: 16-column X tiles (M <= 16 * MT), U: k-steps in
// flight per wave.
template <int NT, int MT, int EPI, int U>
__global__ void __launch_bounds__(sk::kThreads) gemm_skinny_kernel(const bf16_t* __restrict__ X,
                                                                 const bf16_t* __restrict__ W,
                                                                 bf16_t* __restrict__ Y, float* __restrict__ P,
                                                                 int M, int N, int K, int S, GluAct act = {}) {
  constexpr int NO = EPI == sk::kSilu ? NT / 2 : NT;   // output tiles
  __shared__ float red[sk::kWaves][NT * MT][64 * 4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = tid >> 6;
  const int r = lane & 15, kq = lane >> 4;
  // W rows of this block's tiles; SwiGLU: 16-row slices of the gate half of a 128-row group, then of its up half
  int rows[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    if constexpr (EPI == sk::kSilu) {
      const int sub = blockIdx.x * NO + t % NO;
      rows[t] = (sub >> 2) * 128 + (t / NO) * 64 + (sub & 3) * 16;
    } else {
      rows[t] = (blockIdx.x * NT + t) * 16;
    }
  }
  const int kz = blockIdx.y;
  const int Kb = K / S;             // this block's K range
  const int Kw = Kb / sk::kWaves;   // this wave's
  const int k0 = kz * Kb + w * Kw;
  const int steps = Kw / 32;

  const u16x8* wp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) wp[t] = reinterpret_cast<const u16x8*>(W + (int64_t)(rows[t] + r) * K + k0 + kq * 8);
  const u16x8* xp[MT];
  bool xv[MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int m = j * 16 + r;
    xv[j] = m < M;
    xp[j] = reinterpret_cast<const u16x8*>(X + (int64_t)(xv[j] ? m : 0) * K + k0 + kq * 8);
  }
  f32x4 acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const u16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  int s = 0;
  for (; s + U <= steps; s += U) {
    u16x8 a[U][NT], b[U][MT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int t = 0; t < NT; ++t) a[u][t] = __builtin_nontemporal_load(wp[t] + (s + u) * 4);
#pragma unroll
      for (int j = 0; j < MT; ++j) b[u][j] = xv[j] ? xp[j][(s + u) * 4] : zero;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < MT; ++j)
          acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8s_t, a[u][t]),
                                                              __builtin_bit_cast(bf16x8s_t, b[u][j]), acc[t][j], 0, 0,
                                                              0);
  }
  for (; s < steps; ++s) {  // remainder (< U steps)
    u16x8 a[NT], b[MT];
#pragma unroll
    for (int t = 0; t < NT; ++t) a[t] = __builtin_nontemporal_load(wp[t] + s * 4);
#pragma unroll
    for (int j = 0; j < MT; ++j) b[j] = xv[j] ? xp[j][s * 4] : zero;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 0; j < MT; ++j)
        acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8s_t, a[t]),
                                                            __builtin_bit_cast(bf16x8s_t, b[j]), acc[t][j], 0, 0, 0);
  }

  // ---- sum the 4 waves' partial tiles: C lane l -> W row 4 (l >> 4) + i, X row (column) l & 15
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[w][t * MT + j][i * 64 + lane] = acc[t][j][i];
  __syncthreads();
  // thread -> (output tile, X tile j, element e): 64 lanes x 4 regs per tile
  for (int e = tid; e < NO * MT * 256; e += sk::kThreads) {
    const int t = e / (MT * 256), j = (e >> 8) % MT, i = (e >> 6) & 3, l = e & 63;
    const int m = j * 16 + (l & 15);
    const int rr = 4 * (l >> 4) + i;  // row within the 16-row tile
    if (m >= M) continue;
    auto sum = [&](int tile) {
      float v = 0.f;
#pragma unroll
      for (int ww = 0; ww < sk::kWaves; ++ww) v += red[ww][tile * MT + j][i * 64 + l];
      return v;
    };
    if constexpr (EPI == sk::kSilu) {
      const float g = bf2f(f2bf(sum(t)));
      const float u = bf2f(f2bf(sum(NO + t)));
      const float sg = bf2f(f2bf(glu_gate(g, act)));
      const int f = (blockIdx.x * NO + t) * 16 + rr;
      Y[(int64_t)m * (N / 2) + f] = f2bf(sg * u);
    } else if constexpr (EPI == sk::kPartial) {
      P[((int64_t)kz * M + m) * N + (blockIdx.x * NT + t) * 16 + rr] = sum(t);
    } else {
      Y[(int64_t)m * N + (blockIdx.x * NT + t) * 16 + rr] = f2bf(sum(t));
    }
  }
}

template <int NT, int U>
static void launch_skinny(const bf16_t* X, const bf16_t* W, bf16_t* Y, float* P, int M, int N, int K, int S, int glu,
                          hipStream_t stream) {
  const dim3 grid(N / (16 * NT), S);
  if (glu) {
    if constexpr (NT > 1) {
      if (M <= 16) gemm_skinny_kernel<NT, 1, sk::kSilu, U><<<grid, sk::kThreads, 0, stream>>>(X, W, Y, P, M, N, K, 1, glu_act(glu));
      else gemm_skinny_kernel<NT, 2, sk::kSilu, U><<<grid, sk::kThreads, 0, stream>>>(X, W, Y, P, M, N, K, 1, glu_act(glu));
    }
  } else if (S > 1) {
    if (M <= 16) gemm_skinny_kernel<NT, 1, sk::kPartial, U><<<grid, sk::kThreads, 0, stream>>>(X, W, Y, P, M, N, K, S);
    else gemm_skinny_kernel<NT, 2, sk::kPartial, U><<<grid, sk::kThreads, 0, stream>>>(X, W, Y, P, M, N, K, S);
  } else {
    if (M <= 16) gemm_skinny_kernel<NT, 1, sk::kStore, U><<<grid, sk::kThreads, 0, stream>>>(X, W, Y, P, M, N, K, 1);
    else gemm_skinny_kernel<NT, 2, sk::kStore, U><<<grid, sk::kThreads, 0, stream>>>(X, W, Y, P, M, N, K, 1);
  }
}

// 16-row W tiles of a workgroup. It reads the X rows of its K range once for all of them, and a CU takes in X and W at the same rate:
// 32 rows of 128256 x 4096 429 us on one tile, 345 on two, 304 on four; 16 rows of 4096 x 14336 in 2 slices 38 on one, 30 on two
// (256 workgroups), 48 on four (128: half the CUs idle). So the tiles whose rounds of one workgroup per CU take in the fewest rows;
// more tiles stream a little worse (one row of the vocabulary 196 on one, 203 and 252), which two tiles are charged as the bytes of 3300 / Kb more rows
// a round. Of up to 12 X rows and W rows 16 KiB apart or a larger power of two, whose tiles fall on the same memory channels, each tile more is charged
// a tenth: one row of 128256 x 8192 400 on one, 438 on two, of 8192 x 8192 31 and 34. Over 477 products of 27 shapes, 1 to 32 rows, the choices take
// 1 % more than the best ones and 8 % less than one tile. The sums' order is the same on any.
constexpr int kCus = 256;
static int skinny_tiles(int M, int N, int Kb, int S, int glu) {
  int best = 0;
  double least = 0;
  for (int nt = glu ? 2 : 1; nt <= 4; nt *= 2) {
    if (N % (16 * nt)) break;
    const int rounds = (N / (16 * nt) * S + kCus - 1) / kCus;
    const double far = M <= 12 && Kb >= 8192 && (Kb & (Kb - 1)) == 0 ? 1.0 + 0.1 * (nt - 1) : 1.0;
    const double cost = rounds * ((16.0 * nt * far * (nt == 4 ? 1.15 : 1.0) + 0.8 * M) * Kb + (nt == 2 && !glu ? 3300 : 0));
    if (best == 0 || cost < least) best = nt, least = cost;
  }
  return best;
}

int gemm_skinny(const bf16_t* X, const bf16_t* W, bf16_t* Y, float* P, int M, int N, int K, int S, int glu, int blocks,
                hipStream_t stream) {
  if (M < 1 || M > 32) return -1;
  if (S < 1 || S > 8 || K % (S * sk::kWaves * 32) != 0) return -2;
  if (glu && (S != 1 || N % 128 != 0)) return -3;
  if (N % 16 != 0) return -4;
  if (S > 1 && P == nullptr) return -5;
  if (blocks > 0) {
    if (const int rc = gemm_rows(X, W, Y, P, M, N, K, S, glu, blocks, nullptr, stream)) return rc;
    if (S > 1 && Y != nullptr) {
      if ((int64_t)M * N % 4 != 0) return -6;
      return splitk_reduce(P, Y, (int64_t)M * N, S, stream);
    }
    return 0;
  }
  const int nt = skinny_tiles(M, N, K / S, S, glu), steps = K / S / (sk::kWaves * 32), rounds = (N / (16 * nt) * S + kCus - 1) / kCus;
  // k-steps in flight: long streams of many rounds take more (128256 x 4096, one row: 16 steps 191 us, 8 196; 8 rows on two tiles: 8 steps
  // 222, 4 226), but not where it leaves a remainder, whose steps wait one by one
  if (nt == 4) launch_skinny<4, 2>(X, W, Y, P, M, N, K, S, glu, stream);
  else if (nt == 2 && steps % 8 == 0 && (glu || rounds >= 4)) launch_skinny<2, 8>(X, W, Y, P, M, N, K, S, glu, stream);
  else if (nt == 2) launch_skinny<2, 4>(X, W, Y, P, M, N, K, S, glu, stream);
  else if (steps % 16 == 0 && rounds >= 4) launch_skinny<1, 16>(X, W, Y, P, M, N, K, S, glu, stream);
  else launch_skinny<1, 8>(X, W, Y, P, M, N, K, S, glu, stream);
  OAMD_LAUNCH_CHECK();
  if (S > 1 && Y != nullptr) {  // Y == nullptr: the consumer sums the slabs
    const int64_t MN = (int64_t)M * N;
    if (MN % 4 != 0) return -6;
    return splitk_reduce(P, Y, MN, S, stream);
  }
  return 0;
}

}  // namespace oamd
