// 32-bit forms of the model's products, for models served in fp32 (32-bit operands, products and
// sums): GEMMs (plain, gated, per-expert row groups) on the fp32 matrix instruction and attention
// for any head size. Larger GEMMs run in gemm_f32_split.hip.
#include "common.h"
#include "gemm_f32.h"
#include "kernels.h"

namespace oamd {

namespace {

// Rows the skinny kernel runs: one 16-row fragment streams W best (1 row of 2048 x 8192: 26 us); with two the
// repeated rows cost more than K slices of the tile kernel do (33 rows 33 us, 32 rows 55 skinny), unless K is
// too short to cut (32 rows of 1536 x 768: 9 us against 14).
inline bool skinny_rows(int M, int K) { return M <= 16 || (M <= 32 && K < 2048); }

constexpr int kStages = 3;   // LDS ring of the tile kernel: two 32-column pieces of K in flight

__device__ __forceinline__ f32x4 mfma4(const f32x4& a, const f32x4& b, f32x4 c) {   // k = 4 (lane / 16) + 0..3 of both
#pragma unroll
  for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
  return c;
}

// 4 neighbouring values of a row, n valid ones, the others 0
__device__ __forceinline__ f32x4 get4(const float* x, int n) {
  f32x4 v{};
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (e < n) v[e] = x[e];
  return v;
}

}  // namespace

// Y[M, N] = X[M, K] W[N, K]^T in fp32 on the fp32 matrix instruction (full 32-bit products and sums), 64 x 64
// tiles, four waves of 32 x 32 outputs in 16 x 16 blocks.
// What bounds it: the fp32 MFMA rate, 256 flop per clock and CU (157 TFLOP/s; ordinary FMA reaches half of that without
// packed fp32, which is off). A 32-column step is 1024 clocks of MFMA against 256 of fragment reads and 128 of LDS-DMA
// writes; with two or three workgroups per CU, reads, requests and products one after the other left the MFMAs a third of
// the time (962 rows of 16384 x 2048 gated 632 us). So a step's second fragments are read under its first products, the next step's
// first under its second ones, and the LDS-DMA pieces go out between them: 560 us (123 TFLOP/s with the padding rows, what a large product
// reaches), 12 products of 2048 features 146 -> 131 on average. 64 x 64 tiles because products
// here have few rows (500 rows of 2048 features: 256 tiles) and because routed experts' segments are padded to 64 rows.
// 18 rows of 2048 x 8192 in eight K slices 33 us.
// GLU: W holds gate | up rows interleaved in 64-row blocks; a tile is 64 features, Y [M, N/2]
// = act(c g) * (c u) with c the row's scale (rscale, or 1).
// gtab != nullptr: rows are expert segments padded to 64-row tiles; gtab[0] = tile count,
// gtab[1 + i] = expert of tile i, W [experts][N][K].
// PART: K slice blockIdx.z of S, raw sums into its slab.
template <bool GLU, bool PART>
__global__ void __launch_bounds__(256) gemm_f32_kernel(const GemmF32 a) {
  constexpr int NB = GLU ? 2 : 1;
  constexpr int kRows = 64 + 64 * NB, kStage = kRows * 128, GL = kRows / 32;
  __shared__ __attribute__((aligned(1024))) char lds[kStages * kStage];
  const int K = a.K;
  const int lid = xcd_remap(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
  const int mt = lid % gridDim.x, m0 = mt * 64, f0 = (lid / gridDim.x) * 64;
  const float *X = a.X, *W = a.W;
  float* Y = a.Y;
  if (a.gtab) {
    if (mt >= a.gtab[0]) return;
    W += (int64_t)a.gtab[1 + mt] * a.N * a.K;
  }
  int kbase = 0, T = (a.K + 31) / 32;
  if constexpr (PART) {
    const int t0 = (int)blockIdx.z * T / a.S;
    T = ((int)blockIdx.z + 1) * T / a.S - t0;
    kbase = t0 * 32;
    Y = a.P + (int64_t)blockIdx.z * a.M * a.N;
  } else if (blockIdx.z) {   // one product per head
    X += blockIdx.z * a.xh;
    W += (int64_t)blockIdx.z * a.N * a.K;
    Y += blockIdx.z * a.yh;
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wm = w >> 1, wn = w & 1;

  // LDS-DMA piece i of this wave: stage rows 8 (w + 4 i) .. +7 (X, then W), lane l -> row + l / 8, 16-B slot l % 8;
  // the slot holds source chunk slot ^ (row / 2 % 8), which keeps the fragment reads free of bank conflicts.
  // Rows past M / N repeat the last one, columns past K the row's first (never multiplied).
  const float* src[GL];
  int col[GL];
#pragma unroll
  for (int i = 0; i < GL; ++i) {
    const int row = 8 * (w + 4 * i) + (lane >> 3);
    src[i] = row < 64 ? X + min(m0 + row, a.M - 1) * a.ldx : W + (int64_t)min((GLU ? 2 * f0 : f0) + row - 64, a.N - 1) * a.K;
    col[i] = 4 * ((lane & 7) ^ ((row >> 1) & 7));
  }
  auto issue = [&](int t, int off, int i) {
    const int k = kbase + t * 32 + col[i];
    const float* from = src[i] + (k < K ? k : 0);
    __builtin_amdgcn_global_load_lds(from, (__attribute__((address_space(3))) void*)(lds + off + (w + 4 * i) * 1024), 16, 0, 0);
  };
  const int l15 = lane & 15, g = lane >> 4, sw = (l15 >> 1) & 7;   // row / 2 % 8 depends on the lane only: blocks are 16 rows
  const int xo = (wm * 32 + l15) * 128, wo = (64 + wn * 32 + l15) * 128;
  constexpr int NF = 2 + 2 * NB;   // fragments of a 16-column half: two token blocks, then the features'
  auto rd = [&](int off, int s, f32x4 (&f)[NF], int i) {
    const int at = off + (((4 * s + g) ^ sw) << 4);
    f[i] = *reinterpret_cast<const f32x4*>(lds + at + (i < 2 ? xo + i * 2048 : wo + ((i - 2) >> 1) * 8192 + (i & 1) * 2048));
  };
  // A barrier inside every step (after kBar of the second half's kH MFMAs) says that its stage has been read and the next one
  // has landed: the next step's first fragments are read behind it, and the pieces of the step kStages ahead go into the stage,
  // spread over the 2 kH MFMAs up to the next barrier.
  constexpr int kH = 16 * NB, kBar = kH / 4, kTail = kH - kBar;
  f32x4 acc[NB][2][2] = {};   // [gate | up][feature block][token block]
  auto mul = [&](const f32x4 (&f)[NF], int v) {
    const int e = v / (4 * NB), b = v / 4 % NB, j = v / 2 % 2, i = v % 2;
    acc[b][j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[2 + 2 * b + j][e], f[i][e], acc[b][j][i], 0, 0, 0);
  };
  auto piece = [&](int z, int t, int off) {
    const int i = (z * GL + 2 * kH - 1) / (2 * kH);
    if (i < GL && i * 2 * kH / GL == z && t < T) issue(t, off, i);
  };
#pragma unroll
  for (int st = 0; st < kStages; ++st)
    if (T > st)
#pragma unroll
      for (int i = 0; i < GL; ++i) issue(st, st * kStage, i);
  if (T > 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * GL) : "memory");
  else if (T > 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(GL) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  f32x4 fa[NF], fb[NF];
#pragma unroll
  for (int i = 0; i < NF; ++i) rd(0, 0, fa, i);
  int off = 0, prev = -1;   // this step's stage; the one of the step before, whose refill goes on
  for (int t = 0; t < T; ++t) {
    const int nxt = off + kStage == kStages * kStage ? 0 : off + kStage;
    const int fill = prev < 0 ? T : t + kStages - 1;   // the step that goes into `prev`
#pragma unroll
    for (int v = 0; v < kH; ++v) {
      mul(fa, v);
      __builtin_amdgcn_sched_barrier(0);
      if (v < NF) rd(off, 1, fb, v);
      piece(kTail + v, fill, prev);
      __builtin_amdgcn_sched_barrier(0);
    }
    const bool two = kbase + t * 32 + 16 < K;   // K % 32 == 16: the last step has one half
#pragma unroll
    for (int v = 0; v < kBar; ++v) {
      if (two) mul(fb, v);
      __builtin_amdgcn_sched_barrier(0);
      piece(kTail + kH + v, fill, prev);
      __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (t + 2 < T) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(GL) : "memory");   // all but the pieces of the step after the next
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (two) {
#pragma unroll
      for (int v = kBar; v < kH; ++v) {
        mul(fb, v);
        __builtin_amdgcn_sched_barrier(0);
        if (v - kBar < NF) rd(nxt, 0, fa, v - kBar);
        piece(v - kBar, t + kStages, off);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    prev = off;
    off = nxt;
  }
  // a lane holds features 4 g .. + 3 of each block of token l15
  const int NO = GLU && !PART ? a.N / 2 : a.N;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int m = m0 + wm * 32 + 16 * i + l15;
    if (m >= a.M) continue;
    const float c = a.rscale ? a.rscale[m] : 1.f;
    float* yr = Y + m * (PART ? (int64_t)a.N : a.ldy);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int f = wn * 32 + 16 * j + 4 * g;
      if constexpr (PART) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const int n = (GLU ? 2 * f0 + 64 * b : f0) + f;
          put4(yr + n, acc[b][j][i], NO - n, a.N % 4 == 0);
        }
      } else {
        f32x4 v = acc[0][j][i];
        if constexpr (GLU)
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = glu1(c * v[r], c * acc[NB - 1][j][i][r], a.act);
        put4(yr + f0 + f, v, NO - f0 - f, a.vec);
      }
    }
  }
}

// Y = sum_s P[s] (GLU: of the interleaved gate | up columns, then act(g) u), 4 outputs per thread.
template <bool GLU>
__global__ void __launch_bounds__(256) slabs_f32_kernel(const GemmF32 a) {
  const int NO = GLU ? a.N / 2 : a.N;
  const int64_t at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4, MN = (int64_t)a.M * a.N;
  const int m = (int)(at / NO), f = (int)(at % NO);
  if (m >= a.M) return;
  const float* p = a.P + (int64_t)m * a.N + (GLU ? (f >> 6) * 128 + (f & 63) : f);
  f32x4 v{}, u{};
  for (int s = 0; s < a.S; ++s, p += MN) {
    v += *reinterpret_cast<const f32x4*>(p);
    if constexpr (GLU) u += *reinterpret_cast<const f32x4*>(p + 64);
  }
  if constexpr (GLU)
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = glu1(v[r], u[r], a.act);
  put4(a.Y + m * a.ldy + f, v, 4, a.vec);
}

// The same product for at most 16 MT rows: small decode batches and the last rows of a prefill; up to sixteen of 768 columns and more run in
// gemm_f32_rows.hip (ops.f32_rows_plan).
// What bounds it: streaming W once from HBM (1 row: 16384 x 2048 gated 37 us, 3.6 TB/s; 32000 x 2048 53 us, 5 TB/s; the
// 64-row FMA tiles before took 450 and 180). A workgroup takes 16 features (GLU: 16 gate and 16 up rows); its waves
// take 32-column pieces of K in turn, whole 128-B lines of 16 rows straight into MFMA fragments (two to four pieces
// requested before the first is used), and their sums meet in LDS. The rows come from L2 in the same layout.
template <bool GLU, int MT, int NW>
__global__ void __launch_bounds__(64 * NW) gemm_f32_skinny_kernel(const GemmF32 a) {
  constexpr int NB = GLU ? 2 : 1;
  __shared__ f32x4 red[NW][NB * MT][64];
  const int f0 = blockIdx.x * 16, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int l15 = lane & 15, g = lane >> 4;
  const float* X = a.X + blockIdx.z * a.xh;
  const float* W = a.W + (int64_t)blockIdx.z * a.N * a.K;
  const float *xr[MT], *wr[NB];
#pragma unroll
  for (int i = 0; i < MT; ++i) xr[i] = X + min(16 * i + l15, a.M - 1) * a.ldx + 4 * g;
#pragma unroll
  for (int b = 0; b < NB; ++b) wr[b] = W + (int64_t)min(GLU ? (f0 >> 6) * 128 + 64 * b + (f0 & 63) + l15 : f0 + l15, a.N - 1) * a.K + 4 * g;
  f32x4 acc[NB][MT] = {};
  constexpr int U = MT * NB <= 2 ? 4 : 2;   // pieces requested before the first is used
  const f32x4 zero{};
  for (int c0 = w * U; c0 * 32 < a.K; c0 += NW * U) {
    f32x4 wf[U][NB][2], xf[U][MT][2];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int k = (c0 + u) * 32 + 16 * s;
        const bool in = k < a.K;
#pragma unroll
        for (int b = 0; b < NB; ++b) wf[u][b][s] = in ? *reinterpret_cast<const f32x4*>(wr[b] + k) : zero;
#pragma unroll
        for (int i = 0; i < MT; ++i) xf[u][i][s] = in ? *reinterpret_cast<const f32x4*>(xr[i] + k) : zero;
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int i = 0; i < MT; ++i) acc[b][i] = mfma4(wf[u][b][s], xf[u][i][s], acc[b][i]);
  }
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int i = 0; i < MT; ++i) red[w][b * MT + i][lane] = acc[b][i];
  __syncthreads();
  const int NO = GLU ? a.N / 2 : a.N;
  for (int i = w; i < MT; i += NW) {
    const int m = 16 * i + l15;
    f32x4 v{}, u{};
#pragma unroll
    for (int x = 0; x < NW; ++x) {
      v += red[x][i][lane];
      if constexpr (GLU) u += red[x][MT + i][lane];
    }
    if (m >= a.M) continue;
    const float c = a.rscale ? a.rscale[m] : 1.f;
    if constexpr (GLU)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = glu1(c * v[r], c * u[r], a.act);
    put4(a.Y + blockIdx.z * a.yh + m * a.ldy + f0 + 4 * g, v, NO - f0 - 4 * g, a.vec);
  }
}

bool f32_tiles(int M, int K, bool grouped) { return grouped || !skinny_rows(M, K); }

// K slices of the tile kernel: two workgroups per CU where the tiles alone give fewer, slices of 256 columns at least
int gemm_f32_splits(int M, int N, int K, int glu) {
  if (skinny_rows(M, K) || N % 4) return 1;
  const int64_t tiles = (int64_t)((M + 63) / 64) * (((glu ? N / 2 : N) + 63) / 64);
  int S = 1;
  while (tiles * S < 512 && S < 8 && K / (2 * S) >= 256) S *= 2;
  return S;
}

template <bool GLU, int NW>
static void launch_skinny(const GemmF32& a, dim3 grid, hipStream_t stream) {
  if (a.M <= 16) gemm_f32_skinny_kernel<GLU, 1, NW><<<grid, 64 * NW, 0, stream>>>(a);
  else gemm_f32_skinny_kernel<GLU, 2, NW><<<grid, 64 * NW, 0, stream>>>(a);
}

int sum_f32_slabs(const float* P, float* Y, int S, int M, int N, int ldy, hipStream_t stream) {
  GemmF32 a{nullptr, nullptr, Y, const_cast<float*>(P), M, N, 0, S, 0, ldy, 0, 0, nullptr, nullptr, GluAct{}, ldy % 4 == 0 && reinterpret_cast<uintptr_t>(Y) % 16 == 0};
  slabs_f32_kernel<false><<<(int)(((int64_t)M * N / 4 + 255) / 256), 256, 0, stream>>>(a);
  OAMD_LAUNCH_CHECK();
  return 0;
}

static int run_f32(GemmF32 a, bool glu, int H, int rows, hipStream_t stream) {
  const int nf = glu ? a.N / 2 : a.N;
  a.vec = a.ldy % 4 == 0 && a.yh % 4 == 0 && reinterpret_cast<uintptr_t>(a.Y) % 16 == 0;
  if (rows) {
    if (const int rc = gemm_f32_split(a, glu, rows, stream)) return rc;
  } else if (!f32_tiles(a.M, a.K, a.gtab != nullptr)) {
    const dim3 grid((nf + 15) / 16, 1, H);
    // enough waves to keep the loads of one CU in flight, and work for each of them
    if (glu) launch_skinny<true, 8>(a, grid, stream);
    else if (a.K >= 1024) launch_skinny<false, 8>(a, grid, stream);
    else launch_skinny<false, 4>(a, grid, stream);
  } else {
    const dim3 grid((a.M + 63) / 64, (nf + 63) / 64, a.S > 1 ? a.S : H);
    if (grid.y > 65535) return -1;
    if (a.S > 1 && glu) gemm_f32_kernel<true, true><<<grid, 256, 0, stream>>>(a);
    else if (a.S > 1) gemm_f32_kernel<false, true><<<grid, 256, 0, stream>>>(a);
    else if (glu) gemm_f32_kernel<true, false><<<grid, 256, 0, stream>>>(a);
    else gemm_f32_kernel<false, false><<<grid, 256, 0, stream>>>(a);
  }
  if (a.S > 1) {
    const int blocks = (int)(((int64_t)a.M * nf / 4 + 255) / 256);
    if (glu) slabs_f32_kernel<true><<<blocks, 256, 0, stream>>>(a);
    else slabs_f32_kernel<false><<<blocks, 256, 0, stream>>>(a);
  }
  OAMD_LAUNCH_CHECK();
  return 0;
}

int gemm_f32(const float* X, const float* W, float* Y, float* P, int S, int M, int N, int K, int ldy, int glu, const int* gtab,
             const float* rscale, int rows, hipStream_t stream) {
  if (M == 0) return 0;
  if (rows && ((rows != 64 && rows != 128 && rows != 256) || gtab || rscale)) return -3;
  if (K % 16 || (glu && N % 128) || S < 1 || S > 8) return -1;
  if (S > 1 && (P == nullptr || gtab || rscale || N % 4 || (!rows && skinny_rows(M, K)))) return -2;
  return run_f32({X, W, Y, P, M, N, K, S, K, ldy, 0, 0, gtab, rscale, glu ? glu_act(glu) : GluAct{}, 0}, glu != 0, 1, rows, stream);
}

int head_gemm_f32(const float* X, const float* W, float* Y, int M, int N, int K, int H, int64_t ldx, int64_t xh,
                  int64_t ldy, int64_t yh, hipStream_t stream) {
  if (M == 0) return 0;
  if (K % 16 || ldx % 4 || xh % 4 || H < 1 || H > 65535) return -1;
  return run_f32({X, W, Y, nullptr, M, N, K, 1, ldx, ldy, xh, yh, nullptr, nullptr, GluAct{}, 0}, false, H, 0, stream);
}

// Attention on the fp32 matrix instruction: S^T = K Q^T, so a lane holds scores of one query (l15) and the
// accumulator of the scores is already the operand of O^T += V^T P^T: no round trip for the weights, and the
// running maximum, sum and rescale stay on the query's lanes.
namespace {

struct RowStat { float m = -1e30f, l = 0.f; };

// Scores st[kb][r] of keys j0 + 16 kb + 4 g + r -> softmax weights against the running maximum; the factor
// of what was accumulated. Keys outside [lo, n) get weight 0.
template <int NB>
__device__ __forceinline__ float soften(f32x4 (&st)[NB], int j0, int g, int lo, int n, float scale, RowStat& q) {
  float top = -INFINITY;
#pragma unroll
  for (int kb = 0; kb < NB; ++kb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = j0 + 16 * kb + 4 * g + r;
      st[kb][r] = j >= lo && j < n ? st[kb][r] * scale : -INFINITY;
      top = fmaxf(top, st[kb][r]);
    }
  top = max_rows(top);
  const float mn = fmaxf(q.m, top), alpha = expf(q.m - mn);
  float sum = 0.f;
#pragma unroll
  for (int kb = 0; kb < NB; ++kb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      st[kb][r] = expf(st[kb][r] - mn);
      sum += st[kb][r];
    }
  q.m = mn;
  q.l = q.l * alpha + sum;   // this lane's keys; the query's four lanes meet at the end
  return alpha;
}

}  // namespace

// Prefill: a workgroup is 64 query rows of one sequence and head, a wave 16 of them; 32-key tiles of K and V
// are shared through LDS (rows padded by 16 B) and the next tile's loads are in flight while one is used.
// NG: the even tiles and the odd ones have sums of their own, which meet at the end. Two groups of four waves (NG == 2) take them side
// by side: with few workgroups on the chip one group's softmax would leave the matrix cores idle, and the longest rows bound the
// launch. One group (NG == 1) takes the even tiles, then the odd ones: half the LDS, and nobody waits where there is but one tile. Same
// sums, same bits, so the launch chooses (f32_prefill_groups) and a prompt's numbers do not depend on what it is packed with.
// What bounds it: with few workgroups those with the longest rows, whose 32-key tile is 1.7 us of fp32 MFMAs and about as much of softmax,
// staging and barriers; with many, the MFMA rate. One group and two: 2 x 500 rows of 16 heads of 128 72 and 59 us, 1000 rows of 8 heads of 256
// 250 and 206, 128 x 64 rows of 16 heads of 128 75 and 98, 64 x 16 rows 22 and 33.
// LESS: heads that end before D's last blocks, behind a way out per block: 2000 rows of 32 heads of 192 and 128 columns 1520 us without one, 1140 with it.
// Where no block is left out it would keep reads from crossing it.
// D: instantiated size >= both head sizes. ODD: value heads that are no multiple of 16 columns, or output rows that take no
// 16-B stores (key heads are multiples of 4 in either form).
template <int D, bool ODD, bool LESS, int NG>
__global__ void __launch_bounds__(256 * NG, NG == 1 && D == 64 ? 4 : 1) attn_f32_prefill_kernel(const AttnF32 a) {
  constexpr int BK = 32, LD = D + 4, NC = D / 32;   // NC: 16-B chunks of a row per loading thread
  constexpr int kTile = 2 * BK * LD;   // a group's K and V
  constexpr int kSums = 4 * (D / 16) + 2;   // a lane's
  static_assert(NG == 1 || 256 * kSums <= 2 * kTile, "the second group's sums take the tiles' place");
  __shared__ __attribute__((aligned(16))) float lds[NG * kTile];
  __shared__ int odds[4 * NG];   // of every wave: its values of the tile are not all finite
  const int seq = a.work_seq[blockIdx.x];
  if (seq < 0) return;   // padding item of a graph-captured prefill (fixed grid)
  const int s0 = a.cu_seqlens[seq], slen = a.cu_seqlens[seq + 1] - s0;
  const int q0 = a.work_q0[blockIdx.x] + 64 * blockIdx.z;
  if (q0 >= slen) return;
  const int Hq = gridDim.y, hq = blockIdx.y, kvh = hq / (Hq / a.Hkv);
  const int grp = NG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int tid = threadIdx.x & 255, lane = tid & 63, w = tid >> 6, l15 = lane & 15, g = lane >> 4;
  float *ks = lds + grp * kTile, *vs = ks + BK * LD;
  const int pl = a.seq_pfx ? a.seq_pfx[seq] : 0;
  const int qrow = q0 + 16 * w + l15;
  const int n = qrow < slen ? pl + qrow + 1 : 0, lo = max(0, pl + qrow + 1 - a.window);   // keys [lo, n) of this lane's query
  const int kend = pl + min(slen, q0 + 64), kbeg = max(0, pl + q0 + 1 - a.window) & ~(BK - 1);
  float* out = a.o + (int64_t)(s0 + qrow) * a.o_ld + hq * a.dvp + 4 * g;   // of rows that exist: n > 0

  const f32x4 zero{};
  f32x4 qf[D / 16];
#pragma unroll
  for (int c = 0; c < D / 16; ++c)
    qf[c] = n > 0 && 16 * c + 4 * g < a.dkp ? *reinterpret_cast<const f32x4*>(a.q + ((int64_t)(s0 + qrow) * Hq + hq) * a.dkp + 16 * c + 4 * g) : zero;
  // loader: thread -> row tid / 8 of the tile, chunks tid % 8 + 8 i
  const int lr = tid >> 3, lc = tid & 7;
  f32x4 kn[NC], vn[NC];
  auto load = [&](int j0) {
    const int j = j0 + lr;
    const bool in = j < kend, pre = j < pl;
    const int64_t r = pre ? j : s0 + j - pl;
    const float* kp = (pre ? a.pk : a.k) + (r * a.Hkv + kvh) * a.dkp;
    const float* vp = (pre ? a.pv : a.v) + (r * a.Hkv + kvh) * a.dvp;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = 4 * (lc + 8 * i);
      kn[i] = in && c < a.dkp ? *reinterpret_cast<const f32x4*>(kp + c) : zero;
      if constexpr (ODD) vn[i] = in ? get4(vp + c, a.dvp - c) : zero;
      else vn[i] = in && c < a.dvp ? *reinterpret_cast<const f32x4*>(vp + c) : zero;
    }
  };
  f32x4 acc[D / 16] = {};   // dims 16 b + 4 g + r of query l15
  f32x4 acc0[D / 16];
  RowStat st, st0;          // acc0, st0 (NG == 1): of the even tiles
  // steps of the group: a tile of its own each (NG == 2, the second group's last may be past the end), or the even tiles, then the odd ones
  const int tiles = (kend - kbeg + BK - 1) / BK, evens = (tiles + 1) >> 1, steps = NG == 1 ? tiles : evens;
  auto key0 = [&](int t) { return kbeg + BK * (NG == 2 ? 2 * t + grp : t < evens ? 2 * t : 2 * (t - evens) + 1); };
  load(key0(0));
  for (int t = 0; t < steps; ++t) {
    const int j0 = key0(t);
    __syncthreads();
    bool odd = false;   // a value that must not meet the weight 0 of a query that does not see its key
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      *reinterpret_cast<f32x4*>(ks + lr * LD + 4 * (lc + 8 * i)) = kn[i];
      *reinterpret_cast<f32x4*>(vs + lr * LD + 4 * (lc + 8 * i)) = vn[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) odd |= !(fabsf(vn[i][e]) <= 3.4028234e38f);
    }
    odd = __any(odd);
    if (lane == 0) odds[4 * grp + w] = odd;
    __syncthreads();
    odd = odds[4 * grp] | odds[4 * grp + 1] | odds[4 * grp + 2] | odds[4 * grp + 3];   // of the group's tile alone
    if (t + 1 < steps) load(key0(t + 1));
    if (NG == 1 && t == evens) {   // the odd tiles begin
#pragma unroll
      for (int b = 0; b < D / 16; ++b) {
        acc0[b] = acc[b];
        acc[b] = zero;
      }
      st0 = st;
      st = RowStat{};
    }
    if (j0 >= min(kend, pl + q0 + 16 * w + 16)) continue;   // past every query of this wave
    // the reads of a block go out under the block before, and behind the last block of a smaller head is the way out
    f32x4 s[2] = {}, kf[2][2];
    auto keys = [&](int c) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) kf[c & 1][kb] = *reinterpret_cast<const f32x4*>(ks + (16 * kb + l15) * LD + 16 * c + 4 * g);
    };
    keys(0);
#pragma unroll
    for (int c = 0; c < D / 16; ++c) {
      if (c + 1 < D / 16) keys(c + 1);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) s[kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[c & 1][kb][e], qf[c][e], s[kb], 0, 0, 0);
      if (LESS && 16 * (c + 1) >= a.dkp) break;
    }
    float vf[2][2][8];   // two blocks' values, and the next two's
    auto values = [&](int b) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 8; ++e) vf[(b >> 1) & 1][h][e] = vs[(16 * (e >> 2) + 4 * g + (e & 3)) * LD + 16 * (b + h) + l15];
    };
    values(0);
    const float alpha = soften<2>(s, j0, g, lo, n, a.scale, st);
    if (odd) {   // infinities or NaN among the values: key by key, for the queries that see it
#pragma unroll
      for (int b = 0; b < D / 16; ++b) acc[b] *= alpha;
#pragma unroll
      for (int i = 0; i < BK; ++i) {
        const float p = __shfl(s[i >> 4][i & 3], (i >> 2 & 3) * 16 + l15, kWave);
        if (j0 + i < lo || j0 + i >= n) continue;
#pragma unroll
        for (int b = 0; b < D / 16; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[b][r] = __builtin_fmaf(p, vs[i * LD + 16 * b + 4 * g + r], acc[b][r]);
      }
      continue;
    }
#pragma unroll
    for (int b = 0; b < D / 16; b += 2) {
      if (b + 2 < D / 16) values(b + 2);
      acc[b] *= alpha;
      acc[b + 1] *= alpha;
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          acc[b + h] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[(b >> 1) & 1][h][e], s[e >> 2][e & 3], acc[b + h], 0, 0, 0);
      if (LESS && 16 * (b + 2) >= a.dvp) break;
    }
  }
  // the even tiles' sums f and m0, l0; the odd ones' e and m1, l1
  auto meet = [](float& f, float a0, float e, float a1) { f = __builtin_fmaf(e, a1, f * a0); };
  if constexpr (NG == 2) {
    __syncthreads();   // the tiles are free
    f32x4* sums = reinterpret_cast<f32x4*>(lds) + tid;   // [block][thread], behind them m and l
    float* mine = lds + 1024 * (D / 16) + tid;
    if (grp == 1) {
#pragma unroll
      for (int b = 0; b < D / 16; ++b) sums[256 * b] = acc[b];
      mine[0] = st.m;
      mine[256] = st.l;
    }
    __syncthreads();
    if (grp == 1) return;
    const float m1 = mine[0], mn = fmaxf(st.m, m1), a0 = expf(st.m - mn), a1 = expf(m1 - mn);
    meet(st.l, a0, mine[256], a1);
#pragma unroll
    for (int b = 0; b < D / 16; ++b) {
      const f32x4 e = sums[256 * b];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float f = acc[b][r];
        meet(f, a0, e[r], a1);
        acc[b][r] = f;
      }
    }
  } else if (tiles > 1) {
    const float mn = fmaxf(st0.m, st.m), a0 = expf(st0.m - mn), a1 = expf(st.m - mn);
    meet(st0.l, a0, st.l, a1);
    st.l = st0.l;
#pragma unroll
    for (int b = 0; b < D / 16; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float f = acc0[b][r];
        meet(f, a0, acc[b][r], a1);
        acc[b][r] = f;
      }
  }
  const float l = sum_rows(st.l);
  if (n <= 0) return;
  const float c = (a.gate ? a.gate[(int64_t)(s0 + qrow) * Hq + hq] : 1.f);
#pragma unroll
  for (int b = 0; b < D / 16; ++b) {
    if (16 * b >= a.dvp) break;
    f32x4 v;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = a.gate ? acc[b][r] / l * c : acc[b][r] / l;
    if constexpr (ODD) put4(out + 16 * b, v, a.dvp - 16 * b - 4 * g, false);
    else *reinterpret_cast<f32x4*>(out + 16 * b) = v;
  }
}

// Two groups pay until their workgroups, twice as large, come in more than a round or two of the CUs, and not where most query rows have a single
// tile of keys (two, of the largest heads, which have a workgroup per CU either way). `blocks` is about the number of workgroups that have rows. Over 26
// packings of 4 to 8192 rows and ten head layouts the choices take 0.3 % more than the better form; nowhere more than 7 %.
static int f32_prefill_groups(int D, int64_t rows, int items, int Hq) {
  const int64_t blocks = (items + rows / 128) * Hq;
  return rows > (int64_t)items * (D == 256 ? 64 : 32) && blocks <= (D == 64 ? 600 : D == 128 ? 400 : 2000) ? 2 : 1;
}

template <int D, bool ODD>
static void launch_f32_prefill(const AttnF32& a, int64_t rows, const dim3& grid, hipStream_t stream) {
  const bool less = a.dkp <= D - 16 || a.dvp <= D - 32;   // loops that may end before D
  if (f32_prefill_groups(D, rows, grid.x, grid.y) == 1) {
    if (less) attn_f32_prefill_kernel<D, ODD, true, 1><<<grid, 256, 0, stream>>>(a);
    else attn_f32_prefill_kernel<D, ODD, false, 1><<<grid, 256, 0, stream>>>(a);
  } else {
    if (less) attn_f32_prefill_kernel<D, ODD, true, 2><<<grid, 512, 0, stream>>>(a);
    else attn_f32_prefill_kernel<D, ODD, false, 2><<<grid, 512, 0, stream>>>(a);
  }
}

int attn_f32_prefill(const AttnF32& a, int64_t rows, int items, int Hq, hipStream_t stream) {
  if (items == 0) return 0;
  const int top = a.dkp > a.dvp ? a.dkp : a.dvp;
  if (a.dkp < 4 || a.dkp % 4 || a.dvp < 1 || top > 256 || Hq % a.Hkv || a.window < 1) return -1;
  const dim3 grid(items, Hq, 2);   // items are 128 query rows
  const bool odd = a.dvp % 16 || a.o_ld % 4;
#define OAMD_PF(D)                                                   \
  if (odd) launch_f32_prefill<D, true>(a, rows, grid, stream);       \
  else launch_f32_prefill<D, false>(a, rows, grid, stream)
  if (top <= 64) {
    OAMD_PF(64);
  } else if (top <= 128) {
    OAMD_PF(128);
  } else {
    OAMD_PF(256);
  }
#undef OAMD_PF
  OAMD_LAUNCH_CHECK();
  return 0;
}

// Decode: a workgroup takes one sequence, up to 16 query heads of one key / value head (`chunks` of them) and one of
// `splits` pieces of its context; its eight waves take 16-key tiles in turn, K and V straight from the pages into
// fragments (a tile is in one page, one row read serves all heads), and meet in LDS. One piece writes the
// result, several leave (sums, m, l) to attn_f32_combine. What bounds it: the latency of a wave's tiles, so the loads
// of a tile go out in large groups, with small heads its values before the scores are computed. 18 sequences of 1282
// tokens: 16 heads on one latent row of 288 454 -> 37 us, 4 heads of 128 on a key head, window 512, 202 -> 27 (with a
// workgroup per query head and a key per lane before).
// NB: 16-dim blocks of the value size. ODD: heads that are no multiple of 16 columns (keys: of 4), or output rows that take
// no 16-B stores.
template <int NB, bool ODD>
__global__ void __launch_bounds__(512) attn_f32_decode_kernel(const AttnF32 a, int Hq, int chunks, int splits, float* part, float* ml) {
  constexpr int NW = 8, RB = 4;                // waves, value blocks merged at a time
  constexpr bool kEarly = NB <= 8;             // a tile's values fit in registers beside the sums
  constexpr int KC = NB <= 8 ? 8 : 20;         // 16-column pieces of the keys requested at a time
  __shared__ f32x4 red[NW][RB][64];
  __shared__ float mls[NW][2][16];
  __shared__ __attribute__((aligned(16))) float qs[16 * (640 + 4)];
  const int t = blockIdx.x, kvh = blockIdx.y / chunks, G = Hq / a.Hkv, sp = blockIdx.z;
  const int h0 = kvh * G + (blockIdx.y % chunks) * 16, heads = min(16, (kvh + 1) * G - h0);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, l15 = lane & 15, g = lane >> 4;
  const int n = min(a.seq_lens[t], a.max_pages * a.page_size), lo = max(0, n - a.window);
  const int first = lo >> 4, tiles = n > 0 ? ((n + 15) >> 4) - first : 0;
  const int ta = first + (int)((int64_t)tiles * sp / splits), tb = first + (int)((int64_t)tiles * (sp + 1) / splits);
  const int ldq = a.dkp + 4;
  for (int i = tid * 4; i < heads * a.dkp; i += 64 * NW * 4)
    *reinterpret_cast<f32x4*>(qs + i / a.dkp * ldq + i % a.dkp) = *reinterpret_cast<const f32x4*>(a.q + ((int64_t)t * Hq + h0) * a.dkp + i);
  __syncthreads();
  const float* qp = qs + min(l15, heads - 1) * ldq + 4 * g;
  f32x4 acc[NB] = {};
  RowStat st;
  for (int tl = ta + w; tl < tb; tl += NW) {
    const int j0 = tl * 16;
    const int64_t row = ((int64_t)a.block_tables[(int64_t)t * a.max_pages + j0 / a.page_size] * a.Hkv + kvh) * a.page_size + j0 % a.page_size;
    const float* kp = a.k + (row + l15) * a.k_ld + 4 * g;
    const float* vp = a.v + (row + 4 * g) * a.v_ld + l15;
    // column of value block b: past the head its first block again, its last column in the lanes past that (not stored)
    auto vcol = [&](int b) {
      if constexpr (ODD)
        if (16 * b < a.dvp) return 16 * b + min(l15, a.dvp - 1 - 16 * b) - l15;
      return 16 * b < a.dvp ? 16 * b : ODD ? min(l15, a.dvp - 1) - l15 : 0;
    };
    float vf[8][4];
    if constexpr (kEarly)
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) vf[b][e] = vp[e * a.v_ld + vcol(b)];
    __builtin_amdgcn_sched_barrier(0);   // ... here, not where they are used
    f32x4 s[1] = {};
    const int dk = ODD ? a.dkp & ~15 : a.dkp;
    for (int c0 = 0; c0 < dk; c0 += 16 * KC) {
      f32x4 kf[KC];
#pragma unroll
      for (int c = 0; c < KC; ++c) kf[c] = *reinterpret_cast<const f32x4*>(kp + (c0 + 16 * c < dk ? c0 + 16 * c : 0));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < KC; ++c)
        if (c0 + 16 * c < dk) s[0] = mfma4(kf[c], *reinterpret_cast<const f32x4*>(qp + c0 + 16 * c), s[0]);
    }
    if constexpr (ODD) {   // the last columns of a key
      const f32x4 zero{};
      const bool in = dk + 4 * g < a.dkp;
      const f32x4 kt = in ? *reinterpret_cast<const f32x4*>(kp + dk) : zero, qt = in ? *reinterpret_cast<const f32x4*>(qp + dk) : zero;
      s[0] = mfma4(kt, qt, s[0]);
    }
    const float alpha = soften<1>(s, j0, g, lo, n, a.scale, st);
    constexpr int VB = kEarly ? NB : 8;   // value blocks requested at a time
#pragma unroll
    for (int b0 = 0; b0 < NB; b0 += VB) {
      if constexpr (!kEarly) {
#pragma unroll
        for (int b = 0; b < VB; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e) vf[b][e] = vp[e * a.v_ld + vcol(b0 + b)];
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int b = 0; b < VB; ++b) {
        if (16 * (b0 + b) >= a.dvp) continue;
        acc[b0 + b] *= alpha;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = j0 + 4 * g + e;
          const float v = j >= lo && j < n ? vf[b][e] : 0.f;   // rows outside may hold anything
          acc[b0 + b] = __builtin_amdgcn_mfma_f32_16x16x4f32(v, s[0][e], acc[b0 + b], 0, 0, 0);
        }
      }
    }
  }
  const float l = sum_rows(st.l);
  if (g == 0) {
    mls[w][0][l15] = st.m;
    mls[w][1][l15] = l;
  }
  __syncthreads();
  float M = -1e30f, L = 0.f, f[NW];
#pragma unroll
  for (int x = 0; x < NW; ++x) M = fmaxf(M, mls[x][0][l15]);
#pragma unroll
  for (int x = 0; x < NW; ++x) {
    f[x] = expf(mls[x][0][l15] - M);
    L += f[x] * mls[x][1][l15];
  }
  const int64_t hq = (int64_t)t * Hq + h0 + l15;
  const bool mine = l15 < heads;
  if (splits > 1 && w == 0 && g == 0 && mine) {
    ml[(hq * splits + sp) * 2] = M;
    ml[(hq * splits + sp) * 2 + 1] = L;
  }
#pragma unroll
  for (int b0 = 0; b0 < NB; b0 += RB) {
    if (16 * b0 >= a.dvp) continue;
    __syncthreads();
#pragma unroll
    for (int b = 0; b < RB && b0 + b < NB; ++b) red[w][b][lane] = acc[b0 + b];
    __syncthreads();
    const int b = b0 + w;   // wave w < RB finishes block b0 + w
    if (w < RB && b < NB && 16 * b < a.dvp && mine) {
      f32x4 o{};
#pragma unroll
      for (int x = 0; x < NW; ++x) o += f[x] * red[x][w][lane];
      float* out = splits > 1 ? part + (hq * splits + sp) * a.dvp : a.o + (int64_t)t * a.o_ld + (h0 + l15) * a.dvp;
      if (splits == 1)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = n <= 0 ? 0.f : a.gate ? o[r] / L * a.gate[hq] : o[r] / L;
      if constexpr (ODD) put4(out + 16 * b + 4 * g, o, a.dvp - 16 * b - 4 * g, false);
      else *reinterpret_cast<f32x4*>(out + 16 * b + 4 * g) = o;
    }
  }
}

// One workgroup per sequence and head: the pieces' sums against their common maximum.
template <bool ODD>
__global__ void __launch_bounds__(64) attn_f32_combine_kernel(const AttnF32 a, int Hq, int splits, const float* part, const float* ml) {
  const int64_t hq = (int64_t)blockIdx.x * Hq + blockIdx.y;
  float* out = a.o + (int64_t)blockIdx.x * a.o_ld + blockIdx.y * a.dvp;
  const bool any = a.seq_lens[blockIdx.x] > 0;
  float M = -1e30f, L = 0.f;
  for (int s = 0; s < splits; ++s) M = fmaxf(M, ml[(hq * splits + s) * 2]);
  for (int s = 0; s < splits; ++s) L += expf(ml[(hq * splits + s) * 2] - M) * ml[(hq * splits + s) * 2 + 1];
  for (int d = 4 * threadIdx.x; d < a.dvp; d += 256) {
    f32x4 o{};
    for (int s = 0; s < splits; ++s) {
      const float* p = part + (hq * splits + s) * a.dvp + d;
      o += expf(ml[(hq * splits + s) * 2] - M) * (ODD ? get4(p, a.dvp - d) : *reinterpret_cast<const f32x4*>(p));
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = !any ? 0.f : a.gate ? o[r] / L * a.gate[hq] : o[r] / L;
    if constexpr (ODD) put4(out + d, o, a.dvp - d, false);
    else *reinterpret_cast<f32x4*>(out + d) = o;
  }
}

int attn_f32_decode(const AttnF32& a, int rows, int Hq, int splits, float* part, float* ml, hipStream_t stream) {
  if (rows == 0) return 0;
  if (a.dkp < 4 || a.dkp % 4 || a.dvp < 1 || a.dkp > 640 || a.dvp > 640 || Hq % a.Hkv || a.window < 1 || a.page_size % 16) return -1;
  if (splits < 1 || splits > 256 || (splits > 1 && (part == nullptr || ml == nullptr))) return -2;
  const int chunks = (Hq / a.Hkv + 15) / 16;
  const dim3 grid(rows, a.Hkv * chunks, splits);
  const bool odd = a.dkp % 16 || a.dvp % 16 || a.o_ld % 4;
#define OAMD_DEC(NB)                                                                                        \
  if (odd) attn_f32_decode_kernel<NB, true><<<grid, 512, 0, stream>>>(a, Hq, chunks, splits, part, ml);     \
  else attn_f32_decode_kernel<NB, false><<<grid, 512, 0, stream>>>(a, Hq, chunks, splits, part, ml)
  if (a.dvp <= 128) {
    OAMD_DEC(8);
  } else if (a.dvp <= 256) {
    OAMD_DEC(16);
  } else {
    OAMD_DEC(40);
  }
#undef OAMD_DEC
  OAMD_LAUNCH_CHECK();
  if (splits > 1) {
    if (odd) attn_f32_combine_kernel<true><<<dim3(rows, Hq), 64, 0, stream>>>(a, Hq, splits, part, ml);
    else attn_f32_combine_kernel<false><<<dim3(rows, Hq), 64, 0, stream>>>(a, Hq, splits, part, ml);
    OAMD_LAUNCH_CHECK();
  }
  return 0;
}

}  // namespace oamd
