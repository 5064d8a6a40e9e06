// Decode-shape GEMM: Y[M, N] = X[M, K] . W[N, K]^T, bf16 in, fp32 accumulate
// (the explanation model's projections at decode batch).
//
// At decode the activations are small (M = bucket size, 64..256 rows) and the
// weights are streamed once per step, so the kernel is designed around the
// two streams rather than around a square tile:
//   * W (HBM, read once) and X (L2-resident, re-read by every column tile) are
//     both staged through LDS by LDS-DMA (global_load_lds_dwordx4) in full
//     128-B lines — no VGPR round trip, no fragment-shaped global loads
//     (cdna_hip_programming.md §5 "Projection GEMM at M = 256", item 3);
//   * a 3-deep LDS ring with a counted vmcnt + raw s_barrier keeps two stages
//     of both operands in flight across every barrier (never a vmcnt(0) drain
//     inside the k-loop);
//   * the LDS image is XOR-swizzled on the SOURCE address (the DMA writes LDS
//     lane-linearly), slot = chunk ^ ((row >> 1) & 7), which makes every
//     ds_read_b128 fragment read conflict-free;
//   * 8 waves (4 x 2), two per SIMD; the tile is BM = M rows x 64 columns; K is split S ways when N / 64
//     column tiles alone cannot fill 256 CUs. Split-K partials are fp32 slabs
//     [S][M][N] summed by gemm_splitk_reduce (or by a consumer kernel). With
//     S | 8 the blocks of one K-slice share an XCD (block id % 8), so each
//     XCD's L2 holds only its slice of X; other S (<= 16) cut K into slices
//     that differ by at most one 64-column step;
//   * where rows lie a multiple of 4 KB apart (K % 2048 == 0), column tile n starts its slice at K step n % steps and goes round: tiles in step would
//     all read the same 128 columns of such rows, which HBM serves from some of its channels (times of weights that no cache holds): 64 rows of
//     128256 x 4096 217 -> 181 us (4.8 -> 5.8 TB/s), 57344 x 8192 gated 194 -> 158, 28672 x 6144 80 -> 63. At other distances it costs 1 to 10 %,
//     most beside a multiple (64 rows of 4032 or 4160 columns 10 %, 3584 2 %; 128-row tiles 5 %), and gains in none but 11008 columns (5 %).
//     Experts' tiles of 64 rows start 5 steps further an expert: 8 rows for each of 8 experts of 4096 x 4096 183 -> 140 us, of 64 of 2048 x 1024
//     179 -> 155 (by the product over 2048 columns; 16 of 3456 x 2368 151 in step, 159 round); of 128 rows, whose X weighs more, they keep
//     step (112 rows each 242, 258 round).
// MFMA v_mfma_f32_16x16x32_bf16; fragment maps as in attn_decode.hip.
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace oamd {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

constexpr int kBK = 64;     // K per stage: one 128-B line per row
constexpr int kStages = 3;  // default LDS ring depth (2: two blocks per CU for the smaller tiles; 4 / 5 / 6:
                            // three / four / five stages in flight for tiles with BM + BN <= 320 / 256 /
                            // 192 rows, 160 KB of LDS at most)

// 8 waves (2 per SIMD: one wave's LDS-read latency hides under the other's
// MFMAs) laid out 4 (M) x 2 (N).
constexpr int kWaves = 8;
// Most elements of X whose K steps go round. Tiles in step share a piece of X while it is in their XCD's L2, tiles that are not need all of
// X there (4 MiB): 128 rows of 8192 x 28672 88 us in step, 96 round, of 3584 x 18944 30 and 41. 256-row tiles are not bound by HBM (32768 x 2048 40 and 43).
constexpr int64_t kTurnX = 1 << 20;
// Fewest columns of Y whose K steps go round, by the rows of X and of a tile, in 64: fewer tiles leave channels idle either way, and the addresses
// cost a little. 64 rows of K = 4096 and 8192: 14336 columns 37.0 us in step, 37.0 round and 70.1, 68.4, 20480 41.0, 39.6 and 80.8, 73.4, 8192
// 32.1, 33.4 and 61.4, 65.1; 128 rows in 64-row tiles: 20480 69.0, 70.8 and 132.7, 133.4, 28672 86.2, 79.6 and 168, 152; in 128-row tiles: 28672 53.1, 55.1
// and 97.0, 99.0, 34176 97.9, 92.8 and 186, 179.
constexpr int kTurnN = 8192;

// BN = 128 halves the LDS fragment traffic per MFMA (64 x 64 wave tiles at
// M = 256: 0.5 KB of ds_read per MFMA vs 0.75 KB at BN = 64, where the LDS
// port, not the MFMA, sets the pace); BN = 64 gives twice the column tiles for
// the narrow projections.
template <int BM, int BN, int NS = kStages>
struct GemmCfg {
  static constexpr int WM = 4;                           // waves along M
  static constexpr int WN = kWaves / WM;                 // waves along N
  static constexpr int FM = BM / WM / 16;                // 16-row fragments per wave
  static constexpr int FN = BN / WN / 16;                // 16-col fragments per wave
  static constexpr int ROWS = BM + BN;                   // rows of one stage (A then B)
  static constexpr int STAGE_BYTES = ROWS * kBK * 2;     // bf16
  static constexpr int GL = (ROWS / 8 + kWaves - 1) / kWaves;   // LDS-DMA instructions per wave per stage, one fewer ...
  static constexpr int FULL = ROWS / 8 % kWaves;                // ... from wave FULL on (0: as many)
  static constexpr int LDS_BYTES = NS * STAGE_BYTES;
  static_assert(ROWS % 8 == 0, "whole LDS-DMA instructions");
};

__device__ __forceinline__ int swz(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Epilogues: plain bf16 store, fp32 split-K slab, or the fused SwiGLU of the
// gate|up projection (weights interleaved in 64-row blocks: tile columns
// [0,64) = gate, [64,128) = up of the same 64 features; output [M, N/2]). Gated tiles of 64 and 160 columns take the gate and up rows of 32 and 80 features
// from wherever they are: a workgroup takes in 45 bytes per ns whatever its tile, so the width is chosen for one full round of the
// CUs (ops.gate_up_tile: 64 rows of 37888 x 3584 62 us in 296 workgroups of 128 columns, 44 in 237 of 160; 256 rows 112 -> 75).
enum { kEpiStore = 0, kEpiPartial = 1, kEpiSiluGU = 2 };

// GRP: routed experts. Row tile y holds rows of one expert (moe_sort with bm = BM): gtab[0] = row
// tiles, gtab[1 + y] = its expert, W [experts][N][K]; src != nullptr: row r reads X row src[r]
// (< 0: padding, any row), and rscale[r] multiplies both SwiGLU operands.
// TURN: K steps go round by column tile (and expert)
template <int BM, int BN, int EPI, int NS = kStages, bool GRP = false, bool TURN = false>
__global__ void __launch_bounds__(kWaves * 64, NS == 2 ? 2 : 1) gemm_tn_kernel(const bf16_t* __restrict__ X,
                                                                 const bf16_t* __restrict__ W, bf16_t* __restrict__ Y,
                                                                 float* __restrict__ P, int M, int N, int K, int S,
                                                                 int w_tiled, const int* __restrict__ gtab = nullptr,
                                                                 const int* __restrict__ src = nullptr,
                                                                 const float* __restrict__ rscale = nullptr, GluAct act = {}) {
  using C = GemmCfg<BM, BN, NS>;
  __shared__ __attribute__((aligned(1024))) char lds[C::LDS_BYTES];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kz = blockIdx.x % S, nt = blockIdx.x / S;
  const int n0 = nt * BN;
  const int m0 = blockIdx.y * BM;  // row tile (M may be split into BM-row tiles)
  // gated tiles that are not an interleaved block of 64: BN / 2 features' gate rows, then their up rows, wherever those are
  constexpr bool kSplitGU = EPI == kEpiSiluGU && BN != 128;
  int turn = kSplitGU ? nt * (BN / 2) >> 6 : nt;   // a block's tiles start alike, so a column's sum does not depend on the tile
  if constexpr (GRP) {
    if ((int)blockIdx.y >= gtab[0]) return;
    const int e = gtab[1 + blockIdx.y];
    W += (int64_t)e * N * K;
    turn += 5 * e;
  }
  if (!GRP || src == nullptr) X += (int64_t)m0 * K;
  // K-slice kz = K-steps [kz * TK / S, (kz + 1) * TK / S): slices differ by at most one step
  // when S does not divide TK (S = 5 puts 240 workgroups of the 48-tile qkv on 256 CUs)
  const int TK = K / kBK;
  const int t0 = kz * TK / S;
  const int kbase = t0 * kBK;
  const int T = (kz + 1) * TK / S - t0;

  // ---- LDS-DMA issue of one stage: instruction q covers rows 8q..8q+7 of the
  // stage (A rows [0, BM), then B rows [BM, BM + BN)); lane l -> row 8q + l/8,
  // LDS slot l%8, global chunk swz(row, slot).
  const int lrow = lane >> 3, lslot = lane & 7;
  int xrow[C::GL];   // X row of this lane's piece i (rows past BM are W's)
#pragma unroll
  for (int i = 0; i < C::GL; ++i) {
    xrow[i] = 8 * (w + kWaves * i) + lrow;
    if constexpr (GRP) {
      if (src != nullptr && xrow[i] < BM) xrow[i] = max(src[m0 + xrow[i]], 0);
    } else if constexpr (EPI == kEpiStore) {   // rows past M repeat the last one
      if (xrow[i] < BM) xrow[i] = min(xrow[i], M - 1 - m0);
    }
  }
  const int off = TURN ? turn % T : 0;
  auto issue_one = [&](int t, int buf, int i) {
    const int k0 = kbase + (!TURN ? t : t + off < T ? t + off : t + off - T) * kBK;
    char* sbase = lds + buf * C::STAGE_BYTES;
    {
      const int q = w + kWaves * i;
      const int row = 8 * q + lrow;
      const int chunk = swz(row, lslot);
      int wn_ = n0 + row - BM;
      if constexpr (kSplitGU) {
        const int up = row - BM >= BN / 2, f = min(nt * (BN / 2) + row - BM - up * (BN / 2), N / 2 - 1);   // past the last feature: any row
        wn_ = (f >> 6) * 128 + up * 64 + (f & 63);
      }
      // tiled W ([N/64][K/64][64][64]): each 8-row x 128-B piece of a stage is one
      // contiguous 1 KB of HBM instead of 8 separate 128-B row segments
      const bf16_t* wsrc = (w_tiled & 1) ? W + ((int64_t)(wn_ >> 6) * (K >> 6) + (k0 >> 6)) * 4096 + (wn_ & 63) * 64 + chunk * 8
                                   : W + (int64_t)wn_ * K + k0 + chunk * 8;
      const bf16_t* from = (row < BM) ? X + (int64_t)xrow[i] * K + k0 + chunk * 8 : wsrc;
      if ((w_tiled & 2) && row >= BM)   // wave-uniform (8-row pieces): weights stream non-temporal
        __builtin_amdgcn_global_load_lds(from, (__attribute__((address_space(3))) void*)(sbase + q * 1024), 16, 0, 2);
      else
        __builtin_amdgcn_global_load_lds(from, (__attribute__((address_space(3))) void*)(sbase + q * 1024), 16, 0, 0);
    }
  };
  const bool full = C::FULL == 0 || w < C::FULL;   // this wave has a last instruction
  auto issue = [&](int t, int buf) {
#pragma unroll
    for (int i = 0; i < C::GL; ++i)
      if (i < C::GL - 1 || full) issue_one(t, buf, i);
  };

  const int wm = w / C::WN, wn = w % C::WN;
  const int l15 = lane & 15, lg = lane >> 4;
  f32x4 acc[C::FM][C::FN];
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // One stage of MFMAs; the LDS-DMA pieces of stage `tn` are spread between them
  // (piece g after MFMA ((g+1) * TOT) / (GL+1)) so the issue cost of the DMA
  // overlaps MFMA execution instead of stalling both waves of a SIMD after the
  // barrier.
  constexpr int TOT = (kBK / 32) * C::FM * C::FN;
  auto compute = [&](int buf, int tn, bool do_issue) {
    const char* sbase = lds + buf * C::STAGE_BYTES;
#pragma unroll
    for (int s = 0; s < kBK / 32; ++s) {
      const int chunk = 4 * s + lg;
      u16x8 a[C::FM], b[C::FN];
#pragma unroll
      for (int i = 0; i < C::FM; ++i) {
        const int row = wm * (BM / C::WM) + 16 * i + l15;
        a[i] = *reinterpret_cast<const u16x8*>(sbase + row * 128 + (swz(row, chunk) << 4));
      }
#pragma unroll
      for (int j = 0; j < C::FN; ++j) {
        const int row = BM + wn * (BN / C::WN) + 16 * j + l15;
        b[j] = *reinterpret_cast<const u16x8*>(sbase + row * 128 + (swz(row, chunk) << 4));
      }
#pragma unroll
      for (int i = 0; i < C::FM; ++i)
#pragma unroll
        for (int j = 0; j < C::FN; ++j) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a[i]),
                                                              __builtin_bit_cast(bf16x8_t, b[j]), acc[i][j], 0, 0, 0);
          const int idx = (s * C::FM + i) * C::FN + j + 1;
#pragma unroll
          for (int g = 0; g < C::GL; ++g)
            if (idx == ((g + 1) * TOT) / (C::GL + 1) && do_issue && (g < C::GL - 1 || full)) issue_one(tn, tn % NS, g);
        }
    }
  };

  // prologue: stages 0 .. NS-2 in flight; iteration t issues stage t + NS - 1
  // into the buffer compute(t - 1) just released (fenced by the barrier)
  issue(0, 0);
#pragma unroll
  for (int st = 1; st < NS - 1; ++st)
    if (T > st) issue(st, st);
  for (int t = 0; t < T; ++t) {
    // stages issued so far: min(T, t + NS - 1); leave all but stage t in flight
    const int rem = min(T - 1 - t, NS - 2);   // stages younger than t in flight
    auto wait = [&](auto gl) {
      constexpr int GL = decltype(gl)::value;
      if (NS >= 6 && rem >= 4) wait_vmcnt<4 * GL>();
      else if (NS >= 5 && rem >= 3) wait_vmcnt<3 * GL>();
      else if (NS >= 4 && rem >= 2) wait_vmcnt<2 * GL>();
      else if (NS >= 3 && rem >= 1) wait_vmcnt<GL>();
      else wait_vmcnt<0>();
    };
    if (full) wait(std::integral_constant<int, C::GL>{});
    else wait(std::integral_constant<int, C::GL - 1>{});
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    compute(t % NS, t + NS - 1, t + NS - 1 < T);
  }

  if constexpr (EPI == kEpiSiluGU) {
    // Stage the tile through LDS (the ring is idle now) so each thread sees a
    // feature's gate and up values: HF numerics, act(bf16(g)) rounded to bf16,
    // times bf16(u), rounded.
    constexpr int LD = BN + 4;  // fp32 row stride (+4: spreads the column writes over banks)
    constexpr int HR = BM * LD * 4 <= C::LDS_BYTES ? BM : BM / 2;   // rows at a time: the whole C tile, or half of it
    static_assert(HR * LD * 4 <= C::LDS_BYTES && HR % (BM / C::WM) == 0, "C tile must fit the LDS ring, halves are whole waves'");
    float* ct = reinterpret_cast<float*>(lds);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int NO = N / 2;  // output features
#pragma unroll
    for (int h0 = 0; h0 < BM; h0 += HR) {
    __syncthreads();
    if (HR == BM || (wm * (BM / C::WM) >= h0 && wm * (BM / C::WM) < h0 + HR)) {
#pragma unroll
      for (int i = 0; i < C::FM; ++i)
#pragma unroll
        for (int j = 0; j < C::FN; ++j) {
          const int col = wn * (BN / C::WN) + 16 * j + l15;
#pragma unroll
          for (int r = 0; r < 4; ++r) ct[(wm * (BM / C::WM) - h0 + 16 * i + 4 * lg + r) * LD + col] = acc[i][j][r];
        }
    }
    __syncthreads();
    for (int v = tid; v < HR * (BN / 16); v += kWaves * 64) {
      const int row = h0 + v / (BN / 16), f0 = v % (BN / 16) * 8;
      if (kSplitGU && nt * (BN / 2) + f0 >= NO) continue;
      const float* cr = ct + (row - h0) * LD;
      float c = 1.f;
      if constexpr (GRP) c = rscale[m0 + row];
      u16x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if constexpr (GRP) {   // as the list kernel of moe.hip: one rounding
          const float g = c * cr[f0 + e], u = c * cr[BN / 2 + f0 + e];
          o[e] = f2bf(g / (1.f + __expf(-g)) * u);
        } else {
          const float g = bf2f(f2bf(cr[f0 + e])), u = bf2f(f2bf(cr[BN / 2 + f0 + e]));
          o[e] = f2bf(bf2f(f2bf(glu_gate(g, act))) * u);
        }
      }
      *reinterpret_cast<u16x8*>(Y + (int64_t)(m0 + row) * NO + nt * (BN / 2) + f0) = o;
    }
    }
  } else {
    // ---- C lane l -> row 4*lg + r, col l15 of each fragment ----
#pragma unroll
    for (int i = 0; i < C::FM; ++i)
#pragma unroll
      for (int j = 0; j < C::FN; ++j) {
        const int col = n0 + wn * (BN / C::WN) + 16 * j + l15;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = wm * (BM / C::WM) + 16 * i + 4 * lg + r;
          if constexpr (EPI == kEpiPartial) P[((int64_t)kz * M + m0 + row) * N + col] = acc[i][j][r];
          else if (GRP || m0 + row < M) Y[(int64_t)(m0 + row) * N + col] = f2bf(acc[i][j][r]);
        }
      }
  }
}

// Y[m, n] = bf16(sum_s P[s, m, n]); 4 columns per thread.
__global__ void gemm_splitk_reduce_kernel(const float* __restrict__ P, bf16_t* __restrict__ Y, int64_t MN, int S) {
  const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (i >= MN) return;
  f32x4 a = *reinterpret_cast<const f32x4*>(P + i);
  for (int s = 1; s < S; ++s) a += *reinterpret_cast<const f32x4*>(P + s * MN + i);
  uint2 o;
  o.x = pack_bf2(a[0], a[1]);
  o.y = pack_bf2(a[2], a[3]);
  *reinterpret_cast<uint2*>(Y + i) = o;
}

int splitk_reduce(const float* P, bf16_t* Y, int64_t MN, int S, hipStream_t stream) {
  if (MN % 4 != 0 || S < 1) return -1;
  const int64_t threads = MN / 4;
  gemm_splitk_reduce_kernel<<<(threads + 255) / 256, 256, 0, stream>>>(P, Y, MN, S);
  OAMD_LAUNCH_CHECK();
  return 0;
}

static bool turns(int K) { return K % 2048 == 0; }

int moe_gemm_rows(const bf16_t* X, const bf16_t* W, bf16_t* Y, int max_rows, int N, int K, int bm, bool silu_gu,
                  const int* gtab, const int* src, const float* rscale, hipStream_t stream) {
  if (max_rows == 0) return 0;
  if ((bm != 64 && bm != 128) || max_rows % bm != 0 || N % 128 != 0 || K % kBK != 0 || gtab == nullptr) return -1;
  if (silu_gu && rscale == nullptr) return -2;
  const dim3 grid(N / 128, max_rows / bm);
#define OAMD_ROWS(BM, EPI, TURN) \
  gemm_tn_kernel<BM, 128, EPI, 3, true, TURN><<<grid, kWaves * 64, 0, stream>>>(X, W, Y, nullptr, max_rows, N, K, 1, 2, gtab, src, rscale)
  if (bm == 128 && silu_gu) OAMD_ROWS(128, kEpiSiluGU, false);
  else if (bm == 128) OAMD_ROWS(128, kEpiStore, false);
  else if (turns(K) && silu_gu) OAMD_ROWS(64, kEpiSiluGU, true);
  else if (turns(K)) OAMD_ROWS(64, kEpiStore, true);
  else if (silu_gu) OAMD_ROWS(64, kEpiSiluGU, false);
  else OAMD_ROWS(64, kEpiStore, false);
#undef OAMD_ROWS
  OAMD_LAUNCH_CHECK();
  return 0;
}

int gemm_decode(const bf16_t* X, const bf16_t* W, bf16_t* Y, float* P, int M, int N, int K, int S, int BN,
                int BM, int glu, bool w_tiled_b, int stages, hipStream_t stream) {
  // bit 0: tiled W layout; bit 1: W streams with the non-temporal policy (OAMD_BF16_WNT)
  static const int wnt = [] { const char* e = getenv("OAMD_BF16_WNT"); return e && e[0] == '0' ? 0 : 2; }();
  const int w_tiled = (w_tiled_b ? 1 : 0) | wnt;
  if (BM != 64 && BM != 128 && BM != 256) return -1;
  const int mt = (M + BM - 1) / BM, Mt = mt * BM;   // tiles' rows: a part of one tile has the sums of a whole one
  if (M < 1 || (M != Mt && (M > BM || glu || S != 1))) return -1;
  const bool turn = turns(K) && Mt <= 128 && (int64_t)Mt * K <= kTurnX && (int64_t)N * S >= kTurnN * ((Mt + BM) / 64);
  if (w_tiled_b && (N % 64 != 0 || K % 64 != 0)) return -6;
  if (glu) {  // fused SwiGLU: one K slice, tiles of BN / 2 gate and as many up rows
    if ((BN != 64 && BN != 128 && BN != 160) || S != 1 || N % 128 != 0 || K % kBK != 0) return -5;
    if (BN != 128) {
      if (w_tiled_b) return -6;
      const dim3 grid((N + BN - 1) / BN, mt);
#define OAMD_GLU(BM, BNN, NSS)                                                                                                                 \
  if (turn) gemm_tn_kernel<BM, BNN, kEpiSiluGU, NSS, false, BM <= 128><<<grid, kWaves * 64, 0, stream>>>(X, W, Y, P, M, N, K, 1, w_tiled, nullptr, nullptr, nullptr, glu_act(glu)); \
  else gemm_tn_kernel<BM, BNN, kEpiSiluGU, NSS, false, false><<<grid, kWaves * 64, 0, stream>>>(X, W, Y, P, M, N, K, 1, w_tiled, nullptr, nullptr, nullptr, glu_act(glu))
      if (BM == 64 && BN == 64 && stages == 6) { OAMD_GLU(64, 64, 6); }
      else if (BM == 64 && BN == 64) { OAMD_GLU(64, 64, 4); }
      else if (BM == 64 && stages == 5) { OAMD_GLU(64, 160, 5); }
      else if (BM == 64) { OAMD_GLU(64, 160, 4); }
      else if (BM == 128 && BN == 64) { OAMD_GLU(128, 64, 4); }
      else if (BM == 128 && stages == 4) { OAMD_GLU(128, 160, 4); }
      else if (BM == 128) { OAMD_GLU(128, 160, 3); }
      else if (BN == 64 && stages == 4) { OAMD_GLU(256, 64, 4); }
      else if (BN == 64) { OAMD_GLU(256, 64, 3); }
      else { OAMD_GLU(256, 160, 3); }
#undef OAMD_GLU
      OAMD_LAUNCH_CHECK();
      return 0;
    }
    const dim3 grid(N / 128, mt);
#define OAMD_GLU(BM, NSS, TURN) \
  gemm_tn_kernel<BM, 128, kEpiSiluGU, NSS, false, TURN><<<grid, kWaves * 64, 0, stream>>>(X, W, Y, P, M, N, K, 1, w_tiled, nullptr, nullptr, nullptr, glu_act(glu))
    if (BM == 64) {
      if (stages == 2) OAMD_GLU(64, 2, false);
      else if (stages == 4 && turn) OAMD_GLU(64, 4, true);
      else if (stages == 4) OAMD_GLU(64, 4, false);
      else if (turn) OAMD_GLU(64, 3, true);
      else OAMD_GLU(64, 3, false);
    } else if (BM == 128) {
      if (stages == 4 && turn) OAMD_GLU(128, 4, true);
      else if (stages == 4) OAMD_GLU(128, 4, false);
      else if (turn) OAMD_GLU(128, 3, true);
      else OAMD_GLU(128, 3, false);
    } else {
      OAMD_GLU(256, 3, false);
    }
#undef OAMD_GLU
    OAMD_LAUNCH_CHECK();
    return 0;
  }
  if ((BN != 64 && BN != 128) || N % BN != 0) return -2;
  if (S < 1 || S > 16 || K % kBK != 0 || K / kBK < S) return -3;
  if (S > 1 && P == nullptr) return -4;
  const dim3 grid((N / BN) * S, mt);
#define OAMD_GEMM4(BM, BNN, NSS, TURN)                                                                                                        \
  if (S > 1) gemm_tn_kernel<BM, BNN, kEpiPartial, NSS, false, TURN><<<grid, kWaves * 64, 0, stream>>>(X, W, Y, P, M, N, K, S, w_tiled);         \
  else gemm_tn_kernel<BM, BNN, kEpiStore, NSS, false, TURN><<<grid, kWaves * 64, 0, stream>>>(X, W, Y, P, M, N, K, S, w_tiled)
#define OAMD_GEMM3(BM, BNN, NSS)                                                    \
  if constexpr (BM == 64 || (BM == 128 && BNN == 128)) {                            \
    if (turn) { OAMD_GEMM4(BM, BNN, NSS, true); } else { OAMD_GEMM4(BM, BNN, NSS, false); } \
  } else {                                                                          \
    OAMD_GEMM4(BM, BNN, NSS, false);                                                \
  }
#define OAMD_GEMM2(BM, BNN)                                   \
  if (stages == 2 && BM <= 128) {                              \
    OAMD_GEMM3(BM, BNN, 2);                                    \
  } else if (stages == 4 && BM + BNN <= 320) {                 \
    OAMD_GEMM3(BM, BNN, (BM + BNN <= 320 ? 4 : 3));            \
  } else if (stages == 5 && BM + BNN <= 256) {                 \
    OAMD_GEMM3(BM, BNN, (BM + BNN <= 256 ? 5 : 3));            \
  } else if (stages == 6 && BM + BNN <= 192) {                 \
    OAMD_GEMM3(BM, BNN, (BM + BNN <= 192 ? 6 : 3));            \
  } else {                                                     \
    OAMD_GEMM3(BM, BNN, 3);                                    \
  }
#define OAMD_GEMM(BM) \
  if (BN == 64) { OAMD_GEMM2(BM, 64); } else { OAMD_GEMM2(BM, 128); }
  switch (BM) {
    case 64: OAMD_GEMM(64); break;
    case 128: OAMD_GEMM(128); break;
    default: OAMD_GEMM(256); break;
  }
#undef OAMD_GEMM
#undef OAMD_GEMM2
#undef OAMD_GEMM3
#undef OAMD_GEMM4
  OAMD_LAUNCH_CHECK();
  if (S > 1 && Y != nullptr) {  // Y == nullptr: the consumer sums the slabs (rmsnorm)
    const int64_t MN = (int64_t)M * N;
    const int64_t threads = MN / 4;
    gemm_splitk_reduce_kernel<<<(threads + 255) / 256, 256, 0, stream>>>(P, Y, MN, S);
    OAMD_LAUNCH_CHECK();
  }
  return 0;
}

}  // namespace oamd
