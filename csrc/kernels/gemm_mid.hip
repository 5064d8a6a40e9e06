// GEMM for a few hundred rows: Y[M, N] = X[M, K] . W[N, K]^T, bf16 in, fp32 accumulate, bf16 out -- the
// projections of one or a few prompts, and vocabularies of up to 128 rows.
//
// What bounds it: not the matrix cores but the CUs a launch keeps busy. The 256 x 256 tiles of gemm_tile make 64
// workgroups of an 885 x 4096 product, each walking the whole K at 1.2 us per 64 columns. Here a tile is 64 to 160 rows by
// 64, 128 or 256 columns, or 192 to 256 by 128 (ops.tile_rows, ops.prompt_tile), and its K may be cut into S slices (fp32 slabs, summed by the consumer or by a reduce pass),
// so that the workgroups come close to one per CU or to whole rounds of them:
//   885 rows (weights from HBM)   6144 x 4096, 192 x 128 tiles: 45 us (96 x 256 49, 128 x 256 55); 4096 x 4096 in 2 slices, 224 x 128: 33
//                                 (128 x 256 36); 4096 x 14336 in 2, 224 x 128: 96 (101; 297 on the 256-row tiles)
//   300 rows                      28672 x 4096, 160-row tiles: 68 us (128 rows 110, 256 rows 95)
//   1500 rows                     6144 x 4096, 160-row tiles: 62 us (128 rows 93, 256 rows 90)
//   100 rows                      6144 x 4096 in 2 slices, 192 tiles of 128 x 64: 18 us (48 of 128 x 256 31); 4096 x 14336 in 4, 256 of
//                                 128 x 64: 29 (55); 28672 x 4096 gated, 224 of 128 x 128: 56 (65)
//   200 rows                      4096 x 14336 in 4 slices, 160 x 128 tiles: 37 us (96 x 256 48); 28672 x 4096 gated, 224 x 128: 60 (128 x 256 64)
//   vocabulary 128256 x 8192, 64 rows: 373 us (5.6 TB/s of weights; the 256-row tiles 422)
// The first slice carries a bias (4608 x 3584, 300 rows: 54 us in one slice, 22 in 3).
// A 128 x 256 step takes 0.63 us alone, 0.79 with every CU busy (clock). Its MFMAs are 0.47, its LDS-DMA pieces by themselves 0.45 (a CU's
// address unit takes about 20 clocks per KiB piece), its fragment reads 0.23. A wave whose piece has to wait issues no MFMA, so
// the pieces are spread over the whole step: within the 24 MFMAs behind the barrier, as before, 885 rows of 6144 x 4096 took 60 us
// and not 55, of 4096 x 4096 38 and not 35. A 64-row tile's step is no shorter than a 96-row one's (0.61, 0.65: the weight pieces).
//
// Why this shape: four waves, one per SIMD, 16 MI x 16 NW outputs each in AGPRs, so a step's fragment reads of the wide tiles stay below its
// MFMA time; three stages of those (44, 48 or 52 KiB) leave one to two steps in flight behind one barrier per step, up to six of the narrow ones as
// many bytes of the weights, which bound them. 128-B rows with the
// chunk swizzle slot ^ (bit1(row) << 1 | bit3(row) << 2) read without bank conflicts; W fragments take interleaved feature
// rows, so a lane ends with 8 neighbouring features: 16-B stores. A workgroup walks its units (tile, slice) in one
// continuous LDS-DMA stream: the next unit's first stages load while this one's outputs are stored.
#include "common.h"
#include "kernels.h"

namespace oamd {

namespace {

constexpr int kBK = 64;      // K per step: one 128-B line per row

enum { kEpiStore = 0, kEpiBias = 1, kEpiGlu = 2, kEpiPartial = 3 };   // partial: fp32 slab [M][N] of a K slice

template <int N>
__device__ __forceinline__ void vm_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// accumulator tied in AGPRs (the builtin makes hipcc copy accumulators between the files)
__device__ __forceinline__ void mfma_tied(f32x4& acc, const u16x8& a, const u16x8& b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

// act(gate) * up in the numerics of the other fused epilogues: gate, up and act(gate) rounded to bf16
__device__ __forceinline__ f32x4 glu4(const f32x4& gate, const f32x4& up, const GluAct& act) {
  f32x4 o;
#pragma unroll
  for (int r = 0; r < 4; ++r) o[r] = bf2f(f2bf(glu_gate(bf2f(f2bf(gate[r])), act))) * bf2f(f2bf(up[r]));
  return o;
}

__device__ __forceinline__ void add_bias(const bf16_t* b, f32x4& v0, f32x4& v1) {
  const u16x8 bb = *reinterpret_cast<const u16x8*>(b);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    v0[r] += bf2f(bb[r]);
    v1[r] += bf2f(bb[4 + r]);
  }
}

__device__ __forceinline__ void store8(bf16_t* y, const f32x4& v0, const f32x4& v1) {
  *reinterpret_cast<uint4*>(y) = make_uint4(pack_bf2(v0[0], v0[1]), pack_bf2(v0[2], v0[3]), pack_bf2(v1[0], v1[1]), pack_bf2(v1[2], v1[3]));
}

}  // namespace

// MI: 32-row blocks of a tile, NW: its 32-column blocks
template <int MI, int NW, int EPI>
__global__ void __launch_bounds__(256) gemm_mid_kernel(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W,
                                                       bf16_t* __restrict__ Y, const bf16_t* __restrict__ bias,
                                                       float* __restrict__ P, int M, int N, int K, int ldy, int S, GluAct act) {
  constexpr int AUX = 16;
  constexpr int kBM = 32 * MI;                   // a wave has MI X fragments and as many X pieces per step
  constexpr int kBN = 32 * NW;                   // ... and NW W fragments and pieces
  constexpr int NP = MI + NW;                    // LDS-DMA pieces of a wave per step
  constexpr int NS = 40 / NP < 6 ? 40 / NP : 6;  // stages of 4 NP KiB within 160
  constexpr int kAhead = (NS - 2) * NP;          // pieces in flight behind a step's own
  constexpr int kGroupM = 32 / MI;               // row tiles that share a W panel before the next one
  constexpr int kX = kBM * 128, kStage = kX + kBN * 128;
  __shared__ __attribute__((aligned(1024))) char lds[NS * kStage];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w >> 1, wn = w & 1;
  const int mt = (M + kBM - 1) / kBM, nt = (N + kBN - 1) / kBN, tiles = mt * nt;
  const int units = tiles * S, G = gridDim.x;
  const int slot = xcd_remap(blockIdx.x, G);
  const int TK = K / kBK, gsz = kGroupM * nt;

  auto swz = [](int row) { return (((row >> 1) & 1) << 1) | (((row >> 3) & 1) << 2); };
  const int lrow = lane >> 3, lslot = lane & 7;
  constexpr int NV = MI > NW ? MI : NW;
  uint32_t vo[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    const int row = 8 * (w + 4 * q) + lrow;
    vo[q] = ((uint32_t)row * (uint32_t)K + (uint32_t)((lslot ^ swz(row)) * 8)) * 2u;
  }
  // unit u = K slice u / tiles of tile u % tiles: first row, first column, first step, steps (slices differ by at most one)
  auto unit = [&](int u, int& m0, int& n0, int& kz, int& t0, int& T) {
    const int tile = u % tiles;
    kz = u / tiles;
    t0 = kz * TK / S;
    T = (kz + 1) * TK / S - t0;
    const int first_m = (tile / gsz) * kGroupM, gm = min(mt - first_m, kGroupM);
    m0 = (first_m + (tile % gsz) % gm) * kBM;
    n0 = ((tile % gsz) / gm) * kBN;
  };
  // the (unit, step) whose pieces go out next; an operand tile is a buffer resource (rows past M / N
  // read as zeros). Past the block's last unit its last step is loaded again, into free stages.
  int cu = slot, ck, cT;
  const bf16_t *cxp, *cwp;
  int cxn, cwn;
  auto point = [&](int u) {
    int m0, n0, kz, t0;
    unit(u, m0, n0, kz, t0, cT);
    cxp = X + (int64_t)m0 * K + t0 * kBK;
    cwp = W + (int64_t)n0 * K + t0 * kBK;
    cxn = (int)((uint32_t)min(M - m0, kBM) * (uint32_t)K * 2u - (uint32_t)t0 * (kBK * 2));
    cwn = (int)((uint32_t)min(N - n0, kBN) * (uint32_t)K * 2u - (uint32_t)t0 * (kBK * 2));
    ck = 0;
  };
  auto advance = [&]() {
    if (++ck < cT) return;
    if (cu + G < units) point(cu += G);
    else ck = cT - 1;
  };
  auto dma_ = [&](const bf16_t* cp, int cn, int step, int off, int q) {
    char* dst = lds + off + (w + 4 * q) * 1024;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)cp, (short)0, cn, 0x00020000),
                                             (__attribute__((address_space(3))) void*)dst, 16, (int)vo[q], step * (kBK * 2), 0, AUX);
  };
  // piece p of the cursor's step into stage `off`
  auto dma = [&](int off, int p) {
    if (p < MI) dma_(cxp, cxn, ck, off, p);
    else dma_(cwp, cwn, ck, off + kX, p - MI);
  };

  const int l15 = lane & 15, lq = lane >> 4;
  const int xs = swz(l15), wr = 8 * (l15 >> 2) + (l15 & 3), ws = swz(wr);
  const int xb0 = (wm * (kBM / 2) + l15) * 128, wb0 = kX + (wn * 32 + wr) * 128;
  const int xo[2] = {xb0 + ((lq ^ xs) << 4), xb0 + (((4 + lq) ^ xs) << 4)};
  const int wo[2] = {wb0 + ((lq ^ ws) << 4), wb0 + (((4 + lq) ^ ws) << 4)};
  // read f of a k-half: the X fragments, then the W ones (j = f-block * 4 + gate|up half * 2 + jj)
  auto rd = [&](int off, int h, u16x8 (&xf)[MI], u16x8 (&wf)[NW], int f) {
    if (f < MI) {
      xf[f] = *reinterpret_cast<const u16x8*>(lds + off + xo[h] + f * 2048);
    } else {
      const int j = f - MI, r = (j >> 2) * 128 + ((j >> 1) & 1) * 64 + (j & 1) * 4;
      wf[j] = *reinterpret_cast<const u16x8*>(lds + off + wo[h] + r * 128);
    }
  };

  f32x4 acc[MI][NW];
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NW; ++j) {
        acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        asm volatile("" : "+a"(acc[i][j]));
      }
    asm volatile("s_nop 4");
  };
  clear();

  // A barrier inside every step (after kBar of k-half 1's kH MFMAs) says that the step's stage has been read and the
  // next one has landed. The NP pieces of the step NS ahead go into that stage, spread over the 2 kH MFMAs up to
  // the next barrier: piece p with MFMA number p * 2 kH / NP behind it.
  constexpr int kH = NW * MI, kBar = kH / 4, kTail = kH - kBar;
  auto piece = [&](int z, int o) {
    const int p = (z * NP + 2 * kH - 1) / (2 * kH);
    if (p < NP && p * 2 * kH / NP == z) {
      dma(o, p);
      if (p == NP - 1) advance();
    }
  };
  point(slot);
#pragma unroll
  for (int st = 0; st < NS - 1; ++st) {
#pragma unroll
    for (int p = 0; p < NP; ++p) dma(st * kStage, p);
    advance();
  }
#pragma unroll
  for (int z = 0; z < kTail; ++z) piece(z, (NS - 1) * kStage);   // of the last stage, what k-half 1 of a step before would issue
  vm_wait<kAhead>();
  __builtin_amdgcn_s_barrier();
  u16x8 xa[MI], wa[NW], xb[MI], wb[NW];
#pragma unroll
  for (int f = 0; f < NP; ++f) rd(0, 0, xa, wa, f);

  int off = 0, prev = (NS - 1) * kStage;   // this step's stage, the one before
  int relax = 0;   // so many waits may leave a whole tile's stores in flight behind the pieces
  constexpr int kStores = MI * NW / (EPI == kEpiGlu ? 4 : EPI == kEpiPartial ? 1 : 2);
  static_assert(kAhead + kStores < 64 && NP <= kH, "a wait's count, a read per MFMA");
  for (int u = slot; u < units; u += G) {
    int m0, n0, kz, t0, T;
    unit(u, m0, n0, kz, t0, T);
    for (int t = 0; t < T; ++t) {
      const int nxt = off + kStage == NS * kStage ? 0 : off + kStage;
      // k-half 0; the reads of k-half 1 ride on its first MFMAs
#pragma unroll
      for (int v = 0; v < kH; ++v) {
        mfma_tied(acc[v % MI][v / MI], wa[v / MI], xa[v % MI]);
        __builtin_amdgcn_sched_barrier(0);
        if (v < NP) rd(off, 1, xb, wb, v);
        piece(kTail + v, prev);
        __builtin_amdgcn_sched_barrier(0);
      }
      // k-half 1; behind the barrier the next step's first reads ride along
#pragma unroll
      for (int v = 0; v < kH; ++v) {
        if (v == kBar) {
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          if (relax > 0) {
            vm_wait<kAhead + kStores>();
            --relax;
          } else {
            vm_wait<kAhead>();
          }
          __builtin_amdgcn_sched_barrier(0);
          __builtin_amdgcn_s_barrier();
          __builtin_amdgcn_sched_barrier(0);
        }
        mfma_tied(acc[v % MI][v / MI], wb[v / MI], xb[v % MI]);
        __builtin_amdgcn_sched_barrier(0);
        if (v < kBar) {
          piece(kTail + kH + v, prev);
        } else {
          const int z = v - kBar;
#pragma unroll
          for (int f = 0; f < NP; ++f)
            if (f * kTail / NP == z) rd(nxt, 0, xa, wa, f);
          piece(z, off);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      prev = off;
      off = nxt;
    }

    asm volatile("s_nop 7\n s_nop 7\n s_nop 7" ::: "memory");
    // a lane holds features 8 lq .. + 7 of each 32-feature block (fragments jj = 0, 1) of token l15
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int tok = m0 + wm * (kBM / 2) + i * 16 + l15;
#pragma unroll
      for (int f = 0; f < (NW + 3) / 4; ++f) {
        if constexpr (EPI == kEpiGlu) {
          f32x4 o[2];
#pragma unroll
          for (int jj = 0; jj < 2; ++jj) o[jj] = glu4(acc[i][f * 4 + jj], acc[i][f * 4 + 2 + jj], act);
          const int col = (n0 >> 1) + f * 64 + wn * 32 + 8 * lq;
          if (tok < M && 2 * col < N) store8(Y + (int64_t)tok * ldy + col, o[0], o[1]);
        } else {
#pragma unroll
          for (int ty = 0; ty < (NW == 2 ? 1 : 2); ++ty) {
            f32x4 v0 = acc[i][f * 4 + ty * 2], v1 = acc[i][f * 4 + ty * 2 + 1];
            const int col = n0 + f * 128 + ty * 64 + wn * 32 + 8 * lq;
            if (tok >= M || col >= N) continue;
            if constexpr (EPI == kEpiPartial) {
              if (bias != nullptr && kz == 0) add_bias(bias + col, v0, v1);
              float* pr = P + ((int64_t)kz * M + tok) * N + col;
              *reinterpret_cast<f32x4*>(pr) = v0;
              *reinterpret_cast<f32x4*>(pr + 4) = v1;
            } else {
              if constexpr (EPI == kEpiBias) add_bias(bias + col, v0, v1);
              store8(Y + (int64_t)tok * ldy + col, v0, v1);
            }
          }
        }
      }
    }
    // a whole tile issued kStores stores: the next waits count past them
    relax = m0 + kBM <= M && n0 + kBN <= N ? NS - 2 : 0;
    clear();
  }
  vm_wait<0>();   // the trailing re-loads land before the workgroup's LDS is released
}

template <int MI, int NW>
static void launch_mid(const bf16_t* X, const bf16_t* W, bf16_t* Y, const bf16_t* bias, float* P, int M, int N, int K, int ldy,
                       int glu, int S, int grid, hipStream_t stream) {
  if (S > 1) gemm_mid_kernel<MI, NW, kEpiPartial><<<grid, 256, 0, stream>>>(X, W, Y, bias, P, M, N, K, ldy, S, GluAct{});
  else if (bias) gemm_mid_kernel<MI, NW, kEpiBias><<<grid, 256, 0, stream>>>(X, W, Y, bias, P, M, N, K, ldy, S, GluAct{});
  else if (!glu) gemm_mid_kernel<MI, NW, kEpiStore><<<grid, 256, 0, stream>>>(X, W, Y, bias, P, M, N, K, ldy, S, GluAct{});
  else if constexpr (NW >= 4) gemm_mid_kernel<MI, NW, kEpiGlu><<<grid, 256, 0, stream>>>(X, W, Y, bias, P, M, N, K, ldy, S, glu_act(glu));
}

int gemm_mid(const bf16_t* X, const bf16_t* W, bf16_t* Y, const bf16_t* bias, float* P, int M, int N, int K, int ldy, int glu,
             int S, int rows, int cols, hipStream_t stream) {
  if (M < 1 || N < 16 || N % 16 || K % kBK || S < 1 || S > 16 || K / kBK < S) return -1;
  if (glu && (N % 128 || bias)) return -2;
  if (S > 1 && P == nullptr) return -3;
  if (Y == nullptr ? (S == 1 || glu) : (ldy % 8 || reinterpret_cast<uintptr_t>(Y) % 16)) return -4;
  if (S > 1 && Y != nullptr && ldy != (glu ? N / 2 : N)) return -5;
  const int64_t units = (int64_t)((M + rows - 1) / rows) * ((N + cols - 1) / cols) * S;
  if (units > (1LL << 30)) return -6;
  if (cols == 64 && glu && S == 1) return -7;
  const int grid = (int)min((int64_t)device_cus(), units);
#define OAMD_MID(R, C) \
  if (rows == R && cols == C) launch_mid<R / 32, C / 32>(X, W, Y, bias, P, M, N, K, ldy, glu, S, grid, stream)
  OAMD_MID(96, 256);
  else OAMD_MID(128, 256);
  else OAMD_MID(160, 256);
  else OAMD_MID(64, 256);
  else OAMD_MID(64, 128);
  else OAMD_MID(96, 128);
  else OAMD_MID(128, 128);
  else OAMD_MID(160, 128);
  else OAMD_MID(192, 128);
  else OAMD_MID(224, 128);
  else OAMD_MID(256, 128);
  else OAMD_MID(64, 64);
  else OAMD_MID(128, 64);
  else return -8;
#undef OAMD_MID
  OAMD_LAUNCH_CHECK();
  if (S == 1 || Y == nullptr) return 0;
  return glu ? splitk_silu(P, Y, M, N, S, glu, stream) : splitk_reduce(P, Y, (int64_t)M * N, S, stream);
}

}  // namespace oamd
