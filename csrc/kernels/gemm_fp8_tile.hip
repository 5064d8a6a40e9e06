// FP8 (e4m3fn) GEMM for prompts: Y[M, N] = (X8[M, K] . W8[N, K]^T) * sx[m] * sw[n], fp32 accumulate, bf16 out.
//
// What bounds it: what a CU takes in (a 128-row step's 48 pieces of 1 KiB are 960 clocks of its address unit, its MFMAs 1024) and
// the rounds of tiles on the CUs. This is gemm_mid's continuous pipeline (tiles of 96, 128 or 160 rows by 256 columns,
// ops.fp8_tile_rows, four waves of 16 MI x 128 outputs in AGPRs, three stages filled by LDS-DMA, units (tile, K slice) walked
// by persistent workgroups) with 128 of K per 128-B line. The f8f6f4 MFMA of unit block scales takes a whole line of 16
// rows, so a step's fragments are read one step ahead, each W fragment into the registers of the one just used, while
// the MFMAs of this step run, and the stage that was read goes back to the LDS-DMA, its pieces spread over the step.
//   57344 x 8192: 512 rows 306 -> 218 us (gemm_fp8 before), 8640 rows 4.78 -> 3.28 ms (2.5 PFLOP/s; 128-row tiles 3.37)
//   8192 x 28672: 1200 rows 440 -> 215 us (128-row tiles 354); 8192 x 8192: 700 rows 69 -> 48 (57), 4096 rows 287 -> 203
// Fragments, steps and slices are gemm_fp8's, so the sums are the same bits.
// The row and column scales of a unit come through LDS-DMA too, behind its first steps: a plain load would make the
// epilogue wait for the stages in flight.
#include "common.h"
#include "kernels.h"

namespace oamd {

namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kBN = 256;              // tile columns
constexpr int kBK = 128;              // K (bytes) per step: one 128-B line per row
constexpr int kMinSteps = 3;          // steps of a unit: its scales have landed when it ends

template <int N>
__device__ __forceinline__ void vm_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// accumulator tied in AGPRs; an operand written by a vector instruction is readable two wait states later (the
// compiler sees no MFMA here, and the slots pass under the one before)
__device__ __forceinline__ void mfma_tied(f32x4& acc, const v8i& a, const v8i& b) {
  asm volatile("s_nop 1\n v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

}  // namespace

// MI: 32-row blocks of a tile
template <int MI, bool PARTIAL>
__global__ void __launch_bounds__(256) gemm_fp8_tile_kernel(const uint8_t* __restrict__ X, const uint8_t* __restrict__ W,
                                                            const float* __restrict__ sx, const float* __restrict__ sw,
                                                            bf16_t* __restrict__ Y, float* __restrict__ P, int M, int N, int K, int S) {
  constexpr int AUX = 16;
  constexpr int kBM = 32 * MI;       // a wave has MI X fragments and as many X pieces per step
  constexpr int NP = MI + 8;         // LDS-DMA pieces of a wave per step
  constexpr int NS = 3;              // stages
  constexpr int kGroupM = 32 / MI;   // row tiles that share a W panel before the next one
  constexpr int kX = kBM * kBK, kStage = kX + kBN * kBK;
  constexpr int kScales = NS * kStage, kScaleBytes = (kBN + 256) * 4;   // sw, then sx; two sets
  __shared__ __attribute__((aligned(1024))) char lds[kScales + 2 * kScaleBytes];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w >> 1, wn = w & 1;
  const int mt = (M + kBM - 1) / kBM, nt = (N + kBN - 1) / kBN, tiles = mt * nt;
  const int units = tiles * S, G = gridDim.x;
  const int slot = xcd_remap(blockIdx.x, G);
  const int TK = K / kBK, gsz = kGroupM * nt;

  // chunk swizzles of gemm_fp8 over the lane's fragment row: rows of X in order, of W 8 (l15 >> 2) + (l15 & 3)
  auto swz_x = [](int row) { return ((row >> 1) & 1) | (((row >> 2) & 1) << 2); };
  auto swz_w = [](int row) { return ((row >> 1) & 1) | (((row >> 3) & 1) << 2); };
  const int lrow = lane >> 3, lslot = lane & 7;
  uint32_t vx[MI], vw[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int row = 8 * (w + 4 * q) + lrow;
    vw[q] = (uint32_t)row * (uint32_t)K + (uint32_t)((lslot ^ swz_w(row)) * 16);
    if (q < MI) vx[q < MI ? q : 0] = (uint32_t)row * (uint32_t)K + (uint32_t)((lslot ^ swz_x(row)) * 16);
  }
  // unit u = K slice u / tiles of tile u % tiles: first row, first column, first step, steps
  auto unit = [&](int u, int& m0, int& n0, int& kz, int& t0, int& T) {
    const int tile = u % tiles;
    kz = u / tiles;
    t0 = kz * TK / S;
    T = (kz + 1) * TK / S - t0;
    const int first_m = (tile / gsz) * kGroupM, gm = min(mt - first_m, kGroupM);
    m0 = (first_m + (tile % gsz) % gm) * kBM;
    n0 = ((tile % gsz) / gm) * kBN;
  };
  // the (unit, step) whose pieces go out next; an operand tile is a buffer resource (rows past M / N read as
  // zeros). Past the block's last unit its last step is loaded again, into free stages.
  int cu = slot, ck, cT;
  const uint8_t *cxp, *cwp;
  int cxn, cwn;
  auto point = [&](int u) {
    int m0, n0, kz, t0;
    unit(u, m0, n0, kz, t0, cT);
    cxp = X + (int64_t)m0 * K + t0 * kBK;
    cwp = W + (int64_t)n0 * K + t0 * kBK;
    cxn = (int)((uint32_t)min(M - m0, kBM) * (uint32_t)K - (uint32_t)t0 * kBK);
    cwn = (int)((uint32_t)min(N - n0, kBN) * (uint32_t)K - (uint32_t)t0 * kBK);
    ck = 0;
  };
  auto advance = [&]() {
    if (++ck < cT) return;
    if (cu + G < units) point(cu += G);
    else ck = cT - 1;
  };
  auto dma_ = [&](const uint8_t* cp, int cn, uint32_t vo, int step, int off, int q) {
    char* dst = lds + off + (w + 4 * q) * 1024;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)cp, (short)0, cn, 0x00020000),
                                             (__attribute__((address_space(3))) void*)dst, 16, (int)vo, step * kBK, 0, AUX);
  };
  // piece p of the cursor's step into stage `off`: W first (it comes from further away)
  auto dma = [&](int off, int p) {
    if (p < 8) dma_(cwp, cwn, vw[p], ck, off + kX, p);
    else dma_(cxp, cxn, vx[p - 8], ck, off, p - 8);
  };
  // 64 column scales per wave and 64 row scales (past the tile's: zeros): 2 pieces
  auto scales = [&](int m0, int n0, int set) {
    char* dst = lds + kScales + set * kScaleBytes;
    const float *swp = sw + n0, *sxp = sx + m0;
    const int swn = min(N - n0, kBN) * 4, sxn = min(M - m0, kBM) * 4;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)swp, (short)0, swn, 0x00020000),
                                             (__attribute__((address_space(3))) void*)(dst + w * 256), 4, (w * 64 + lane) * 4, 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)sxp, (short)0, sxn, 0x00020000),
                                             (__attribute__((address_space(3))) void*)(dst + kBN * 4 + w * 256), 4,
                                             (w * 64 + lane) * 4, 0, 0, 0);
  };

  const int l15 = lane & 15, lq = lane >> 4;
  const int xs = swz_x(l15), wr = 8 * (l15 >> 2) + (l15 & 3), ws = swz_w(wr);
  const int xb0 = (wm * (kBM / 2) + l15) * 128, wb0 = kX + (wn * 32 + wr) * 128;
  const int xo[2] = {xb0 + (((2 * lq) ^ xs) << 4), xb0 + (((2 * lq + 1) ^ xs) << 4)};
  const int wo[2] = {wb0 + (((2 * lq) ^ ws) << 4), wb0 + (((2 * lq + 1) ^ ws) << 4)};
  // a fragment: chunks 2 lq and 2 lq + 1 of its row, as gemm_fp8 (the same sums, bit for bit) (W fragment j = f-block * 4 + 64-column half * 2 + jj)
  auto frag = [&](int a0, int a1) -> v8i {
    const v4i lo = *reinterpret_cast<const v4i*>(lds + a0), hi = *reinterpret_cast<const v4i*>(lds + a1);
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto xfrag = [&](int off, int i) { return frag(off + xo[0] + i * 2048, off + xo[1] + i * 2048); };
  auto wfrag = [&](int off, int j) {
    const int r = ((j >> 2) * 128 + ((j >> 1) & 1) * 64 + (j & 1) * 4) * 128;
    return frag(off + wo[0] + r, off + wo[1] + r);
  };

  f32x4 acc[MI][8];
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        asm volatile("" : "+a"(acc[i][j]));
      }
    asm volatile("s_nop 4");
  };
  clear();

  point(slot);
#pragma unroll
  for (int st = 0; st < NS; ++st) {
#pragma unroll
    for (int p = 0; p < NP; ++p) dma(st * kStage, p);
    advance();
  }
  vm_wait<(NS - 1) * NP>();
  __builtin_amdgcn_s_barrier();
  v8i xf[MI], wf[8];
#pragma unroll
  for (int i = 0; i < MI; ++i) xf[i] = xfrag(0, i);
#pragma unroll
  for (int j = 0; j < 8; ++j) wf[j] = wfrag(0, j);

  int off = 0;       // this step's stage
  int relax = 0;     // steps whose wait may leave a whole tile's stores and scales in flight behind the pieces
  constexpr int kStores = MI * (PARTIAL ? 8 : 4);
  int set = 0;
  for (int u = slot; u < units; u += G, set ^= 1) {
    int m0, n0, kz, t0, T;
    unit(u, m0, n0, kz, t0, T);
    scales(m0, n0, set);
    for (int t = 0; t < T; ++t) {
      // This step's fragments are in registers: every wave has read its stage, so the step NS ahead goes into it, and
      // the next stage, landed, is read: a W fragment into the registers of the one just used, X beside this step's.
      const int nxt = off + kStage == NS * kStage ? 0 : off + kStage;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (relax > 0) {
        vm_wait<(NS - 2) * NP + kStores + 2>();
        --relax;
      } else {
        vm_wait<(NS - 2) * NP>();
      }
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      v8i xn[MI];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          const int v = j * MI + i;
          mfma_tied(acc[i][j], wf[j], xf[i]);
          __builtin_amdgcn_sched_barrier(0);
          if (v % 8 == 1) xn[v / 8] = xfrag(nxt, v / 8);
          if (i == MI - 1) wf[j] = wfrag(nxt, j);
          const int p = (v * NP + 8 * MI - 1) / (8 * MI);   // a piece every 8 MI / NP MFMAs
          if (p < NP && p * 8 * MI / NP == v) dma(off, p);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
#pragma unroll
      for (int i = 0; i < MI; ++i) xf[i] = xn[i];
      advance();
      off = nxt;
    }

    asm volatile("s_nop 7\n s_nop 7\n s_nop 7" ::: "memory");
    const float* sc = reinterpret_cast<const float*>(lds + kScales + set * kScaleBytes);
    // a lane holds features 8 lq .. + 7 of each 32-feature block (fragments jj = 0, 1) of token l15
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int rt = wm * (kBM / 2) + i * 16 + l15, tok = m0 + rt;
      const float sr = sc[kBN + rt];
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int ty = 0; ty < 2; ++ty) {
          __builtin_amdgcn_sched_barrier(0);   // one block's scales in registers at a time
          const int ct = f * 128 + ty * 64 + wn * 32 + 8 * lq, col = n0 + ct;
          f32x4 v0 = acc[i][f * 4 + ty * 2], v1 = acc[i][f * 4 + ty * 2 + 1];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            v0[r] = v0[r] * sr * sc[ct + r];
            v1[r] = v1[r] * sr * sc[ct + 4 + r];
          }
          if (tok >= M || col >= N) continue;
          if constexpr (PARTIAL) {
            float* pr = P + ((int64_t)kz * M + tok) * N + col;
            *reinterpret_cast<f32x4*>(pr) = v0;
            *reinterpret_cast<f32x4*>(pr + 4) = v1;
          } else {
            *reinterpret_cast<uint4*>(Y + (int64_t)tok * N + col) =
                make_uint4(pack_bf2(v0[0], v0[1]), pack_bf2(v0[2], v0[3]), pack_bf2(v1[0], v1[1]), pack_bf2(v1[2], v1[3]));
          }
        }
    }
    relax = m0 + kBM <= M && n0 + kBN <= N ? NS - 1 : 0;
    clear();
  }
  vm_wait<0>();   // the trailing re-loads land before the workgroup's LDS is released
}

template <int MI>
static void launch_fp8(const uint8_t* X, const uint8_t* W, const float* sx, const float* sw, bf16_t* Y, float* P, int M, int N, int K,
                       int S, int grid, hipStream_t stream) {
  if (S > 1) gemm_fp8_tile_kernel<MI, true><<<grid, 256, 0, stream>>>(X, W, sx, sw, Y, P, M, N, K, S);
  else gemm_fp8_tile_kernel<MI, false><<<grid, 256, 0, stream>>>(X, W, sx, sw, Y, P, M, N, K, S);
}

int gemm_fp8_tile(const uint8_t* X, const uint8_t* W, const float* sx, const float* sw, bf16_t* Y, float* P, int M, int N, int K,
                  int S, int rows, hipStream_t stream) {
  if (M <= 0) return 0;
  if (N < 16 || N % 16 || K % kBK || S < 1 || S > 16 || K / kBK / S < kMinSteps) return -1;
  if (reinterpret_cast<uintptr_t>(X) % 16 || reinterpret_cast<uintptr_t>(W) % 16) return -2;
  if (S > 1 ? P == nullptr : Y == nullptr) return -3;
  if (rows != 96 && rows != 128 && rows != 160) return -5;
  const int64_t units = (int64_t)((M + rows - 1) / rows) * ((N + kBN - 1) / kBN) * S;
  if (units > (1LL << 30) || (int64_t)K * kBN >= (1LL << 31)) return -4;
  const int grid = (int)min((int64_t)device_cus(), units);
  if (rows == 96) launch_fp8<3>(X, W, sx, sw, Y, P, M, N, K, S, grid, stream);
  else if (rows == 128) launch_fp8<4>(X, W, sx, sw, Y, P, M, N, K, S, grid, stream);
  else launch_fp8<5>(X, W, sx, sw, Y, P, M, N, K, S, grid, stream);
  OAMD_LAUNCH_CHECK();
  return S > 1 && Y != nullptr ? splitk_reduce(P, Y, (int64_t)M * N, S, stream) : 0;
}

}  // namespace oamd
