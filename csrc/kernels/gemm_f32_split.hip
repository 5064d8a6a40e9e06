// fp32 products on the bf16 matrix instruction: each operand as the sum of three bf16 numbers (8 significand bits each: all 24 are kept),
// six of the nine partial products, 32-bit sums. What is left out, the second part of one operand by the third of the other and the third
// by the third, is at most 2^-24 of a product (just above a power of two: 1.0038986 squared), an fp32 rounding, and 2^-26.5
// of evenly spread ones (root mean square); this is the splitting of Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations" (2019). A sum is rounded 6 times per 16 columns where the fp32 instruction rounds it for each: 962 rows of
// 2048 x 2048 are 7.0e-7 from the 64-bit result (the fp32 instruction's 8.1e-7), of 2048 x 8192 in one slice 1.4e-6 (1.6e-6), in four 7.3e-7.
//
// What bounds it: the bf16 matrix instruction's power. Six partial products are 192 clocks of MFMAs per 32 x 32 x 16 products where the fp32
// instruction takes 512. An operand element costs 6 VALU instructions, done once per workgroup on the way into LDS and spread between
// the MFMAs of the step before; at the clock that is left 213 TFLOP/s (1.3 PFLOP/s of bf16 products, what a large bf16 product reaches), against
// 122 of the fp32 instruction's kernel:
//   962 rows   16384 x 2048 gated 560 -> 315 us, 2048 x 8192 298 -> 168, 2048 x 2048 80 -> 54
//   2018 rows  16384 x 2048 gated 1110 -> 634          40 rows   16384 x 2048 gated 80 -> 37, 2048 x 8192 91 -> 36
//
// Why this shape: 256 rows x 128 features are 8 waves of 64 x 64, two per SIMD, so one wave's conversions, reads and waits run under the
// other's MFMAs (four waves of 64 x 64 took 728 us where these take 634), and both operands' parts fit in LDS twice (147 KB): one barrier per
// 32 columns. Pieces are requested two steps before they are split, in registers. With fewer rows 128-row tiles of eight waves
// and 64-row ones of four, two to a CU, fill more CUs (ops.f32_split_rows); all sum K in the same order, and what
// is done again is so by itself, so the bits are the same.
#include <utility>

#include "common.h"
#include "f32_piece.h"
#include "gemm_f32.h"
#include "kernels.h"

namespace oamd {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// f(0) .. f(N - 1) with the numbers as constants: a loop this long is not unrolled whole
template <class F, int... I>
__device__ __forceinline__ void each(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}

// (a, b) rounded to bf16, a in the low half
__device__ __forceinline__ uint32_t cvt2(float a, float b) {
  uint32_t r;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// One of the three parts of (a, b): what is left of them, rounded to nearest; (a, b) is then what is left after it, exactly. The three
// sum to the value (to 2^-134 where the third would fall below bf16's range). An infinity, a NaN or a value that rounds to an
// infinity leaves a NaN behind, which reaches every sum it is part of.
__device__ __forceinline__ uint32_t part(float& a, float& b) {
  const uint32_t q = cvt2(a, b);
  a -= __uint_as_float(q << 16);
  b -= __uint_as_float(q & 0xffff0000u);
  return q;
}

}  // namespace

// Y[M, N] = X[M, K] W[N, K]^T (GLU: act of the interleaved gate | up rows, PART: K slice blockIdx.z of S into its slab), tiles of
// 32 WM TB tokens x 128 rows of W; 2 WM waves of 32 TB tokens x 64.
template <int WM, int TB, bool GLU, bool PART>
__global__ void __launch_bounds__(128 * WM, 2) gemm_f32_split_kernel(const GemmF32 a) {
  constexpr int kX = 32 * WM * TB, kPass = 32 * WM, kRows = kX + 128, kPlane = kRows * 64, kBuf = 3 * kPlane, NR = kRows / kPass;
  __shared__ __attribute__((aligned(1024))) char lds[2 * kBuf];
  __shared__ uint32_t kind[kRows / 4];   // a byte per row of X and W: 1 it holds an operand of 2^32 or more, 2 one other than 0
  const int K = a.K;
  const int lid = xcd_remap(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
  const int m0 = lid % gridDim.x * kX, n0 = lid / gridDim.x * 128;
  int kbase = 0, kend = K;
  if constexpr (PART) {
    const int T = (K + 31) / 32;
    kbase = (int)blockIdx.z * T / a.S * 32;
    kend = min(K, ((int)blockIdx.z + 1) * T / a.S * 32);
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wm = w >> 1, wn = w & 1;

  // loader: thread -> 8 columns 8 (tid % 4) of rows tid / 4 + 32 WM i of a 32-column piece, X's rows, then W's; rows past M / N repeat the last
  const int lr = tid >> 2, lc = tid & 3;
  const float* src[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int row = lr + kPass * i;
    src[i] = row < kX ? a.X + min(m0 + row, a.M - 1) * a.ldx : a.W + (int64_t)min(n0 + row - kX, a.N - 1) * K;
  }
  struct Piece { f32x4 v[2 * NR]; } even, uneven;
  auto load = [&](Piece& p, int i, int k) {
    const float* from = src[i] + split_column(k, lc, K);
    p.v[2 * i] = *reinterpret_cast<const f32x4*>(from);
    p.v[2 * i + 1] = *reinterpret_cast<const f32x4*>(from + 4);
  };
  // a plane's row is 64 B, its 16-B chunk c in slot c ^ (row / 4 % 4): 16 neighbouring rows' chunks c lie in the 64 banks once
  char* to = lds + lr * 64 + ((lc ^ (lr >> 2 & 3)) << 4);
  const int l31 = lane & 31, half = lane >> 5, sw = l31 >> 2 & 3;
  const char *xr = lds + (wm * 32 * TB + l31) * 64, *wr = lds + (kX + wn * 32 + l31) * 64;

  f32x16 acc[2][TB] = {};   // [W rows 32 wn and 64 + 32 wn][token block]
  constexpr int NF = 3 * (TB + 2);   // fragments of a 16-column half
  bf16x8 xf[2][3][TB], wf[2][3][2];
  // partial product p: part pw[p] of W by part px[p] of X, the small ones first; fragments in the order in which they are used
  constexpr int pw[6] = {0, 2, 1, 0, 1, 0}, px[6] = {2, 0, 1, 1, 0, 0}, order[3] = {0, 2, 1};
  auto rd = [&](int buf, int h, int i) {
    const int at = buf * kBuf + (((2 * h + half) ^ sw) << 4), s = i / (TB + 2), j = i % (TB + 2);
    if (j < 2) wf[h][order[s]][j] = *reinterpret_cast<const bf16x8*>(wr + order[s] * kPlane + j * 4096 + at);
    else xf[h][2 - order[s]][j - 2] = *reinterpret_cast<const bf16x8*>(xr + (2 - order[s]) * kPlane + (j - 2) * 2048 + at);
  };
  constexpr int kH = 12 * TB;   // MFMAs of a half
  auto mul = [&](int h, int v) {
    const int p = v / (2 * TB), b = v / TB % 2, i = v % TB;
    acc[b][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[h][pw[p]][b], xf[h][px[p]][i], acc[b][i], 0, 0, 0);
  };
  // level l of the work that makes a piece's parts: part l % 3 of pair l / 3 % 4 of 16-B row chunk l / 12; behind a chunk's last level
  // its parts are written and its registers are requested again, two pieces on
  constexpr int NL = 12 * NR;
  uint32_t q[3][4];
  float most[NR] = {};   // of the magnitudes of this thread's part of its rows
  auto level = [&](Piece& p, int buf, int l, int k) {
    const int i = l / 12, j = l / 3 % 4, s = l % 3;
    f32x4 v = p.v[2 * i + (j >> 1)];
    float a = v[2 * (j & 1)], b = v[2 * (j & 1) + 1];
    if (s == 0) asm volatile("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(most[i]) : "v"(a), "v"(b));   // here, or the operands are kept for later
    q[s][j] = s < 2 ? part(a, b) : cvt2(a, b);
    v[2 * (j & 1)] = a;
    v[2 * (j & 1) + 1] = b;
    p.v[2 * i + (j >> 1)] = v;
    if (l % 12 == 11) {
#pragma unroll
      for (int z = 0; z < 3; ++z) *reinterpret_cast<uint4*>(to + buf * kBuf + z * kPlane + i * (kPass * 64)) = make_uint4(q[z][0], q[z][1], q[z][2], q[z][3]);
      load(p, i, k);
    }
  };
  auto clear_tail = [&](Piece& p, int k) {
    if (k + 32 > K && lc >= 2) {   // K % 32 == 16: the last piece is 16 columns
#pragma unroll
      for (int i = 0; i < 2 * NR; ++i) p.v[i] = f32x4{};
    }
  };
  // The step of columns k .. + 31, whose parts are in buffer `buf`: the next piece's parts go into the other one between its MFMAs; a barrier
  // behind the last of them, and the next step's first fragments are read under the MFMAs that are left.
  constexpr int kBar = 2 * kH - (NF + 1) / 2;
  auto step = [&](Piece& next, int buf, int k) {
    clear_tail(next, k + 32);
    each([&](auto at) {
      constexpr int v = at, l0 = v * NL / kBar, l1 = (v + 1) * NL / kBar, f0 = 2 * (v - kBar);
      mul(v / kH, v % kH);
      __builtin_amdgcn_sched_barrier(0);
      if (v < NF) rd(buf, 1, v);
      if (v < kBar) {
#pragma unroll
        for (int i = 0; i < (NL + kBar - 1) / kBar; ++i)
          if (l0 + i < l1) level(next, 1 - buf, l0 + i, k + 96);
        if (v == kBar - 1) __syncthreads();
      } else {
        rd(1 - buf, 0, f0);
        if (f0 + 1 < NF) rd(1 - buf, 0, f0 + 1);
      }
      __builtin_amdgcn_sched_barrier(0);
    }, std::make_integer_sequence<int, 2 * kH>{});
  };
#pragma unroll
  for (int i = 0; i < NR; ++i) load(even, i, kbase);
#pragma unroll
  for (int i = 0; i < NR; ++i) load(uneven, i, kbase + 32);
  clear_tail(even, kbase);
#pragma unroll
  for (int l = 0; l < NL; ++l) level(even, 0, l, kbase + 64);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NF; ++i) rd(0, 0, i);
  int k = kbase;
  for (; k + 32 < kend; k += 64) {
    step(uneven, 0, k);
    step(even, 1, k + 32);
  }
  if (k < kend) step(uneven, 0, k);

  // What is done again in 32-bit products: a sum that is infinite or NaN (so are operands, or one rounds to infinity in bf16), and one whose
  // operands may have lost parts that count. Parts lose what lies below 2^-126, so a product of operands below 2^32 is off by 2^-92 at most, and
  // a sum of up to 2^20 of them by no more than an fp32 rounding of 2^-48: a sum below that (0 too, but for rows of zeros) or of a row with an
  // operand of 2^32 or more is done again. Largest and not smallest operands are looked for, as zeros are common and half an instruction
  // finds the largest (2018 rows of 16384 x 2048 gated 655 us with and without on 256-row tiles, 832 and 797 on 64-row ones). That sum alone is replaced: the wave does its block again, but the others stay as they are, whoever shares the block.
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const uint64_t large = __ballot(most[i] >= 0x1p32f), some = __ballot(most[i] != 0.f);
    if (lc == 0) reinterpret_cast<char*>(kind)[lr + kPass * i] = (large >> lane & 15 ? 1 : 0) | (some >> lane & 15 ? 2 : 0);
  }
  __syncthreads();
  int kx[TB];
  uint32_t kw[2][4];   // of rows 8 q + 4 half .. + 3
#pragma unroll
  for (int i = 0; i < TB; ++i) kx[i] = reinterpret_cast<const char*>(kind)[(wm * TB + i) * 32 + l31];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int z = 0; z < 4; ++z) kw[b][z] = kind[(kX + 64 * b + wn * 32 + 8 * z) / 4 + half];
  auto odd = [&](int b, int i, int r) {
    const float v = fabsf(acc[b][i][r]);
    const int w = kw[b][r >> 2] >> 8 * (r & 3);
    return !(v <= 3.4028234e38f) || ((kx[i] | w) & 1) || (v < 0x1p-48f && (kx[i] & w & 2));
  };
  float odds = 0.f, least = 0x1p32f;   // NaN where a sum is no number; the smallest: most blocks are passed by these
  uint32_t kinds = 0;
  bool any = false;
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int i = 0; i < TB; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        odds = __builtin_fmaf(acc[b][i][r], 0.f, odds);
        least = fminf(least, fabsf(acc[b][i][r]));
        kinds |= kx[i] | kw[b][r >> 2];
      }
  if (odds != 0.f || least < 0x1p-48f || (kinds & 0x01010101)) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < TB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) any |= odd(b, i, r);
  }
  if (__any(any)) {
#pragma unroll
    for (int i = 0; i < TB; ++i) {
      const float* x = a.X + min(m0 + (wm * TB + i) * 32 + l31, a.M - 1) * a.ldx + 4 * half;
      const float *w0 = a.W + (int64_t)min(n0 + wn * 32 + l31, a.N - 1) * K + 4 * half, *w1 = a.W + (int64_t)min(n0 + 64 + wn * 32 + l31, a.N - 1) * K + 4 * half;
      f32x16 g{}, u{};
      for (int k = kbase; k < kend; k += 8) {
        const f32x4 xv = *reinterpret_cast<const f32x4*>(x + k), gv = *reinterpret_cast<const f32x4*>(w0 + k), uv = *reinterpret_cast<const f32x4*>(w1 + k);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          g = __builtin_amdgcn_mfma_f32_32x32x2f32(gv[e], xv[e], g, 0, 0, 0);
          u = __builtin_amdgcn_mfma_f32_32x32x2f32(uv[e], xv[e], u, 0, 0, 0);
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[0][i][r] = odd(0, i, r) ? g[r] : acc[0][i][r];
        acc[1][i][r] = odd(1, i, r) ? u[r] : acc[1][i][r];
      }
    }
  }

  // a lane holds rows 8 q + 4 half .. + 3 of each 32-row block of W, of token l31
  const int NO = GLU && !PART ? a.N / 2 : a.N;
#pragma unroll
  for (int i = 0; i < TB; ++i) {
    const int m = m0 + (wm * TB + i) * 32 + l31;
    if (m >= a.M) continue;
    float* yr = PART ? a.P + ((int64_t)blockIdx.z * a.M + m) * a.N : a.Y + m * a.ldy;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int f = wn * 32 + 8 * q + 4 * half;
      f32x4 v[2];
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[b][r] = acc[b][i][4 * q + r];
      if constexpr (GLU && !PART) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[0][r] = glu1(v[0][r], v[1][r], a.act);
        put4(yr + (n0 >> 1) + f, v[0], NO - (n0 >> 1) - f, a.vec);
      } else {
#pragma unroll
        for (int b = 0; b < 2; ++b) put4(yr + n0 + 64 * b + f, v[b], NO - n0 - 64 * b - f, PART ? a.N % 4 == 0 : a.vec);
      }
    }
  }
}

template <int WM, int TB>
static void launch_split(const GemmF32& a, bool glu, hipStream_t stream) {
  const dim3 grid((a.M + 32 * WM * TB - 1) / (32 * WM * TB), (a.N + 127) / 128, a.S);
  if (a.S > 1 && glu) gemm_f32_split_kernel<WM, TB, true, true><<<grid, 128 * WM, 0, stream>>>(a);
  else if (a.S > 1) gemm_f32_split_kernel<WM, TB, false, true><<<grid, 128 * WM, 0, stream>>>(a);
  else if (glu) gemm_f32_split_kernel<WM, TB, true, false><<<grid, 128 * WM, 0, stream>>>(a);
  else gemm_f32_split_kernel<WM, TB, false, false><<<grid, 128 * WM, 0, stream>>>(a);
}

int gemm_f32_split(const GemmF32& a, bool glu, int rows, hipStream_t stream) {
  if ((a.N + 127) / 128 > 65535) return -1;
  if (rows == 64) launch_split<2, 1>(a, glu, stream);
  else if (rows == 128) launch_split<4, 1>(a, glu, stream);
  else launch_split<4, 2>(a, glu, stream);
  return 0;
}

}  // namespace oamd
