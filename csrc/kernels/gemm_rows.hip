// GEMM for the fewest rows (one to eight): Y[M, N] = X[M, K] . W[N, K]^T, bf16 in, fp32 sums.
//
// Nothing but the weights' stream bounds it. On the matrix units a wave's load takes 64 B of each of 16 rows, half a line a request,
// and reaches 4.5 to 5.8 TB/s; here a wave reads 1 KB of one row per request, past the caches (nothing is read twice): 6.9 TB/s, where a bare
// read loop reaches 7.2. The products are v_dot2 on the vector units, which eight rows still leave behind the stream; X stays in
// registers, so a workgroup reads it once for all its rows of W. Four waves share K; a row's sums go over 16 lanes by DPP and over the
// rest through LDS at the workgroup's end, with no barrier inside the stream. Two register sets of RF rows each are in flight by turns.
// With an RMSNorm in front of it (decode steps of one to four rows, where that kernel is a launch of 4.5 us) every workgroup normalises the rows while
// its first rows of W are under way; the first workgroup stores the residual stream, in a buffer of its own as others still read the old
// one. One row, us with rmsnorm and without: 6144 x 4096 13.4, 10.7; 4096 x 4096 10.7, 7.9; 28672 x 4096 gated 41, 38; 128256 x 4096 163, 154.
// Measured against gemm_skinny, us: 128256 x 4096 of 1, 4 and 8 rows 151, 155, 164 (183, 199, 217); one row of 28672 x 4096 gated 36 (48),
// 4096 x 14336 19.4 (24.4), 37888 x 3584 gated 42 (58), 128256 x 8192 301 (380).
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "row_sums.h"

namespace oamd {

namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
enum { kRowsStore = 0, kRowsPartial = 1, kRowsGlu = 2 };

}  // namespace

// A workgroup takes rows of W from f0 to f1 (GLU: of gate and up), its four waves a quarter each of the K slice; lane l of wave w holds the
// X values of its 8 columns in every 512 of the quarter. MT: rows of X, J: 512-column pieces of the quarter, RF: rows of W requested at a time.
template <int MT, int J, int RF, int EPI, bool NORM>
__global__ void __launch_bounds__(256) gemm_rows_kernel(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W, bf16_t* __restrict__ Y,
                                                        float* __restrict__ P, int M, int N, int K, int S, GluAct act, RowsNorm nm) {
  constexpr int HALVES = EPI == kRowsGlu ? 2 : 1;
  extern __shared__ float red[];   // [slot][MT][wave, its 16 lanes]
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int units = N / HALVES;
  const int f0 = (int)((int64_t)units * blockIdx.x / gridDim.x), nf = (int)((int64_t)units * (blockIdx.x + 1) / gridDim.x) - f0;
  const int n = nf * HALVES, kz = blockIdx.y, Kw = K / S / 4, k0 = kz * (K / S) + w * Kw;
  const bool tail = ((J - 1) * 64 + lane) * 8 < Kw;   // this lane has columns in the last piece
  auto col = [&](int j) { return k0 + (j < J - 1 || tail ? (j * 64 + lane) * 8 : 0); };
  struct Rows { u32x4 v[RF][J]; } even, odd;
  auto load = [&](Rows& r, int s0) {
#pragma unroll
    for (int i = 0; i < RF; ++i) {
      const int s = min(s0 + i, n - 1), f = f0 + s / HALVES;
      const int row = EPI == kRowsGlu ? (f >> 6) * 128 + (f & 63) + (s & 1) * 64 : f;
      const bf16_t* p = W + (int64_t)row * K;
#pragma unroll
      for (int j = 0; j < J; ++j) r.v[i][j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p + col(j)));
    }
  };
  auto clear = [&](u32x4& v) {   // where the last piece has no columns both operands are 0
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = tail ? v[e] : 0;
  };
  u32x4 x[MT][J];   // requested in front of the first rows: their loop waits for none of its own loads
  if constexpr (!NORM) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int j = 0; j < J; ++j) x[m][j] = *reinterpret_cast<const u32x4*>(X + (int64_t)min(m, M - 1) * K + col(j));
    load(even, 0);
    load(odd, RF);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < MT; ++m) clear(x[m][J - 1]);
  } else {
    // the steps and roundings of rmsnorm_kernel; only the order of the sum of squares is another
    __shared__ float squares[MT][16];
    u32x4 wn[J], res[MT][J];
    f32x4 slab[MT][J][2];
#pragma unroll
    for (int j = 0; j < J; ++j) wn[j] = *reinterpret_cast<const u32x4*>(nm.w + col(j));
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const int64_t at = (int64_t)min(m, M - 1) * K + col(j);
        if (nm.p) {
          slab[m][j][0] = *reinterpret_cast<const f32x4*>(nm.p + at);
          slab[m][j][1] = *reinterpret_cast<const f32x4*>(nm.p + at + 4);
        } else {
          x[m][j] = *reinterpret_cast<const u32x4*>(X + at);
        }
        if (nm.res) res[m][j] = *reinterpret_cast<const u32x4*>(nm.res + at);
      }
    load(even, 0);
    load(odd, RF);
    __builtin_amdgcn_sched_barrier(0);
    if (nm.p) {
      for (int s = 1; s < nm.S; ++s)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int j = 0; j < J; ++j) {
            const float* q = nm.p + ((int64_t)s * M + min(m, M - 1)) * K + col(j);
            slab[m][j][0] += *reinterpret_cast<const f32x4*>(q);
            slab[m][j][1] += *reinterpret_cast<const f32x4*>(q + 4);
          }
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) x[m][j][e] = pack_bf2(slab[m][j][e >> 1][2 * (e & 1)], slab[m][j][e >> 1][2 * (e & 1) + 1]);
    }
    auto lo = [](uint32_t v) { return __uint_as_float(v << 16); };
    auto hi = [](uint32_t v) { return __uint_as_float(v & 0xffff0000u); };
    float sq[MT] = {};
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma unroll
      for (int j = 0; j < J; ++j) {
        if (nm.res) {
#pragma unroll
          for (int e = 0; e < 4; ++e) x[m][j][e] = pack_bf2(lo(x[m][j][e]) + lo(res[m][j][e]), hi(x[m][j][e]) + hi(res[m][j][e]));
          if (blockIdx.x == 0 && m < M && (j < J - 1 || tail)) *reinterpret_cast<u32x4*>(nm.out + (int64_t)m * K + col(j)) = x[m][j];
        }
        if (j == J - 1) clear(x[m][j]);
#pragma unroll
        for (int e = 0; e < 4; ++e) sq[m] += lo(x[m][j][e]) * lo(x[m][j][e]) + hi(x[m][j][e]) * hi(x[m][j][e]);
      }
    }
    const float t = sums16<MT>(sq, lane);
    if ((lane & 15) >= 16 - MT) squares[lane & (MT - 1)][4 * w + (lane >> 4)] = t;
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      float tot = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(&squares[m][4 * i]);
        tot += (v[0] + v[1]) + (v[2] + v[3]);
      }
      const float rs = rsqrtf(tot / static_cast<float>(K) + nm.eps);
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          x[m][j][e] = pack_bf2(bf2f(f2bf(lo(x[m][j][e]) * rs)) * lo(wn[j][e]), bf2f(f2bf(hi(x[m][j][e]) * rs)) * hi(wn[j][e]));
      clear(x[m][J - 1]);
    }
  }
  auto mul = [&](Rows& r, int s0) {
    float t[RF];
#pragma unroll
    for (int i = 0; i < RF; ++i) {
      clear(r.v[i][J - 1]);
      float a[MT] = {};
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            a[m] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, (uint32_t)r.v[i][j][e]), __builtin_bit_cast(bf16x2, (uint32_t)x[m][j][e]), a[m], false);
      t[i] = sums16<MT>(a, lane);
    }
    load(r, s0 + 2 * RF);
    if ((lane & 15) >= 16 - MT)
#pragma unroll
      for (int i = 0; i < RF; ++i) red[((s0 + i) * MT + (lane & (MT - 1))) * 16 + 4 * w + (lane >> 4)] = t[i];
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
    for (int i = 0; i < 4; ++i) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(red + (slot * MT + m) * 16 + 4 * i);
      t += (v[0] + v[1]) + (v[2] + v[3]);
    }
    return t;
  };
  for (int e = threadIdx.x; e < nf * M; e += 256) {
    const int m = e / nf, f = e % nf;
    if constexpr (EPI == kRowsGlu) {
      const float g = bf2f(f2bf(sum(2 * f, m))), u = bf2f(f2bf(sum(2 * f + 1, m)));
      Y[(int64_t)m * units + f0 + f] = f2bf(bf2f(f2bf(glu_gate(g, act))) * u);
    } else if constexpr (EPI == kRowsPartial) {
      P[((int64_t)kz * M + m) * N + f0 + f] = sum(f, m);
    } else {
      Y[(int64_t)m * N + f0 + f] = f2bf(sum(f, m));
    }
  }
}

template <int MT, int J, bool NORM>
static int launch_rows(const bf16_t* X, const bf16_t* W, bf16_t* Y, float* P, int M, int N, int K, int S, int glu, int blocks, const RowsNorm& nm,
                       hipStream_t stream) {
  if constexpr (MT * J > (NORM ? 8 : 32) || (NORM && MT > 4)) {
    return -1;
  } else {
    constexpr int RF = J == 1 ? 8 : J == 2 ? 4 : J <= 4 ? 2 : 1;
    constexpr int GF = RF < 2 ? 2 : RF;
    const int units = glu ? N / 2 : N, most = (units + blocks - 1) / blocks * (glu ? 2 : 1) + GF;   // slots, and what the last rows run over
    const size_t lds = (size_t)most * MT * 64;
    if (lds > (48 << 10)) return -4;
    const dim3 grid(blocks, S);
    if (glu) gemm_rows_kernel<MT, J, GF, kRowsGlu, NORM><<<grid, 256, lds, stream>>>(X, W, Y, P, M, N, K, 1, glu_act(glu), nm);
    else if (S > 1 || Y == nullptr) gemm_rows_kernel<MT, J, RF, kRowsPartial, NORM><<<grid, 256, lds, stream>>>(X, W, Y, P, M, N, K, S, GluAct{}, nm);
    else gemm_rows_kernel<MT, J, RF, kRowsStore, NORM><<<grid, 256, lds, stream>>>(X, W, Y, P, M, N, K, 1, GluAct{}, nm);
    return 0;
  }
}

template <int MT, bool NORM>
static int rows_of(const bf16_t* X, const bf16_t* W, bf16_t* Y, float* P, int M, int N, int K, int S, int glu, int blocks, const RowsNorm& nm,
                   hipStream_t stream) {
  switch ((K / S / 4 + 511) / 512) {
    case 1: return launch_rows<MT, 1, NORM>(X, W, Y, P, M, N, K, S, glu, blocks, nm, stream);
    case 2: return launch_rows<MT, 2, NORM>(X, W, Y, P, M, N, K, S, glu, blocks, nm, stream);
    case 3: return launch_rows<MT, 3, NORM>(X, W, Y, P, M, N, K, S, glu, blocks, nm, stream);
    case 4: return launch_rows<MT, 4, NORM>(X, W, Y, P, M, N, K, S, glu, blocks, nm, stream);
    case 5: return launch_rows<MT, 5, NORM>(X, W, Y, P, M, N, K, S, glu, blocks, nm, stream);
    case 6: return launch_rows<MT, 6, NORM>(X, W, Y, P, M, N, K, S, glu, blocks, nm, stream);
    case 7: return launch_rows<MT, 7, NORM>(X, W, Y, P, M, N, K, S, glu, blocks, nm, stream);
    case 8: return launch_rows<MT, 8, NORM>(X, W, Y, P, M, N, K, S, glu, blocks, nm, stream);
    default: return -1;
  }
}

int gemm_rows(const bf16_t* X, const bf16_t* W, bf16_t* Y, float* P, int M, int N, int K, int S, int glu, int blocks, const RowsNorm* norm,
              hipStream_t stream) {
  if (M < 1 || M > 8 || S < 1 || S > 8 || K % (32 * S) || N < 1 || blocks < 1) return -1;
  if (glu && (S != 1 || N % 128)) return -2;
  if ((S > 1 || Y == nullptr) && P == nullptr) return -3;
  if (norm && S != 1) return -5;
  blocks = blocks < (glu ? N / 2 : N) ? blocks : (glu ? N / 2 : N);
  auto run = [&](auto mt) {
    constexpr int MT = decltype(mt)::value;
    return norm ? rows_of<MT, true>(X, W, Y, P, M, N, K, S, glu, blocks, *norm, stream)
                : rows_of<MT, false>(X, W, Y, P, M, N, K, S, glu, blocks, RowsNorm{}, stream);
  };
  const int rc = M == 1 ? run(std::integral_constant<int, 1>{}) : M == 2 ? run(std::integral_constant<int, 2>{})
                 : M <= 4 ? run(std::integral_constant<int, 4>{}) : run(std::integral_constant<int, 8>{});
  if (rc) return rc;
  OAMD_LAUNCH_CHECK();
  return 0;
}

}  // namespace oamd
