// Causal flash attention for prefill with any query/key size and any value size (each up to
// 256), packed variable-length sequences, GQA: the swapped-operand 32x32 MFMA structure of
// attn_prefill.hip with the head sizes as template parameters and the group size at run time.
//
// A work item is 128 query rows of one sequence; grid (items, key/value head x head chunk,
// sub-block). A head chunk is GC <= 4 of the G query heads that share a key/value head (GC
// divides G), a workgroup is 4 waves: wave w takes head w % GC and 32 query rows of row block
// w / GC (4 / GC row blocks), so one staged K / V tile feeds GC heads. Layers with different
// head counts share one work list.
// Per 64-key tile: S^T = K Q^T (query row on the lane, so the softmax is lane-local), then
// O^T += V^T P^T with P straight from the accumulator registers and V^T through the
// transposing LDS read. The rescale is deferred (a running maximum is kept until a tile
// raises it by more than 8 in log2 units).
// seq_pfx: keys of a shared prompt prefix (rows of pk / pv) come before a sequence's own.
// window: tiles that no row of the workgroup sees are never loaded.
// Two LDS buffers of a K and a V tile, filled by LDS-DMA while the tile before is used, one barrier a tile. What bounds it is a wave's
// chain through a tile (products, softmax, products), and of short prompts the longest row's tiles; one buffer filled from registers behind two
// barriers put loads, LDS writes and waits into that chain. us, before and now, of 8 sequences of 900 tokens: 32 heads of 192 / 128 208 -> 137 (480
// TFLOP/s), 32 / 8 of 128 115 -> 97, of 96 96 -> 80, of 64 / 256 260 -> 128, 16 of 64 37 -> 34; one of 300: 32 of 192 / 128 21 -> 13, 32 / 8 of 128 16 -> 13.
// Both buffers fit twice into a CU's 160 KB (192 / 128 exactly), as two workgroups did before, up to 320 columns of K and V together; larger ones have
// a CU alone (16 / 4 heads of 256: 233 -> 168). K's fragments requested four steps ahead and the halves' maximum without LDS:
// 16 / 4 heads of 256 168 -> 146, 8 / 2 of 160 79 -> 72, 32 / 8 of 128 97 -> 94, 16 of 64 34 -> 32; 192 / 128 as before.
#include "attn_gd.h"

namespace oamd {

using namespace gd;

namespace {

__device__ __forceinline__ s16x4 tr16(const char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p));
}

}  // namespace

// DK, DV: instantiated sizes >= the stored sizes dkp, dvp (the rest is zero in LDS)
template <int DK, int DV>
__global__ void __launch_bounds__(256, (DK + DV <= 320) ? 2 : 1) attn_gd_prefill_kernel(const AttnPrefill a) {
  constexpr int BK = 64, RK = 2 * DK;            // LDS row bytes of the tiles
  constexpr int RV = DV <= 32 ? 64 : DV <= 64 ? 128 : DV <= 128 ? 256 : 512;   // a power of two: the swizzle below
  constexpr int CK = RK / 16, CV = RV / 16;      // 16-B chunks of a row = KiB of a tile
  constexpr int NPK = CK / 4, NPV = CV / 4;      // KiB pieces a wave stages per tile
  constexpr int kKTile = BK * RK, kTile = kKTile + BK * RV;
  constexpr int KS = DK / 16, DB = DV / 32;
  __shared__ __attribute__((aligned(1024))) char lds[2 * kTile];

  int wi = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
  if (gridDim.y % 8 == 0) {   // a head's workgroups on one XCD, an item's sub-blocks next to each other
    const int L = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const int j = L >> 3;
    bz = j % gridDim.z;
    wi = j / gridDim.z % gridDim.x;
    by = j / gridDim.z / gridDim.x * 8 + (L & 7);
  }
  const int seq = a.work_seq[wi];
  if (seq < 0) return;   // padding item of a graph-captured prefill (fixed grid)
  const int GC = a.gc, nch = a.G / GC;
  const int kvh = by / nch, hc = by % nch;
  const int RG = 4 / GC, BQ = 32 * RG;
  const int s0 = a.cu_seqlens[seq];
  const int slen = a.cu_seqlens[seq + 1] - s0;
  const int q0 = a.work_q0[wi] + bz * BQ;
  if (q0 >= slen) return;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r32 = lane & 31, h = lane >> 5;
  const int hq = kvh * a.G + hc * GC + (w % GC);
  const int rbase = q0 + 32 * (w / GC);
  const int qrow = rbase + r32;
  const bool wave_used = w < GC * RG;
  const int Hq = a.Hkv * a.G;

  u16x8 qb[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s)
    qb[s] = (wave_used && qrow < slen && 16 * s + 8 * h < a.dkp)
                ? *reinterpret_cast<const u16x8*>(a.q + ((int64_t)(s0 + qrow) * Hq + hq) * a.dkp + 16 * s + 8 * h)
                : u16x8{0, 0, 0, 0, 0, 0, 0, 0};
  float scale = a.scale_log2;   // positive from here on, see attn_prefill.hip
  if (scale <= 0.f) {
#pragma unroll
    for (int s = 0; s < KS; ++s) qb[s] = scale < 0.f ? qb[s] ^ (uint16_t)0x8000 : u16x8{0, 0, 0, 0, 0, 0, 0, 0};
    scale = scale < 0.f ? -scale : 1.f;
  }
  f32x16 oacc[DB];
#pragma unroll
  for (int dd = 0; dd < DB; ++dd)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[dd][i] = 0.f;
  float mrow = -INFINITY, lpart = 0.f;

  const int kend = min(slen, q0 + BQ);
  const int pl = a.seq_pfx != nullptr ? a.seq_pfx[seq] : 0;
  const int npt = (pl + BK - 1) / BK;
  const int ntiles = npt + (kend + BK - 1) / BK;
  // first tile with a key that the first row sees (keys count from the prefix's start)
  const int lo = pl + q0 - a.window + 1;
  const int kt0 = lo <= 0 ? 0 : lo < pl ? lo / BK : npt + (lo - pl) / BK;
  const bool active = wave_used && rbase < slen;
  const int wend = min(slen, rbase + 32);   // own keys this wave can see: < wend

  const int gi = lane & 15, g = lane >> 4;
  const int trq = gi >> 2, trp = gi & 3;
  // Images: chunk ch of row r in a slot that depends on the row, as the LDS-DMA's source order. K: 16 rows' reads of one chunk hit 16
  // slots of the banks; a row of CK chunks shifts those by CK % 16, its swizzle covers the rest.
  constexpr int kP = CK % 16 == 0 ? 16 : CK % 8 == 0 ? 8 : 4;   // chunks that trade places
  auto k_swz = [](int r) { return (r / (16 / kP)) & (kP - 1); };
  // V: the transposed reads take 4 chunks of 4 neighbouring rows at a time.
  auto v_swz = [](int r) { return CV >= 16 ? ((r & 3) << 2) | ((r >> 2) & 3) : CV == 8 ? (r & 2) << 1 : 0; };
  auto v_img = [&](int r, int ch) { return RV * r + 16 * (ch ^ v_swz(r)); };

  // staging: slot 64 p + lane of piece p; chunks past the stored sizes and rows past the end read as zeros
  const int rbk = a.Hkv * a.dkp * 2, rbv = a.Hkv * a.dvp * 2;   // bytes from row to row
  uint32_t vk[NPK], vv[NPV];
#pragma unroll
  for (int i = 0; i < NPK; ++i) {
    const int at = 64 * (w + 4 * i) + lane, row = at / CK, ch = (at % CK) ^ k_swz(row);
    vk[i] = 8 * ch < a.dkp ? (uint32_t)(row * rbk + 16 * ch) : 0x7ffffff0u;
  }
#pragma unroll
  for (int i = 0; i < NPV; ++i) {
    const int at = 64 * (w + 4 * i) + lane, row = at / CV, ch = (at % CV) ^ v_swz(row);
    vv[i] = 8 * ch < a.dvp ? (uint32_t)(row * rbv + 16 * ch) : 0x7ffffff0u;
  }
  auto stage = [&](int kt, int buf) {   // key tile kt: a prefix tile (kt < npt) or own tile kt - npt
    const bf16_t *kp, *vp;
    int rows;
    if (kt < npt) {
      const int64_t r = (int64_t)kt * BK * a.Hkv + kvh;
      kp = a.pk + r * a.dkp; vp = a.pv + r * a.dvp; rows = pl - kt * BK;
    } else {
      const int64_t r = (int64_t)(s0 + (kt - npt) * BK) * a.Hkv + kvh;
      kp = a.k + r * a.dkp; vp = a.v + r * a.dvp; rows = slen - (kt - npt) * BK;
    }
    const int last = min(rows, BK) - 1, nk = last * rbk + 2 * a.dkp, nv = last * rbv + 2 * a.dvp;
    char* dst = lds + buf * kTile + w * 1024;
#pragma unroll
    for (int i = 0; i < NPK; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)kp, (short)0, nk, 0x00020000),
                                               (__attribute__((address_space(3))) void*)(dst + 4096 * i), 16, (int)vk[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < NPV; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)vp, (short)0, nv, 0x00020000),
                                               (__attribute__((address_space(3))) void*)(dst + kKTile + 4096 * i), 16, (int)vv[i], 0, 0, 0);
  };

  const int ks = h ^ k_swz(r32);
  stage(kt0, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (int kt = kt0, buf = 0; kt < ntiles; ++kt, buf ^= 1) {
    if (kt + 1 < ntiles) stage(kt + 1, buf ^ 1);
    const int kb = (kt - npt) * BK;   // own-key coordinates (negative: a prefix tile)
    const char *Ks = lds + buf * kTile, *Vs = Ks + kKTile;
    if (active && kb < wend) {   // wave-uniform: a key this wave sees
      f32x16 sacc[2];
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) sacc[b][i] = 0.f;
      constexpr int KA = KS < 4 ? KS : 4;
      u16x8 ka[KA][2];   // fragments of four 16-dim steps, requested that far ahead
      auto rdk = [&](int s) {
#pragma unroll
        for (int b = 0; b < 2; ++b) ka[s % KA][b] = *reinterpret_cast<const u16x8*>(Ks + RK * (32 * b + r32) + 16 * ((2 * s) ^ ks));
      };
#pragma unroll
      for (int s = 0; s < KA; ++s) rdk(s);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
#pragma unroll
        for (int b = 0; b < 2; ++b) sacc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bf8(ka[s % KA][b]), bf8(qb[s]), sacc[b], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (s + KA < KS) rdk(s + KA);
        __builtin_amdgcn_sched_barrier(0);
      }
      // register i of block b is key kb + 32b + (i&3) + 8(i>>2) + 4h
      const bool ptile = kb < 0;
      const int pend = pl - kt * BK;
      const int wlo = qrow - a.window - (ptile ? kt * BK - pl : kb);   // tile keys up to here are out of the row's window
      const bool mask = (ptile ? (pend < BK) : ((kb + BK > rbase + 1) || (kb + BK > slen))) ||
                        rbase + 31 - a.window >= (ptile ? kt * BK - pl : kb);
      if (mask) {   // the tile's first key past those the row sees, the last one before them
        const int end = (ptile ? pend : min(qrow + 1, slen) - kb) - 4 * h, out = wlo - 4 * h;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int j = 32 * b + (i & 3) + 8 * (i >> 2);
            if (j >= end || j <= out) sacc[b][i] = -INFINITY;
          }
      }
      float mx = sacc[0][0];
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, sacc[b][i]);
      mx = max_halves(mx) * scale;
      float mnew = fmaxf(mrow, mx);
      const bool rescale = mrow == -INFINITY || mnew > mrow + 8.f;
      if (!rescale) mnew = mrow;
      const float msafe = (mnew == -INFINITY) ? 0.f : mnew;
      const float alpha = rescale ? exp2_weight(mrow - msafe) : 1.f;
      mrow = mnew;
      float rs = 0.f;
      u16x8 pb[2][2];
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          f32x8 p;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            p[j] = exp2_weight(weight_arg(sacc[b][8 * s + j], scale, msafe));
            rs += p[j];
          }
          pb[b][s] = __builtin_bit_cast(u16x8, __builtin_convertvector(p, bf16x8));
        }
      lpart = lpart * alpha + rs;
      if (__any(rescale)) {
#pragma unroll
        for (int dd = 0; dd < DB; ++dd)
#pragma unroll
          for (int i = 0; i < 16; ++i) oacc[dd][i] *= alpha;
      }
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const int r0 = 32 * b + 16 * s + 4 * h + trq;
#pragma unroll
          for (int dd = 0; dd < DB; ++dd) {
            const int d = 32 * dd + 16 * (g & 1) + 4 * trp;
            const s16x4 lo = tr16(Vs + v_img(r0, d >> 3) + 8 * ((d >> 2) & 1));
            const s16x4 hi = tr16(Vs + v_img(r0 + 8, d >> 3) + 8 * ((d >> 2) & 1));
            const s16x8 va = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            oacc[dd] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, va), bf8(pb[b][s]), oacc[dd], 0, 0, 0);
          }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }
  if (!active) return;
  const float lsum = lpart + __shfl_xor(lpart, 32, kWave);
  if (qrow >= slen) return;
  float inv = lsum > 0.f ? 1.f / lsum : 0.f;
  if (a.gate) inv *= a.gate[(int64_t)(s0 + qrow) * Hq + hq];
  bf16_t* dst = a.o + (int64_t)(s0 + qrow) * a.o_ld + hq * a.dvp;
  // register i of block dd is dim 32 dd + (i&3) + 8(i>>2) + 4h
#pragma unroll
  for (int dd = 0; dd < DB; ++dd)
    if (32 * dd < a.dvp) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        u16x4 st;
#pragma unroll
        for (int e = 0; e < 4; ++e) st[e] = f2bf(oacc[dd][4 * c + e] * inv);
        *reinterpret_cast<u16x4*>(dst + 32 * dd + 8 * c + 4 * h) = st;
      }
    }
}

template <int DK>
static int launch_dv(const AttnPrefill& a, dim3 grid, hipStream_t stream) {
  switch (dim_bin(a.dvp)) {
    case 32: attn_gd_prefill_kernel<DK, 32><<<grid, 256, 0, stream>>>(a); break;
    case 64: attn_gd_prefill_kernel<DK, 64><<<grid, 256, 0, stream>>>(a); break;
    case 96: attn_gd_prefill_kernel<DK, 96><<<grid, 256, 0, stream>>>(a); break;
    case 128: attn_gd_prefill_kernel<DK, 128><<<grid, 256, 0, stream>>>(a); break;
    case 192:
    case 256: attn_gd_prefill_kernel<DK, 256><<<grid, 256, 0, stream>>>(a); break;
    default: return -2;
  }
  OAMD_LAUNCH_CHECK();
  return 0;
}

int attn_gd_prefill(const AttnPrefill& a, int num_work, hipStream_t stream) {
  if (num_work == 0) return 0;
  if (a.dkp % 8 || a.dvp % 32 || a.G < 1 || a.gc < 1 || a.gc > 4 || a.G % a.gc || a.window < 1) return -1;
  const int rg = 4 / a.gc, sub = 4 / rg;   // 32 rg rows per workgroup, 128 per work item
  const dim3 grid(num_work, a.Hkv * (a.G / a.gc), sub);
  switch (dim_bin(a.dkp)) {
    case 32: return launch_dv<32>(a, grid, stream);
    case 64: return launch_dv<64>(a, grid, stream);
    case 96: return launch_dv<96>(a, grid, stream);
    case 128: return launch_dv<128>(a, grid, stream);
    case 192: return launch_dv<192>(a, grid, stream);
    case 256: return launch_dv<256>(a, grid, stream);
    default: return -2;
  }
}

}  // namespace oamd
