// Transposed W4A16 product for the PEFT backward: out = g @ W^T.
//
// g fp16 [M, N] (the output gradient), W the packed [K, N] int4 matrix,
// out fp16 [M, K] in the checkpoint's row order.  The reference computes it
// by dequantising W into an fp16 K x N buffer and running a dense GEMM
// (cuda_extends/exllama/q4_transpose_matmul.cu:115-167, exllama.py:528-544);
// here the packed words are read once and never expanded in memory.
//
// MFMA reduces over the elements a lane holds, and a packed word gives a lane
// 8 rows k of one column n; the reduction here runs over n.  Each dequantised
// word is therefore turned around by the matrix core itself: a
// v_mfma_f32_16x16x32_f16 with the word as its A operand (rows n, reduction
// k) and a one-hot B operand selecting 16 of the 32 k returns, in the D
// layout, 4 consecutive n of one k per lane -- exactly the B operand of a
// v_mfma_f32_16x16x16_f16 whose reduction runs over n.  The values pass
// through fp32 unchanged (one product with 1.0 each), so the weight that
// enters the product is the exact fp16 dequantised weight fp16(s * (q - z)),
// as dw4_dequant writes it.
//
// Grid: x = (K/128 chunk rows) x (NS N-ranges), z = 64-row blocks of M.  A
// workgroup of 4 waves owns one chunk row (128 outputs k) of one N-range;
// its waves take the range's 16-column strips round-robin and stream each
// strip's 1 KB chunk through a register ring.  The waves' fp32 partial tiles
// meet in LDS in a fixed order; with one N-range the tile is rounded and
// stored (scattered through perm for act-order), otherwise it goes to an
// fp32 plane of the workspace and a second kernel sums the planes in order.

#include <hip/hip_runtime.h>

#include <algorithm>

#include "w4a16_device.h"
#include "w4a16_transpose.h"

namespace dw4 {

namespace {

__device__ __forceinline__ f4 mfma16x16x16(h4 a, h4 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
}

// fp32 -> fp16 for values that are fp16 already (exact under any rounding)
__device__ __forceinline__ h4 to_h4(f4 v) {
  const h2 lo = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pkrtz(v[0], v[1]));
  const h2 hi = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pkrtz(v[2], v[3]));
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3);
}

// KBR: 16-row k-blocks reduced per LDS round (8 / KBR rounds, each with
// WAVES x KBR x MT x 1 KB of LDS).
template <int MT, int WAVES, int U, int GPC, bool ACT, int KBR>
__global__ void __launch_bounds__(WAVES * 64)
gemm_t_kernel(const _Float16* __restrict__ g, int64_t ldg, int M,
              const u4* __restrict__ pq, const uint32_t* __restrict__ pz,
              const uint32_t* __restrict__ ps32, const int32_t* __restrict__ perm,
              uint16_t* __restrict__ out, int64_t ldo, float* __restrict__ part,
              int K, int N, int gs, int G, int spr) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  constexpr int T = WAVES * 64;
  const int KC = K / kChunkK;
  const int NSTR = N / kStripN;
  const int c = blockIdx.x % KC;           // chunk row: outputs k in [128c, 128c + 128)
  const int ns = blockIdx.x / KC;          // N-range
  const int m0 = blockIdx.z * 64;          // first row of this M block
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15;
  const int kq = lane >> 4;
  const int s_lo = ns * spr;
  const int s_hi = min(NSTR, s_lo + spr);
  const int nstr = s_hi - s_lo;
  const int nch = wave < nstr ? (nstr - wave + WAVES - 1) / WAVES : 0;  // this wave's strips

  // one-hot selectors: B[kk][jj] = (kk == jj) and (kk == jj + 16), kk = 8 kq + e
  h8 sel0, sel1;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    sel0[e] = (8 * kq + e == j) ? (_Float16)1.0f : (_Float16)0.0f;
    sel1[e] = (8 * kq + e == j + 16) ? (_Float16)1.0f : (_Float16)0.0f;
  }
  // g rows of the A operand (lanes past the last row read row M-1, never stored)
  const _Float16* grow[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    grow[mt] = g + (size_t)min(m0 + mt * 16 + j, M - 1) * ldg + 4 * kq;

  // ring slot: 4 packed words, per-group scale/zero words, the g fragments
  u4 qb[U];
  uint32_t sb[U][GPC], zb[U][GPC];
  h4 gb[U][MT];
  auto load = [&](int slot, int i) {
    const int s = s_lo + wave + i * WAVES;
    qb[slot] = __builtin_nontemporal_load(pq + ((size_t)s * KC + c) * 64 + lane);
#pragma unroll
    for (int gl = 0; gl < GPC; ++gl) {
      const int grp = GPC == 1 ? (c * kChunkK) / gs : c * GPC + gl;
      sb[slot][gl] = ps32[((size_t)s * G + grp) * 8 + (j >> 1)];
      zb[slot][gl] = pz[((size_t)s * G + grp) * 2 + (j >> 3)];
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) gb[slot][mt] = *(const h4*)(grow[mt] + s * kStripN);
  };

  f4 acc[8][MT];
#pragma unroll
  for (int kb = 0; kb < 8; ++kb)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[kb][mt] = f4{0.f, 0.f, 0.f, 0.f};

  const uint32_t magic = opaque(kMagic);
  const int hsh = (j & 1) * 16;
  const int zsh = (j & 7) * 4;
  constexpr int WPG = 4 / GPC;  // packed words (32-row k-steps) per group
  auto consume = [&](int slot) {
    _Float16 sc = (_Float16)0.f;
    h2 nz1024, nz64;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (w % WPG == 0) {
        const int gl = w / WPG;
        sc = as_h((uint16_t)(sb[slot][gl] >> hsh));
        zero_consts(zb[slot][gl], zsh, nz1024, nz64);
      }
      // exact fp16 weight of rows 32w + 8kq + e, column j of the strip
      const h8 wv = centered8(qb[slot][w], nz1024, nz64, magic) *
                    h8{sc, sc, sc, sc, sc, sc, sc, sc};
      const f4 z = f4{0.f, 0.f, 0.f, 0.f};
      const h4 b0 = to_h4(__builtin_amdgcn_mfma_f32_16x16x32_f16(wv, sel0, z, 0, 0, 0));
      const h4 b1 = to_h4(__builtin_amdgcn_mfma_f32_16x16x32_f16(wv, sel1, z, 0, 0, 0));
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        acc[2 * w][mt] = mfma16x16x16(gb[slot][mt], b0, acc[2 * w][mt]);
        acc[2 * w + 1][mt] = mfma16x16x16(gb[slot][mt], b1, acc[2 * w + 1][mt]);
      }
    }
  };

  // ring: every wave with strips has at least one; refills only where one remains
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (u < nch) load(u, u);
  int i0 = 0;
  for (; i0 + 2 * U <= nch; i0 += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      consume(u);
      load(u, i0 + u + U);
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int i = i0 + u;
    if (i < nch) {
      consume(u);
      if (i + U < nch) load(u, i + U);
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (i0 + U + u < nch) consume(u);

  // Fixed-order reduction across waves, KBR 16-row k-blocks per round (LDS
  // holds WAVES x KBR x MT x 64 f4).
  f4* red = reinterpret_cast<f4*>(smem);
  const float* redf = reinterpret_cast<const float*>(smem);
  const bool direct = part == nullptr;
#pragma unroll
  for (int kb0 = 0; kb0 < 8; kb0 += KBR) {
    if (kb0 > 0) __syncthreads();  // the previous round's reads are done
#pragma unroll
    for (int b = 0; b < KBR; ++b)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) red[((wave * KBR + b) * MT + mt) * 64 + lane] = acc[kb0 + b][mt];
    __syncthreads();
    for (int idx = tid; idx < KBR * MT * 256; idx += T) {
      const int llo = idx & 15;
      const int r = (idx >> 4) & 3;
      const int lhi = (idx >> 6) & 3;
      const int bm = idx >> 8;  // b * MT + mt
      const int mt = bm % MT;
      const int b = bm / MT;
      const int m = m0 + mt * 16 + lhi * 4 + r;
      if (m >= M) continue;
      const int L = lhi * 16 + llo;
      float sum = 0.f;
#pragma unroll
      for (int wv = 0; wv < WAVES; ++wv) sum += redf[(((wv * KBR + b) * MT + mt) * 64 + L) * 4 + r];
      const int k = c * kChunkK + 16 * (kb0 + b) + llo;  // sorted row
      if (direct) {
        const int row = ACT ? perm[k] : k;
        out[(size_t)m * ldo + row] = h_bits((_Float16)sum);
      } else {
        part[((size_t)ns * M + m) * K + k] = sum;
      }
    }
  }
}

// The product above 64 rows: 16 MT rows by one chunk row (128 outputs k) of
// one N-range per workgroup of eight waves.  What bounds it is the L1's rate
// on the g fragments (16 rows, one cache line each, per load), so a lane takes
// 16 bytes of a row, eight consecutive n, where gemm_t_kernel takes 8: the
// reduction runs as 16x16x32 steps over the 32 columns of two strips.  For
// that the B operand needs n = 8 kq + e in lane group kq, and a turn returns
// n rows 4 kq + r; so the lanes load the packed words of permuted columns
// (half h of the pair: row j of the turn holds column 8 (j >> 2) + 4 h + (j & 3)),
// which costs nothing.  The integers q - z are turned and the scale multiplies
// after it, in the same fp16 rounding, so a weight that is not finite stays at
// its own k.  The waves split the range's strip pairs and share nothing until
// the end (no barrier in the loop); their tiles meet in LDS in wave order.
// 4096 x 11008: M = 128 37.5 -> 29.4 us (gemm_t_kernel before), M = 384 57.6 us
// (dequantise and a library product: 75.5); with 8-byte loads of g in strip
// order M = 384 took 75.8, with four waves of 96 rows 95.6.
template <int MT, int GPC>
__global__ void __launch_bounds__(512)
gemm_t_tall_kernel(const _Float16* __restrict__ g, int64_t ldg, int M,
                   const u4* __restrict__ pq, const uint32_t* __restrict__ pz,
                   const _Float16* __restrict__ ps, const int32_t* __restrict__ perm,
                   uint16_t* __restrict__ out, int64_t ldo, float* __restrict__ part,
                   int K, int N, int gs, int G, int spr) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  constexpr int WAVES = 8, QU = 2, U = 2, KBR = 4;
  const int KC = K / kChunkK;
  const int NSTR = N / kStripN;
  // XCD-aware order: workgroup b runs on XCD b % 8; each XCD takes a run of
  // consecutive tiles, chunk rows fastest, which share one slice of g in its L2.
  const int per = gridDim.x >> 3, rem = gridDim.x & 7;
  const int xcd = blockIdx.x & 7;
  const int tile = xcd * per + min(xcd, rem) + (int)(blockIdx.x >> 3);
  const int c = tile % KC;
  const int mblocks = (M + 16 * MT - 1) / (16 * MT);
  const int m0 = (tile / KC) % mblocks * (16 * MT);
  const int ns = tile / KC / mblocks;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15;
  const int kq = lane >> 4;
  const int s_lo = ns * spr;               // spr is even
  const int s_hi = min(NSTR, s_lo + spr);
  const int npair = (s_hi - s_lo) >> 1;
  const int nch = wave < npair ? (npair - wave + WAVES - 1) / WAVES : 0;  // this wave's pairs

  h8 sel0, sel1;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    sel0[e] = (8 * kq + e == j) ? (_Float16)1.0f : (_Float16)0.0f;
    sel1[e] = (8 * kq + e == j + 16) ? (_Float16)1.0f : (_Float16)0.0f;
  }
  // the block's rows: a uniform base and 32-bit lane offsets (ldg <= 2^24)
  const char* gblk = reinterpret_cast<const char*>(g + (size_t)m0 * ldg);
  uint32_t grow[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    grow[mt] = (uint32_t)min(mt * 16 + j, M - 1 - m0) * (uint32_t)(ldg * 2) + 16 * kq;

  u4 qb[QU][2];
  h8 sb[QU][GPC];
  uint32_t zb[QU][GPC];
  h8 gb[U][MT];
  // column of the pair (0..31) in half h at row j of the turn: 8 (j >> 2) + 4 h + (j & 3)
  const int col0 = 8 * ((j >> 2) & 1) + (j & 3);
  auto load_q = [&](int slot, int s0, int s1) {
    const int s = j < 8 ? s0 : s1;
    const u4* src = pq + ((size_t)s * KC + c) * 64 + kq * 16 + col0;
    qb[slot][0] = src[0];
    qb[slot][1] = src[4];
    const int ss = kq < 2 ? s0 : s1;
#pragma unroll
    for (int gl = 0; gl < GPC; ++gl) {
      const int grp = GPC == 1 ? (c * kChunkK) / gs : c * GPC + gl;
      sb[slot][gl] = *(const h8*)(ps + ((size_t)ss * G + grp) * 16 + 8 * (kq & 1));
      zb[slot][gl] = pz[((size_t)s * G + grp) * 2 + (col0 >> 3)];
    }
  };
  auto load_g = [&](int slot, int s0) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      gb[slot][mt] = *(const h8*)(gblk + (size_t)s0 * (2 * kStripN) + grow[mt]);
  };
  auto first = [&](int i) { return s_lo + 2 * (wave + min(i, nch - 1) * WAVES); };

  f4 acc[8][MT];
#pragma unroll
  for (int kb = 0; kb < 8; ++kb)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[kb][mt] = f4{0.f, 0.f, 0.f, 0.f};

  const uint32_t magic = opaque(kMagic);
  const int zsh = (j & 3) * 4;  // 4 h columns further on in half h
  constexpr int WPG = 4 / GPC;
  // the two B operands of packed word w: 16 k each, elements n = 8 kq + e
  auto turn = [&](int slot, int w, h8& b0, h8& b1) {
    f4 t[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      h2 nz1024, nz64;
      zero_consts(zb[slot][w / WPG], zsh + 16 * h, nz1024, nz64);
      const h8 wv = centered8(qb[slot][h][w], nz1024, nz64, magic);
      const f4 z = f4{0.f, 0.f, 0.f, 0.f};
      t[h][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv, sel0, z, 0, 0, 0);
      t[h][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv, sel1, z, 0, 0, 0);
    }
    const h8 sc = sb[slot][w / WPG];
    b0 = __builtin_shufflevector(to_h4(t[0][0]), to_h4(t[1][0]), 0, 1, 2, 3, 4, 5, 6, 7) * sc;
    b1 = __builtin_shufflevector(to_h4(t[0][1]), to_h4(t[1][1]), 0, 1, 2, 3, 4, 5, 6, 7) * sc;
  };
  // word w + 1 is turned while the products of word w run
  auto consume = [&](int slot, int gslot) {
    h8 b[2][2];
    turn(slot, 0, b[0][0], b[0][1]);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (w < 3) turn(slot, w + 1, b[(w + 1) & 1][0], b[(w + 1) & 1][1]);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const h8 a = gb[gslot][mt];
        acc[2 * w][mt] = mfma16(a, b[w & 1][0], acc[2 * w][mt]);
        acc[2 * w + 1][mt] = mfma16(a, b[w & 1][1], acc[2 * w + 1][mt]);
      }
    }
  };

  // ring: refills past the last pair read that pair again and go unused
  if (nch > 0) {
#pragma unroll
    for (int u = 0; u < QU; ++u) load_q(u, first(u), first(u) + 1);
#pragma unroll
    for (int u = 0; u < U; ++u) load_g(u, first(u));
    int i = 0;
    for (; i + QU <= nch; i += QU) {
#pragma unroll
      for (int u = 0; u < QU; ++u) {
        consume(u, u % U);
        load_q(u, first(i + u + QU), first(i + u + QU) + 1);
        load_g(u % U, first(i + u + U));
      }
    }
#pragma unroll
    for (int u = 0; u < QU - 1; ++u)
      if (i + u < nch) {
        consume(u, u % U);
        load_g(u % U, first(i + u + U));
      }
  }
  // The last strip of an odd number: one wave, with columns 16..31 of the
  // pair zero in scale and g (their g would lie past the row).
  if (((s_hi - s_lo) & 1) != 0 && wave == WAVES - 1) {
    const h8 zero8 = h8{};
    load_q(0, s_hi - 1, s_hi - 1);
#pragma unroll
    for (int gl = 0; gl < GPC; ++gl) sb[0][gl] = kq < 2 ? sb[0][gl] : zero8;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      gb[0][mt] = zero8;
      if (kq < 2) gb[0][mt] = *(const h8*)(gblk + (size_t)(s_hi - 1) * (2 * kStripN) + grow[mt]);
    }
    consume(0, 0);
  }

  // Fixed-order reduction across waves, as in gemm_t_kernel.
  f4* red = reinterpret_cast<f4*>(smem);
  const float* redf = reinterpret_cast<const float*>(smem);
#pragma unroll
  for (int kb0 = 0; kb0 < 8; kb0 += KBR) {
    if (kb0 > 0) __syncthreads();
#pragma unroll
    for (int b = 0; b < KBR; ++b)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        red[((wave * KBR + b) * MT + mt) * 64 + lane] = acc[kb0 + b][mt];
    __syncthreads();
    for (int idx = tid; idx < KBR * MT * 256; idx += WAVES * 64) {
      const int llo = idx & 15;
      const int r = (idx >> 4) & 3;
      const int lhi = (idx >> 6) & 3;
      const int b = (idx >> 8) % KBR;
      const int mt = (idx >> 8) / KBR;
      const int m = m0 + mt * 16 + lhi * 4 + r;
      if (m >= M) continue;
      const int L = lhi * 16 + llo;
      float sum = 0.f;
#pragma unroll
      for (int wv = 0; wv < WAVES; ++wv) sum += redf[(((wv * KBR + b) * MT + mt) * 64 + L) * 4 + r];
      const int k = c * kChunkK + 16 * (kb0 + b) + llo;  // sorted row
      if (part == nullptr)
        out[(size_t)m * ldo + (perm != nullptr ? perm[k] : k)] = h_bits((_Float16)sum);
      else
        part[((size_t)ns * M + m) * K + k] = sum;
    }
  }
}

// Sum of the N-range planes in order, rounded once, scattered through perm.
// Four outputs k of one row per thread (K is a multiple of 128).
__global__ void gemm_t_reduce_kernel(const f4* __restrict__ part, int ns, int M, int K,
                                     const int32_t* __restrict__ perm, uint16_t* __restrict__ out,
                                     int64_t ldo) {
  const size_t o = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t total = (size_t)M * (K / 4);
  if (o >= total) return;
  // all loads of a batch in flight before the first add; sums in plane order
  f4 sum = f4{0.f, 0.f, 0.f, 0.f};
  for (int i0 = 0; i0 < ns; i0 += 8) {
    f4 v[8];
#pragma unroll
    for (int b = 0; b < 8; ++b)
      v[b] = i0 + b < ns ? part[(size_t)(i0 + b) * total + o] : f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < 8; ++b)
      if (i0 + b < ns) sum += v[b];
  }
  const size_t m = o / (K / 4);
  const int k = (int)(o % (K / 4)) * 4;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int row = perm != nullptr ? perm[k + e] : k + e;
    out[m * ldo + row] = h_bits((_Float16)sum[e]);
  }
}

// Workgroup shape within 128 registers per lane for 16 waves (no spills in
// the build's register report): 16 waves up to 32 rows, a 4-deep ring for
// 16 rows; groups of 32 rows keep four scale/zero pairs per ring slot, so
// they take a 2-deep ring, and 8 waves at 32 rows.
template <int MT, int GPC> constexpr int t_waves() { return MT == 1 || (MT == 2 && GPC < 4) ? 16 : 8; }
template <int MT, int GPC> constexpr int t_ring() { return MT == 1 && GPC < 4 ? 4 : 2; }

// k-blocks per reduction round: as many as 128 KB of LDS holds
template <int MT, int GPC> constexpr int t_kbr() {
  return 128 / (t_waves<MT, GPC>() * MT) >= 8 ? 8 : 128 / (t_waves<MT, GPC>() * MT) >= 4 ? 4 : 2;
}

hipError_t launch_t_reduce(const GemmTArgs& a, const GemmTPlan& p, const float* part,
                           hipStream_t stream) {
  const size_t total = (size_t)a.M * (a.K / 4);
  gemm_t_reduce_kernel<<<(unsigned)((total + 255) / 256), 256, 0, stream>>>(
      (const f4*)part, p.ns, a.M, a.K, a.perm, a.out, a.ldo);
  return hipGetLastError();
}

template <int MT, int GPC>
hipError_t launch_tall_cfg(const GemmTArgs& a, const GemmTPlan& p, float* part, hipStream_t stream) {
  const int mblocks = (a.M + 16 * MT - 1) / (16 * MT);
  const size_t smem = (size_t)8 * 4 * MT * 64 * sizeof(f4);
  auto kern = &gemm_t_tall_kernel<MT, GPC>;
  static std::atomic<uint64_t> allowed{0};
  hipError_t e = allow_lds(reinterpret_cast<const void*>(kern), smem, allowed);
  if (e != hipSuccess) return e;
  kern<<<(unsigned)(a.K / kChunkK * mblocks * p.ns), 512, smem, stream>>>(
      (const _Float16*)a.g, a.ldg, a.M, (const u4*)a.pq, a.pz, (const _Float16*)a.ps, a.perm, a.out,
      a.ldo, p.ns > 1 ? part : nullptr, a.K, a.N, a.gs, a.G, p.spr);
  e = hipGetLastError();
  if (e != hipSuccess || p.ns == 1) return e;
  return launch_t_reduce(a, p, part, stream);
}

template <int MT>
hipError_t launch_tall(const GemmTArgs& a, const GemmTPlan& p, float* part, hipStream_t stream) {
  const int gpc = a.gs >= kChunkK ? 1 : kChunkK / a.gs;
  if (gpc == 1) return launch_tall_cfg<MT, 1>(a, p, part, stream);
  if (gpc == 2) return launch_tall_cfg<MT, 2>(a, p, part, stream);
  return launch_tall_cfg<MT, 4>(a, p, part, stream);
}

template <int MT, int GPC, bool ACT>
hipError_t launch_t_cfg(const GemmTArgs& a, const GemmTPlan& p, float* part, hipStream_t stream) {
  constexpr int WAVES = t_waves<MT, GPC>();
  constexpr int KBR = t_kbr<MT, GPC>();
  const int KC = a.K / kChunkK;
  const dim3 grid((unsigned)(KC * p.ns), 1, (unsigned)((a.M + 63) / 64));
  const size_t smem = (size_t)WAVES * KBR * MT * 64 * sizeof(f4);
  auto kern = &gemm_t_kernel<MT, WAVES, t_ring<MT, GPC>(), GPC, ACT, KBR>;
  if (smem > 64 * 1024) {
    static std::atomic<uint64_t> allowed{0};
    const hipError_t e = allow_lds(reinterpret_cast<const void*>(kern), smem, allowed);
    if (e != hipSuccess) return e;
  }
  kern<<<grid, WAVES * 64, smem, stream>>>(
      (const _Float16*)a.g, a.ldg, a.M, (const u4*)a.pq, a.pz, (const uint32_t*)a.ps, a.perm,
      a.out, a.ldo, p.ns > 1 ? part : nullptr, a.K, a.N, a.gs, a.G, p.spr);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || p.ns == 1) return e;
  return launch_t_reduce(a, p, part, stream);
}

template <int MT, int GPC>
hipError_t launch_t_act(const GemmTArgs& a, const GemmTPlan& p, float* part, hipStream_t stream) {
  return a.perm != nullptr ? launch_t_cfg<MT, GPC, true>(a, p, part, stream)
                           : launch_t_cfg<MT, GPC, false>(a, p, part, stream);
}

template <int MT>
hipError_t launch_t_mt(const GemmTArgs& a, const GemmTPlan& p, float* part, hipStream_t stream) {
  const int gpc = a.gs >= kChunkK ? 1 : kChunkK / a.gs;
  if (gpc == 1) return launch_t_act<MT, 1>(a, p, part, stream);
  if (gpc == 2) return launch_t_act<MT, 2>(a, p, part, stream);
  return launch_t_act<MT, 4>(a, p, part, stream);
}

// Rows above which the tall form runs.
constexpr int kTallRows = 64;
// Largest row stride whose 128-row block a 32-bit byte offset spans.
constexpr int64_t kTallMaxLdg = 1 << 24;

// The row tile (48 or 64 rows) and the number of N-ranges of the tall form:
// the least modelled time.  A round of workgroups (one per CU) takes
// 0.4 MT - 0.09 us per strip pair of a wave plus 4 us; a sum over N-ranges
// 3 us and 0.45 us per MB of planes (fitted to 4096 x 11008 at M = 128: 68.4,
// 41.9, 33.4, 29.4 us with one to four ranges of 64 rows; 4096^2: 27.6, 22.6,
// 20.3, 20.7).
GemmTPlan plan_tall(int m, int kc, int strips, int cus) {
  GemmTPlan best;
  best.us = 1e30;
  for (int mt = 3; mt <= 4; ++mt) {
    const int mb = (m + 16 * mt - 1) / (16 * mt);
    for (int want = 1; want <= 8; ++want) {
      GemmTPlan p;
      p.mt = mt;
      p.spr = ((strips + want - 1) / want + 1) / 2 * 2;
      p.ns = (strips + p.spr - 1) / p.spr;
      const int rounds = (kc * mb * p.ns + cus - 1) / cus;
      const int steps = (p.spr / 2 + 7) / 8;  // strip pairs of one wave
      const double tile_us = steps * (0.4 * mt - 0.09) + 4.;
      const double planes_mb = p.ns > 1 ? 1e-6 * p.ns * m * kc * kChunkK * 4 : 0.;
      p.us = rounds * tile_us + (p.ns > 1 ? 3. + 0.45 * planes_mb : 0.);
      if (p.us < best.us) best = p;
    }
  }
  return best;
}

}  // namespace

GemmTPlan plan_gemm_t(int m, int k, int n, int cus) {
  GemmTPlan p;
  const int kc = k / kChunkK;
  const int strips = n / kStripN;
  if (m > kTallRows) return plan_tall(m, kc, strips, cus);
  const int mt = std::min(4, (m + 15) / 16);
  const int waves = mt <= 2 ? 16 : 8;
  const int mb = (m + 63) / 64;
  // One workgroup per CU (its registers and 128 KB of LDS), all in one
  // round: a grid just above the CU count would run a second round for a
  // few workgroups.  At least one strip per wave; the fp32 partial planes
  // (ns * m * k * 4 bytes, written and read once) kept to about a quarter of
  // the packed weight bytes (k * n / 2).
  const int want = cus / (kc * mb);
  const int cap = std::max(1, n / (16 * std::max(1, m)));
  p.ns = std::max(1, std::min({want, cap, strips / waves}));
  p.spr = (strips + p.ns - 1) / p.ns;
  p.ns = (strips + p.spr - 1) / p.spr;
  return p;
}

// The route this replaces writes and reads the dense weight (8 us + 1.07 us
// per million weights, at least 20 for its two launches) and runs a library
// product (1.35e-3 us per row and million weights).  Groups under 128 rows cost
// the tall form a fifth more.  Measured (us, packed / dense with the weight
// just written / dense over weights out of cache, matrices and rows rotated in
// both): 4096 x 11008 M = 192 37 / 89 / 126, 256 45 / 67 / 86, 384 57 / 76 / 96, 512
// 73 / 87 / 110; 4096^2 M = 192 20 / 40 / 47, 384 26 / 34 / 39, 512 32 / 38 / 43; 11008 x
// 4096 M = 192 47 / 60 / 75, 320 61 / 67 / 83, 384 73 / 68 / 83; in groups of 64 M =
// 160 58 / 56 / 72, 320 68 / 66 / 84; 5120 x 13824 M = 256 77 / 145 / 193, 384 103 / 115 /
// 143, 512 142 / 143 / 164.  The line at 0.6 of the modelled dense time is a
// cautious one: it takes the packed words only where they are ahead by more
// than the model's error on every shape (up to 192 rows on 4096 x 11008, 128 on
// 4096^2), and leaves a band above it, to about 384 rows, where they are
// ahead by 1.1 to 2.
bool gemm_t_beats_dense(const GemmTPlan& p, int m, int k, int n, int gs) {
  if (p.mt == 0) return true;
  const double mw = 1e-6 * k * n;
  const double dense = std::max(20., 8. + 1.07 * mw) + 1.35e-3 * mw * m;
  return (gs < kChunkK ? 1.2 : 1.) * p.us <= 0.6 * dense;
}

size_t gemm_t_ws_bytes(const GemmTPlan& p, int m, int k) {
  return p.ns > 1 ? (size_t)p.ns * m * k * sizeof(float) : 0;
}

hipError_t launch_gemm_t(const GemmTArgs& a, const GemmTPlan& p, float* part,
                         hipStream_t stream) {
  if (p.ns > 1 && part == nullptr) return hipErrorInvalidValue;
  // rows too far apart for the tall form's offsets: the same plan, 64-row blocks
  switch (a.ldg <= kTallMaxLdg ? p.mt : 0) {
    case 0: break;
    case 3: return launch_tall<3>(a, p, part, stream);
    default: return launch_tall<4>(a, p, part, stream);
  }
  switch (std::min(4, (a.M + 15) / 16)) {
    case 1: return launch_t_mt<1>(a, p, part, stream);
    case 2: return launch_t_mt<2>(a, p, part, stream);
    case 3: return launch_t_mt<3>(a, p, part, stream);
    default: return launch_t_mt<4>(a, p, part, stream);
  }
}

}  // namespace dw4
