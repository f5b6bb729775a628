// gfx950 W4A16 GEMM for mid-size M (a few dozen to a few hundred rows): the
// waves of a workgroup split K, not the tile.
//
// A workgroup of 8 waves owns a 32 MT x 32 P output tile; wave w takes the
// 128-row chunks w, w + 8, ... of the workgroup's K range and computes the
// whole tile over them.  Nothing is shared between the waves until the end, so
// there is no barrier in the loop: each wave streams its own activation
// fragments and packed words through registers, one chunk ahead, and the two
// waves of a SIMD drift apart, so that one dequantises while the other feeds
// the matrix cores.  (The LDS-streamed kernel of w4a16_prefill.hip shares a
// taller and wider tile, which reads less per flop, but its waves meet at a
// barrier every chunk and then dequantise and multiply in step.)
//   * activations are loaded as whole 128-byte lines (8 lanes per row, a half
//     chunk of 64 k) and turned into MFMA operand order through the wave's own
//     LDS region: 16-byte unit u of row r sits at u ^ (r & 7), so the stores
//     and the operand reads are conflict-free, and a wave reads only what it
//     wrote.  LDS operations of one wave complete in order, so no wait is
//     needed, but lanes read what other lanes stored: wavefront fences keep
//     the compiler from moving the reads over the stores or the next stores
//     over the reads (they emit no instruction);
//   * B operands as in the LDS-streamed kernel: two strips' packed words
//     rearranged by permlane swaps, the exact fp16 weight fp16(s (q - z)), and
//     v_mfma_f32_32x32x16_f16;
//   * the waves' fp32 partial tiles meet in LDS once, summed in wave order
//     (deterministic); one split writes the result, several write fp32 planes
//     that a second kernel sums in split order.
// What bounds it: the activations and words a CU reads from L2.  At 64 x 64 a
// round of eight chunks (160 KB per CU) takes 2.3 us with the loads alone (70
// GB/s per CU, 18 TB/s over the chip), 1.9 us with the arithmetic alone and 2.7
// us together.  So it wins where its small tiles fill the CUs once and the
// LDS-streamed kernel's larger ones do not (the plan's cost model): 4096^2
// M=256 21.1 -> 16.4 us, M=128 15.7 -> 11.5, 5120^2 M=96 19.9 -> 13.2, 13824 x
// 5120 M=96 35.7 -> 28.7, 4096 x 11008 M=64 19.1 -> 16.1 (before: the register-fed
// kernel up to 128 rows, the LDS-streamed one above).
// Every local array is indexed by constants only: one left to the stack is
// promoted to LDS by the compiler, whose address computation reads the
// dispatch packet in host memory (measured: +12 us on every launch).

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "w4a16_device.h"
#include "w4a16_prefill.h"

namespace dw4 {

namespace {

constexpr int kKsWaves = 8;

// Orders the wave's LDS accesses before and after it (for the compiler: the
// hardware keeps one wave's in order).
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

}  // namespace

template <int MT, int P, int GPC, bool BF>
__global__ void __launch_bounds__(kKsWaves * 64, 2)
kslice_kernel(const _Float16* __restrict__ x, int64_t ldx, int M, const P2Items it,
              float* __restrict__ part, int K, int N, uint32_t gmag, int G, int chunks_per_split,
              int mtiles, int ntiles, int splits, int group_m) {
  constexpr int W = kKsWaves;
  constexpr int BM = 32 * MT, BN = 32 * P;
  constexpr int AI = MT * 4;                  // activation loads per half chunk (8 rows each)
  constexpr int GH = GPC == 4 ? 2 : 1;        // groups per half chunk
  constexpr int kStage = BM * 128;            // bytes of a wave's activation region
  constexpr int kAcc4 = MT * P * 4;           // float4 accumulators per lane
  constexpr int kRed = W * kAcc4 * 64 * 16;   // bytes of the cross-wave sum
  constexpr int kLds = W * kStage > kRed ? W * kStage : kRed;
  __shared__ __attribute__((aligned(256))) unsigned char smem[kLds];
  __shared__ __attribute__((aligned(16))) uint16_t ytile[BM * BN];

  int mtile, unit;
  if (!tile_of(blockIdx.x, mtiles, ntiles * splits, group_m, mtile, unit)) return;
  const int split = unit / ntiles;
  const int item = (unit % ntiles) / it.ntiles_item;
  const int ntile = unit % ntiles - item * it.ntiles_item;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31;
  const int hb = lane >> 5;
  const int hi = (lane >> 4) & 1;  // which strip of a pair holds this lane's B column
  const int j = lane & 15;
  const int KC = K / kChunkK;
  const int c_begin = split * chunks_per_split;
  const int nc = min(KC, c_begin + chunks_per_split) - c_begin;
  const int nch = wave < nc ? (nc - wave + W - 1) / W : 0;  // this wave's chunks
  const int m0 = mtile * BM;
  const int NS = N / kStripN;
  const int strip0 = ntile * 2 * P;

  // ---- sources: a uniform base plus a 32-bit lane offset (bytes)
  const unsigned char* xbase = reinterpret_cast<const unsigned char*>(x + (size_t)m0 * ldx);
  uint32_t aoff[AI];
#pragma unroll
  for (int a = 0; a < AI; ++a)
    aoff[a] = (uint32_t)((min(m0 + 8 * a + (lane >> 3), M - 1) - m0) * (int)ldx + 8 * (lane & 7)) * 2;
  // resources at the tile's first strip; strips past the last (partial
  // column tile) read the first one again, their columns are not stored
  const __amdgpu_buffer_rsrc_t xr = rsrc_of(xbase);
  const __amdgpu_buffer_rsrc_t qr = rsrc_of(it.pq[item] + (size_t)strip0 * KC * 64);
  const __amdgpu_buffer_rsrc_t sr = rsrc_of(it.ps[item] + (size_t)strip0 * G * 8);
  const __amdgpu_buffer_rsrc_t zr = rsrc_of(it.pz[item] + (size_t)strip0 * G * 2);
  int st[2 * P];
#pragma unroll
  for (int s = 0; s < 2 * P; ++s) st[s] = strip0 + s < NS ? s : 0;
  uint32_t soff[P], zoff[P];  // this lane's scale / zero word of each pair, group 0
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int s = strip0 + 2 * p + hi < NS ? 2 * p + hi : 0;
    soff[p] = ((uint32_t)s * G * 8 + (j >> 1)) * 4;
    zoff[p] = ((uint32_t)s * G * 2 + (j >> 3)) * 4;
  }

  // ---- ring: slot h holds half h (64 k) of one chunk
  h8 ab[2][AI];
  uint2 qb[2][2 * P];
  uint32_t sb[2][P][GH], zb[2][P][GH];
  const int c0 = c_begin + wave;
  auto load_a = [&](int h, int i) {
    const int so = ((c0 + i * W) * kChunkK + 64 * h) * 2;
#pragma unroll
    for (int a = 0; a < AI; ++a)
      ab[h][a] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(xr, aoff[a], so, 0));
  };
  auto load_b = [&](int h, int i) {
    const int c = c0 + i * W;
#pragma unroll
    for (int s = 0; s < 2 * P; ++s)
      qb[h][s] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(
                                               qr, lane * 16, (st[s] * KC + c) * 1024 + 8 * h, 0));
#pragma unroll
    for (int gl = 0; gl < GH; ++gl) {
      const int g = GPC == 1 ? div_by_magic(c, gmag) : c * GPC + (GPC == 4 ? 2 * h + gl : h);
#pragma unroll
      for (int p = 0; p < P; ++p) {
        sb[h][p][gl] = __builtin_amdgcn_raw_buffer_load_b32(sr, soff[p], g * 32, 0);
        zb[h][p][gl] = __builtin_amdgcn_raw_buffer_load_b32(zr, zoff[p], g * 8, 0);
      }
    }
  };

  f16v acc[MT][P];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[mt][p][e] = 0.f;

  unsigned char* xs = smem + wave * kStage;
  unsigned char* xw = xs + (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 3)) * 16);
  uint32_t roff[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) roff[t] = (uint32_t)(l32 * 128 + (((2 * t + hb) ^ (l32 & 7)) * 16));
  const uint32_t magic = opaque(kMagic);
  const int hsh = (j & 1) * 16;
  const int zsh = (j & 7) * 4;

  auto stage_a = [&](int h) {
#pragma unroll
    for (int a = 0; a < AI; ++a) *(h8*)(xw + a * 1024) = ab[h][a];
  };
  auto compute = [&](int h) {
    ColGroup col[P][GH];
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int gl = 0; gl < GH; ++gl) col[p][gl].set(sb[h][p][gl], hsh, zb[h][p][gl], zsh);
    uint32_t ev[P], od[P];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int gl = GPC == 4 ? t >> 1 : 0;
      h8 af[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) af[mt] = *(const h8*)(xs + roff[t] + mt * 4096);
#pragma unroll
      for (int p = 0; p < P; ++p) {
        if ((t & 1) == 0)
          strip_pair_to_b32(t ? qb[h][2 * p].y : qb[h][2 * p].x,
                            t ? qb[h][2 * p + 1].y : qb[h][2 * p + 1].x, ev[p], od[p]);
        const h8 bop = weight8<BF>((t & 1) ? od[p] : ev[p], col[p][gl], magic);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt][p] = mfma32_of<BF>(af[mt], bop, acc[mt][p]);
      }
    }
  };

  if (nch > 0) {
    // in the loop's order, so that its waits count the same loads on entry
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      load_a(h, 0);
      __builtin_amdgcn_sched_barrier(0);
      load_b(h, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    for (int i = 0; i < nch; ++i) {
      const int nx = min(i + 1, nch - 1);  // past the end: the last chunk again, unused
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        // (the compiler would sink the loads towards their uses)
        stage_a(h);
        wave_fence();
        load_a(h, nx);
        __builtin_amdgcn_sched_barrier(0);
        compute(h);
        wave_fence();
        __builtin_amdgcn_sched_barrier(0);
        load_b(h, nx);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  // ---- cross-wave sum, in wave order
  __syncthreads();  // every wave is past its activation region
  f4* red = reinterpret_cast<f4*>(smem);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        red[(wave * kAcc4 + (mt * P + p) * 4 + q) * 64 + lane] =
            f4{acc[mt][p][4 * q], acc[mt][p][4 * q + 1], acc[mt][p][4 * q + 2], acc[mt][p][4 * q + 3]};
  __syncthreads();
  const uint16_t* __restrict__ bias = it.bias[item];
  uint16_t* __restrict__ y = it.y[item];
  const int64_t ldy = it.ldy[item];
  const uint16_t* __restrict__ res = it.res[item];
  const int64_t ldres = it.ldres[item];
#pragma unroll
  for (int o = tid; o < kAcc4 * 64; o += W * 64) {
    const int slot = o >> 6;  // (mt * P + p) * 4 + q, wave-uniform
    f4 s = red[o];
#pragma unroll
    for (int w = 1; w < W; ++w) s += red[w * kAcc4 * 64 + o];
    const int q = slot & 3, p = (slot >> 2) % P, mt = slot / (4 * P);
    const int row = mt * 32 + 8 * q + 4 * hb;
    const int col = p * 32 + l32;
    const int n = strip0 * kStripN + col;
    if (splits > 1) {
      if (n < N) {
        float* plane = part + (size_t)split * M * N;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (m0 + row + e < M) plane[(size_t)(m0 + row + e) * N + n] = s[e];
      }
    } else {
      const uint16_t bv = bias != nullptr && n < N ? bias[n] : (uint16_t)0;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        ytile[(row + e) * BN + col] = round_out<BF>(s[e], bias != nullptr, bv);
    }
  }
  if (splits > 1) return;
  __syncthreads();
  const bool vec_y = ((reinterpret_cast<uintptr_t>(y) & 15) == 0) && (ldy % 8 == 0) &&
                     (res == nullptr ||
                      (((reinterpret_cast<uintptr_t>(res) & 15) == 0) && (ldres % 8 == 0)));
  for (int o = tid; o < BM * BN / 8; o += W * 64) {
    const int row = o / (BN / 8), seg = o % (BN / 8);
    const int m = m0 + row, n = strip0 * kStripN + seg * 8;
    if (m >= M || n >= N) continue;
    u4 v = *(const u4*)&ytile[row * BN + seg * 8];
    uint16_t* dst = y + (size_t)m * ldy + n;
    const uint16_t* rsrc = res != nullptr ? res + (size_t)m * ldres + n : nullptr;
    if (vec_y) {
      if (rsrc != nullptr) v = add_h8(v, *(const u4*)rsrc);
      *(u4*)dst = v;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        _Float16 h = as_h((uint16_t)(v[e / 2] >> (16 * (e & 1))));
        if (rsrc != nullptr) h = h + as_h(rsrc[e]);
        dst[e] = h_bits(h);
      }
    }
  }
}

template <int MT, int P, int GPC, bool BF>
static hipError_t launch_kslice_cfg(const GroupArgs& g, int splits, void* ws, hipStream_t stream) {
  const GemmArgs& a = g.a[0];
  P2Items it = prefill_items(g, 32 * P);
  const int mtiles = (a.M + 32 * MT - 1) / (32 * MT);
  const int ntiles = it.ntiles_item * g.count;
  const int KC = a.K / kChunkK;
  const int cps = (KC + splits - 1) / splits;
  const int real_splits = (KC + cps - 1) / cps;
  if (real_splits > 1 && g.count != 1) return hipErrorInvalidValue;  // planes of one matrix
  float* part = real_splits > 1
                    ? reinterpret_cast<float*>(static_cast<unsigned char*>(ws) + kWsHeadBytes)
                    : nullptr;
  const int units = ntiles * real_splits;
  const dim3 grid((unsigned)((units * mtiles + 7) / 8 * 8));
  kslice_kernel<MT, P, GPC, BF><<<grid, kKsWaves * 64, 0, stream>>>(
      (const _Float16*)a.x, a.ldx, a.M, it, part, a.K, a.N, group_magic(a.gs), a.G, cps, mtiles,
      ntiles, real_splits, prefill_group_m(mtiles));
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || real_splits == 1) return e;
  return launch_reduce_planes(part, real_splits, a.M, a.N, a.bias, a.y, a.ldy, a.res, a.ldres,
                              stream, BF);
}

template <int MT, int P, bool BF>
static hipError_t launch_kslice_gpc(const GroupArgs& g, int splits, void* ws, hipStream_t stream) {
  const int gpc = g.a[0].gs >= kChunkK ? 1 : kChunkK / g.a[0].gs;
  if (gpc == 1) return launch_kslice_cfg<MT, P, 1, BF>(g, splits, ws, stream);
  if (gpc == 2) return launch_kslice_cfg<MT, P, 2, BF>(g, splits, ws, stream);
  return launch_kslice_cfg<MT, P, 4, BF>(g, splits, ws, stream);
}

template <int MT, int P>
static hipError_t launch_kslice_tile(const GroupArgs& g, const PrefillPlan& p, void* ws,
                                     hipStream_t stream) {
  if (p.bf16) return launch_kslice_gpc<MT, P, true>(g, p.splits, ws, stream);
  return launch_kslice_gpc<MT, P, false>(g, p.splits, ws, stream);
}

hipError_t launch_kslice_group(const GroupArgs& g, const PrefillPlan& plan, void* ws,
                               hipStream_t stream) {
  if (!same_x_shape(g) || !prefill_x_fits(g.a[0].ldx)) return hipErrorInvalidValue;
  if (plan.bf16 && g.a[0].res != nullptr) return hipErrorInvalidValue;
  if (plan.bm == 64 && plan.bn == 64) return launch_kslice_tile<2, 2>(g, plan, ws, stream);
  if (plan.bm == 64 && plan.bn == 32) return launch_kslice_tile<2, 1>(g, plan, ws, stream);
  if (plan.bm == 32 && plan.bn == 64) return launch_kslice_tile<1, 2>(g, plan, ws, stream);
  return hipErrorInvalidValue;
}

}  // namespace dw4
