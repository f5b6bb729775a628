// Paged-attention decode and the KV-cache slot operations of the decoder
// stage.
//
// Cache layout (the reference's, operators/core/block/common.py:7-60 and
// cuda_extends/vllm/cache_kernels.cu:242-285, in
// /root/reference/After-Revision-DROFELL): the cache is a set of blocks of
// BS token slots; each block has a key part [kv_heads][head_size/8][BS][8]
// and a value part [kv_heads][head_size][BS] (fp16), reached through
// per-block pointer tables, with kv_head_stride elements between the heads
// of a block.  A token's slot s lives in block s / BS at offset s % BS.
//
// paged_attention_kernel: one workgroup per (sequence, kv head, context
// partition).  It serves every query head of the kv head's group
// (head h uses kv head h / (heads / kv_heads)), so each K and V byte is
// read once per group.  Per partition of up to 4096 tokens:
//   logits = scale * q . k (+ alibi slope * (t - ctx + 1));
//   p = exp(logit - max); out = sum p v / sum p.
// HBM-bound (the KV stream), so with grouped heads both products run on the
// matrix cores, whose
// operand layouts the cache's already are: the rows of a 16x16x32 MFMA are 16
// tokens (q . k) or 16 dims (p . v), each lane's 8 reduction elements one
// 16-byte unit of the cache, loaded straight into the operand registers; the
// columns are the group's heads (2 to 8 of 16).  A wave takes steps of 32
// tokens and keeps a running max, sum and output per head (all of head c in
// the lanes of column c), so no logits go through LDS; with row r of q . k's
// two token tiles holding tokens 8 (r / 4) + r % 4 and 4 more, a lane's eight
// logits are those of 8 consecutive tokens, the very p . v operand.
// Measured (us, with the products on the vector ALU, one LDS read of a logit
// per p . v FMA, before): 24 x 3000 tokens, 32 heads on 8 of 128 85 -> 46 (4.8
// TB/s), 32 x 4000, 64 on 8 283 -> 81, 8 x 600, 32 heads 20.5 -> 15.7, 8 x 3000, 16
// heads of 256 123 -> 54.
// Precision: q . k sums exact fp16 products in fp32; the softmax and its sums
// stay in fp32, and p enters p . v as three fp16 parts of 2^15 p, cut one after
// the other, which hold all 24 bits of it (below 2^-16, to 2^-37 of the largest
// p): the numerator is summed from the same p as the denominator.  Two parts
// held 21 bits, all cut downwards; the third costs 0.5 % (24 x 3000 tokens, 32 heads
// on 8: 50.6 -> 51.0 us) to 2 % (1 x 4000).
// Waves take the partition's steps round-robin and meet once in LDS.
// Partitions write their max, sum and unnormalised fp32 output; a second
// kernel combines them in partition order (deterministic).  With a single
// partition the first kernel writes the output directly.  One query head per
// kv head goes to paged_attention_row_kernel, in partitions of up to 512 tokens.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>

#include "w4a16_device.h"
#include "w4a16_attention.h"

namespace dw4 {

namespace {


constexpr float kLog2e = 1.4426950408889634f;
constexpr float kPScale = 32768.f;  // p enters p . v as fp16 parts of 2^15 p

__device__ __forceinline__ float exp_of(float v) { return __builtin_amdgcn_exp2f(v * kLog2e); }

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
  return v;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// Block-wide reduction in a fixed order (waves' results combined 0..W-1).
template <bool MAX, int W>
__device__ __forceinline__ float block_reduce(float v, float* scratch) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  v = MAX ? wave_max(v) : wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float r = scratch[0];
#pragma unroll
  for (int w = 1; w < W; ++w) r = MAX ? fmaxf(r, scratch[w]) : r + scratch[w];
  return r;
}

// The form for one query head per kv head, on the vector ALU: the matrix
// form's 16 columns would hold one head.  For q . k a lane holds one token and
// a slice of 8 dims (one 16-byte load), lanes of one token meet through
// cross-lane adds, the logits stand in LDS; for p . v a lane holds whole dims (a
// row of BS tokens).  Measured: four layers of 8 x 600 tokens, 32 heads of 128,
// 283 -> 270 us when this form took one head at compile time instead of a
// group's; the matrix form 269.  As that gains nothing, this one's order of sums
// stays: a stack of layers turns single roundings of one layer into
// differences of whole percents in a later one (an RMS norm over a row whose
// residuals cancel).
// W waves per workgroup: 4 (several partitions per (sequence, head), about four
// workgroups per CU) or 16 (one workgroup per (sequence, head) covering the
// whole context, no combine launch).
template <int HS, int BS, int W>
__global__ void __launch_bounds__(W * 64)
paged_attention_row_kernel(const uint16_t* __restrict__ query, int64_t q_stride,
                           uint16_t* __restrict__ out, int64_t o_stride,
                           const int64_t* __restrict__ kptr, const int64_t* __restrict__ vptr,
                           int kv_head_stride, int num_heads, float scale,
                           const int32_t* __restrict__ block_tables, int max_blocks,
                           const int32_t* __restrict__ context_lens,
                           const float* __restrict__ alibi, int part_tokens, int num_parts,
                           float* __restrict__ ws_ml, float* __restrict__ ws_out) {
  constexpr int SLICES = HS / 8;                 // 16-byte slices of a key row
  constexpr int TPL = 64 / BS;                   // slice groups per wave (lanes of one token)
  constexpr int SPL = (SLICES + TPL - 1) / TPL;  // slices per lane (the last may be past HS)
  constexpr int DPL = (HS + 63) / 64;            // value dims per lane (the last may be past HS)
  // head sizes that are not multiples of 64 (80, 96, 112) leave some lanes
  // without a last key slice or value dim: those hold zeros and store nothing
  constexpr bool KTAIL = SLICES % TPL != 0, VTAIL = HS % 64 != 0;
  static_assert(HS % 8 == 0 && 64 % BS == 0, "shape");
  extern __shared__ __attribute__((aligned(16))) float sm[];
  float* qs = sm;                               // [HS] fp32 query (scaled)
  float* logit = qs + HS;                   // [part_tokens]
  float* red = logit + part_tokens;         // [waves][HS] partial outputs
  float* scratch = red + W * HS;            // W floats

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int seq = blockIdx.x / num_heads;
  const int head = blockIdx.x % num_heads;
  const int part = blockIdx.y;
  // a context longer than the block table is cut to it (never read past a row)
  const int ctx = min(context_lens[seq], max_blocks * BS);
  const int t0 = part * part_tokens;
  const int t1 = min(ctx, t0 + part_tokens);
  const int nt = t1 - t0;
  const bool direct = num_parts == 1;
  if (nt <= 0) {  // partition past this sequence's context: an empty partial
    if (!direct && tid == 0) {
      const size_t r = ((size_t)seq * num_heads + head) * num_parts + part;
      ws_ml[2 * r] = -FLT_MAX;
      ws_ml[2 * r + 1] = 0.f;
    }
    return;
  }
  const int32_t* btab = block_tables + (size_t)seq * max_blocks + t0 / BS;
  const int nb = (nt + BS - 1) / BS;
  const int nbw = wave < nb ? (nb - wave + W - 1) / W : 0;  // this wave's blocks
  const int tt = lane % BS;   // token of this lane within a block
  const int sg = lane / BS;   // slice group
  // Each wave keeps its next NPF blocks' keys and values in flight: the
  // value loads of the first blocks are issued with the key loads, before
  // the softmax, so their latency overlaps q . k.
  constexpr int NPF = 2;
  h8 kreg[NPF][SPL];
  h8 vreg[NPF][DPL][BS / 8];
  auto kbase = [&](int i) {
    return reinterpret_cast<const uint16_t*>(kptr[btab[wave + W * i]]) +
           (size_t)head * kv_head_stride;
  };
  auto vbase = [&](int i) {
    return reinterpret_cast<const uint16_t*>(vptr[btab[wave + W * i]]) +
           (size_t)head * kv_head_stride;
  };
  auto load_k = [&](int slot, int i) {
    const uint16_t* kb = kbase(i);
#pragma unroll
    for (int j = 0; j < SPL; ++j) {
      if (KTAIL && sg + TPL * j >= SLICES) {
        kreg[slot][j] = h8{};
        continue;
      }
      kreg[slot][j] = *(const h8*)(kb + ((sg + TPL * j) * BS + tt) * 8);
    }
  };
  auto load_v = [&](int slot, int i) {
    const uint16_t* vb = vbase(i);
#pragma unroll
    for (int j = 0; j < DPL; ++j)
#pragma unroll
      for (int u = 0; u < BS / 8; ++u)
        vreg[slot][j][u] = VTAIL && lane + 64 * j >= HS
                                   ? h8{}
                                   : *(const h8*)(vb + (size_t)(lane + 64 * j) * BS + 8 * u);
  };
#pragma unroll
  for (int u = 0; u < NPF; ++u)
    if (u < nbw) {
      load_k(u, u);
      load_v(u, u);
    }
  // The query is staged after the first blocks' key and value loads went
  // out (each behind its block-table and block-pointer loads), so its own
  // load overlaps theirs; the barrier that publishes it waits only for the
  // LDS stores, and the key/value loads stay in flight across it (a
  // __syncthreads would wait for them).
  for (int d = tid; d < HS; d += (W * 64))
    qs[d] = scale * (float)as_h(query[(size_t)seq * q_stride + (size_t)head * HS + d]);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

  // q . k
  auto qk = [&](int slot, int i) {
    const int b = wave + W * i;
    float dot = 0.f;
#pragma unroll
    for (int j = 0; j < SPL; ++j) {
      if (KTAIL && sg + TPL * j >= SLICES) continue;
      const float* qv = qs + (sg + TPL * j) * 8;
#pragma unroll
      for (int e = 0; e < 8; ++e) dot = fmaf(qv[e], (float)kreg[slot][j][e], dot);
    }
#pragma unroll
    for (int off = BS; off < 64; off <<= 1) dot += __shfl_xor(dot, off);
    const int t = t0 + b * BS + tt;
    if (sg == 0) {
      if (alibi != nullptr) dot += alibi[head] * (float)(t - ctx + 1);
      logit[b * BS + tt] = t < t1 ? dot : -FLT_MAX;
    }
  };
  for (int i0 = 0; i0 < nbw; i0 += NPF) {
#pragma unroll
    for (int u = 0; u < NPF; ++u) {
      const int i = i0 + u;
      if (i < nbw) {
        qk(u, i);
        if (i + NPF < nbw) load_k(u, i + NPF);
      }
    }
  }
  __syncthreads();

  // softmax numerators and their sum
  float mx = -FLT_MAX, sum = 0.f;
  for (int t = tid; t < nt; t += (W * 64)) mx = fmaxf(mx, logit[t]);
  mx = block_reduce<true, W>(mx, scratch);
  for (int t = tid; t < nb * BS; t += (W * 64)) {
    const float p = t < nt ? __expf(logit[t] - mx) : 0.f;
    logit[t] = p;
    sum += p;
  }
  sum = block_reduce<false, W>(sum, scratch);
  __syncthreads();

  // p . v: lane holds dims lane + 64 j
  float acc[DPL];
#pragma unroll
  for (int j = 0; j < DPL; ++j) acc[j] = 0.f;
  auto pv = [&](int slot, int i) {
    const int b = wave + W * i;
    const int valid = min(BS, nt - b * BS);  // tokens of this block in the context
#pragma unroll
    for (int j = 0; j < DPL; ++j)
#pragma unroll
      for (int u = 0; u < BS / 8; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int tb = 8 * u + e;
          // slots past the context may hold anything: never multiply them
          const float vf = tb < valid ? (float)vreg[slot][j][u][e] : 0.f;
          acc[j] = fmaf(logit[b * BS + tb], vf, acc[j]);
        }
  };
  for (int i0 = 0; i0 < nbw; i0 += NPF) {
#pragma unroll
    for (int u = 0; u < NPF; ++u) {
      const int i = i0 + u;
      if (i < nbw) {
        pv(u, i);
        if (i + NPF < nbw) load_v(u, i + NPF);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < DPL; ++j)
    if (!VTAIL || lane + 64 * j < HS) red[wave * HS + lane + 64 * j] = acc[j];
  __syncthreads();
  for (int d = tid; d < HS; d += (W * 64)) {
    float o = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) o += red[w * HS + d];
    if (direct) {
      out[(size_t)seq * o_stride + (size_t)head * HS + d] = h_bits((_Float16)(o / sum));
    } else {
      const size_t r = ((size_t)seq * num_heads + head) * num_parts + part;
      ws_out[r * HS + d] = o;
      if (d == 0) {
        ws_ml[2 * r] = mx;
        ws_ml[2 * r + 1] = sum;
      }
    }
  }
}

// W waves per workgroup: 4 (several partitions per (sequence, kv head)) or 8
// (one workgroup per (sequence, kv head) covering the whole context, no
// combine launch).
template <int HS, int BS, int W>
__global__ void __launch_bounds__(W * 64, HS <= 128 ? 2 : 1)  // 256 registers per lane, or 512
paged_attention_kernel(const uint16_t* __restrict__ query, int64_t q_stride,
                       uint16_t* __restrict__ out, int64_t o_stride,
                       const int64_t* __restrict__ kptr, const int64_t* __restrict__ vptr,
                       int kv_head_stride, int num_heads, int num_kv_heads, float scale,
                       const int32_t* __restrict__ block_tables, int max_blocks,
                       const int32_t* __restrict__ context_lens,
                       const float* __restrict__ alibi, int part_tokens, int num_parts,
                       float* __restrict__ ws_ml, float* __restrict__ ws_out) {
  constexpr int SLICES = HS / 8;        // 16-byte units of a key row
  constexpr int NK = (HS + 31) / 32;    // 32-dim reduction steps of q . k (the last may be partial)
  constexpr int ND = HS / 16;           // 16-dim tiles of p . v
  constexpr int NB = 32 / BS;           // blocks of a 32-token step
  constexpr int SLOTS = HS <= 128 ? 2 : 1;  // steps in flight per wave (registers)
  static_assert(HS % 16 == 0 && 32 % BS == 0, "shape");
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int G = num_heads / num_kv_heads;  // query heads per kv head (<= kAttnMaxGroup)
  float* red = sm;                          // [waves][G][HS] outputs
  float* ml = red + W * G * HS;             // [waves][G][2] max, sum

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int seq = blockIdx.x / num_kv_heads;
  const int kvh = blockIdx.x % num_kv_heads;
  const int part = blockIdx.y;
  const int h0 = kvh * G;
  // a context longer than the block table is cut to it (never read past a row)
  const int ctx = min(context_lens[seq], max_blocks * BS);
  const int t0 = part * part_tokens;
  const int t1 = min(ctx, t0 + part_tokens);
  const int nt = t1 - t0;
  const bool direct = num_parts == 1;
  if (nt <= 0) {  // partition past this sequence's context: an empty partial
    if (!direct && tid < G) {
      const size_t r = ((size_t)seq * num_heads + h0 + tid) * num_parts + part;
      ws_ml[2 * r] = -FLT_MAX;
      ws_ml[2 * r + 1] = 0.f;
    }
    return;
  }
  const int c = lane & 15;   // operand row (token, dim) or column (head)
  const int qd = lane >> 4;  // 8-element group of the reduction
  const int nb = (nt + BS - 1) / BS;
  const int nsteps = (nt + 31) / 32;
  const int nsw = wave < nsteps ? (nsteps - wave + W - 1) / W : 0;  // this wave's steps

  // Lane l holds the addresses of the wave's l-th block (its steps' blocks in
  // order; a partition of 4096 tokens has at most 64 per wave); blocks past the
  // partition repeat its last.
  uint64_t kp, vp;
  {
    const int32_t* btab = block_tables + (size_t)seq * max_blocks + t0 / BS;
    const int blk = btab[min((wave + W * (lane / NB)) * NB + lane % NB, nb - 1)];
    const size_t head = (size_t)kvh * kv_head_stride * sizeof(uint16_t);
    kp = (uint64_t)kptr[blk] + head;
    vp = (uint64_t)vptr[blk] + head;
  }
  auto block_of = [&](uint64_t v, int l) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), l);
    return ((uint64_t)hi << 32) | lo;
  };
  // q . k row c of tile u: token 8 (c / 4) + c % 4 + 4 u of the step
  const int ktok = 8 * (c >> 2) + (c & 3);
  const uint32_t koff = (uint32_t)((qd * BS + ktok % BS) * 16);
  const uint32_t voff = (uint32_t)((c * BS + (8 * qd) % BS) * 2);
  h8 kreg[SLOTS][2][NK], vreg[SLOTS][ND];
  auto load_k = [&](int slot, int i) {
    uint64_t base = block_of(kp, i * NB);
    if (NB == 2) {
      const uint64_t second = block_of(kp, i * NB + 1);
      base = c < 8 ? base : second;
    }
    const unsigned char* kb = reinterpret_cast<const unsigned char*>(base) + koff;
#pragma unroll
    for (int j = 0; j < NK; ++j)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (SLICES % 4 != 0 && 4 * j + qd >= SLICES) kreg[slot][u][j] = h8{};
        else kreg[slot][u][j] = *(const h8*)(kb + j * (4 * BS * 16) + u * 64);
      }
  };
  auto load_v = [&](int slot, int i) {
    uint64_t base = block_of(vp, i * NB);
    if (NB == 2) {
      const uint64_t second = block_of(vp, i * NB + 1);
      base = qd < 2 ? base : second;
    }
    const unsigned char* vb = reinterpret_cast<const unsigned char*>(base) + voff;
#pragma unroll
    for (int j = 0; j < ND; ++j) vreg[slot][j] = *(const h8*)(vb + j * (16 * BS * 2));
  };
#pragma unroll
  for (int u = 0; u < SLOTS; ++u)
    if (u < nsw) {
      load_k(u, u);
      load_v(u, u);
    }
  // the group's queries as B operands: column c is head h0 + c, zero past G
  h8 qreg[NK];
  {
    const uint16_t* qp = query + (size_t)seq * q_stride + (size_t)(h0 + min(c, G - 1)) * HS + 8 * qd;
#pragma unroll
    for (int j = 0; j < NK; ++j)
      qreg[j] = c < G && 4 * j + qd < SLICES ? *(const h8*)(qp + 32 * j) : h8{};
  }
  const float slope = alibi != nullptr && c < G ? alibi[h0 + c] : 0.f;

  float m = -FLT_MAX, l = 0.f;  // of head c (l: this lane's tokens)
  f4 o[ND];
#pragma unroll
  for (int j = 0; j < ND; ++j) o[j] = f4{0.f, 0.f, 0.f, 0.f};
  h8 pp[3];
  auto softmax = [&](int slot, int i) {
    f4 s[2] = {f4{0.f, 0.f, 0.f, 0.f}, f4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int j = 0; j < NK; ++j)
#pragma unroll
      for (int u = 0; u < 2; ++u) s[u] = mfma16(kreg[slot][u][j], qreg[j], s[u]);
    const int t = t0 + (wave + W * i) * 32 + 8 * qd;  // token of element 0
    float lg[8], mx = -FLT_MAX;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float v = scale * s[e >> 2][e & 3];
      if (alibi != nullptr) v += slope * (float)(t + e - ctx + 1);
      lg[e] = t + e < t1 ? v : -FLT_MAX;
      mx = fmaxf(mx, lg[e]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float mn = fmaxf(m, mx);
    if (__any(mn != m)) {
      const float a = exp_of(m - mn);
      l *= a;
#pragma unroll
      for (int j = 0; j < ND; ++j) o[j] *= a;
    }
    m = mn;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float p = t + e < t1 ? exp_of(lg[e] - mn) : 0.f;
      l += p;
      const float ps = p * kPScale;
      // p > 0 keeps every part > 0 (at least fp16's smallest), so p times an
      // infinite value is that infinity
      const float least = fminf(ps * 0x1p100f, 0x1p-24f);
      float rest = ps;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const h2 part = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pkrtz(fmaxf(rest, least), 0.f));
        pp[k][e] = part[0];
        rest -= (float)part[0];  // exact
      }
    }
  };
  auto pv = [&](int slot, int i) {
    const int t = (wave + W * i) * 32;  // within the partition
    if (t + 32 > nt) {
      // slots past the context may hold anything: never multiply them
      const int valid = nt - t - 8 * qd;
#pragma unroll
      for (int j = 0; j < ND; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          vreg[slot][j][e] = e < valid ? vreg[slot][j][e] : (_Float16)0.f;
    }
#pragma unroll
    for (int j = 0; j < ND; ++j)
#pragma unroll
      for (int k = 0; k < 3; ++k) o[j] = mfma16(vreg[slot][j], pp[k], o[j]);
  };
  for (int i0 = 0; i0 < nsw; i0 += SLOTS) {
#pragma unroll
    for (int u = 0; u < SLOTS; ++u) {
      const int i = i0 + u;
      if (i < nsw) {
        softmax(u, i);
        if (i + SLOTS < nsw) load_k(u, i + SLOTS);
        pv(u, i);
        if (i + SLOTS < nsw) load_v(u, i + SLOTS);
      }
    }
  }

  // ---- the waves' outputs, combined in wave order
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  if (c < G) {
#pragma unroll
    for (int j = 0; j < ND; ++j) *(f4*)(red + (wave * G + c) * HS + j * 16 + 4 * qd) = o[j];
    if (qd == 0) {
      ml[(wave * G + c) * 2] = m;
      ml[(wave * G + c) * 2 + 1] = l;
    }
  }
  __syncthreads();
  for (int i = tid; i < G * HS; i += W * 64) {
    const int g = i / HS, d = i % HS;
    float gm = ml[g * 2];
#pragma unroll
    for (int w = 1; w < W; ++w) gm = fmaxf(gm, ml[(w * G + g) * 2]);
    float sum = 0.f, acc = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float a = exp_of(ml[(w * G + g) * 2] - gm);
      sum += a * ml[(w * G + g) * 2 + 1];
      acc += a * red[(w * G + g) * HS + d];
    }
    acc *= 1.f / kPScale;
    if (direct) {
      out[(size_t)seq * o_stride + (size_t)(h0 + g) * HS + d] = h_bits((_Float16)(acc / sum));
    } else {
      const size_t r = ((size_t)seq * num_heads + h0 + g) * num_parts + part;
      ws_out[r * HS + d] = acc;
      if (d == 0) {
        ws_ml[2 * r] = gm;
        ws_ml[2 * r + 1] = sum;
      }
    }
  }
}

// Combine the partitions of one (sequence, head) in partition order.
template <int HS>
__global__ void __launch_bounds__(HS)
paged_attention_reduce_kernel(uint16_t* __restrict__ out, int64_t o_stride, int num_heads,
                              const int32_t* __restrict__ context_lens, int max_tokens,
                              int part_tokens,
                              int num_parts, const float* __restrict__ ws_ml,
                              const float* __restrict__ ws_out) {
  const int seq = blockIdx.x / num_heads, h = blockIdx.x % num_heads;
  const int d = threadIdx.x;
  const int ctx = min(context_lens[seq], max_tokens);
  const int parts = min(num_parts, (ctx + part_tokens - 1) / part_tokens);
  const size_t r0 = ((size_t)seq * num_heads + h) * num_parts;
  // Running max and rescaled sums over the partitions in order; the loads
  // of a batch of 8 partitions are all in flight before the first update.
  float gmax = -FLT_MAX, total = 0.f, o = 0.f;
  for (int p0 = 0; p0 < parts; p0 += 8) {
    float m[8], l[8], v[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const bool in = p0 + b < parts;
      m[b] = in ? ws_ml[2 * (r0 + p0 + b)] : -FLT_MAX;
      l[b] = in ? ws_ml[2 * (r0 + p0 + b) + 1] : 0.f;
      v[b] = in ? ws_out[(r0 + p0 + b) * HS + d] : 0.f;
    }
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      if (p0 + b < parts) {
        const float nm = fmaxf(gmax, m[b]);
        const float a = __expf(gmax - nm), w = __expf(m[b] - nm);
        total = total * a + l[b] * w;
        o = o * a + v[b] * w;
        gmax = nm;
      }
    }
  }
  out[(size_t)seq * o_stride + (size_t)h * HS + d] = h_bits((_Float16)(o / total));
}

// One workgroup per token: its key and value rows go to their slot.
// restore: the reverse copy (slots to the token-major tensors).  Used where
// the token rows are not 16-byte aligned; cache_tile_kernel takes the rest.
__global__ void reshape_and_cache_kernel(uint16_t* __restrict__ key, int64_t key_stride,
                                         uint16_t* __restrict__ value, int64_t value_stride,
                                         const int64_t* __restrict__ kptr,
                                         const int64_t* __restrict__ vptr,
                                         const int64_t* __restrict__ slots, int num_kv_heads,
                                         int head_size, int block_size, int kv_head_stride,
                                         bool restore) {
  const int64_t tok = blockIdx.x;
  const int64_t slot = slots[tok];
  if (slot < 0) return;  // padding token
  const int64_t blk = slot / block_size;
  const int off = (int)(slot % block_size);
  uint16_t* kc = reinterpret_cast<uint16_t*>(kptr[blk]);
  uint16_t* vc = reinterpret_cast<uint16_t*>(vptr[blk]);
  const int n = num_kv_heads * head_size;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const int h = i / head_size, d = i % head_size;
    const size_t kt = (size_t)h * kv_head_stride + ((size_t)(d / 8) * block_size + off) * 8 + d % 8;
    const size_t vt = (size_t)h * kv_head_stride + (size_t)d * block_size + off;
    if (restore) {
      key[tok * key_stride + i] = kc[kt];
      value[tok * value_stride + i] = vc[vt];
    } else {
      kc[kt] = key[tok * key_stride + i];
      vc[vt] = value[tok * value_stride + i];
    }
  }
}

// Token rows to their cache slots (RESTORE: back), one workgroup per (32
// tokens, kv head).  HBM-bound: every byte is read and written once, so what
// counts is that both sides move whole 16-byte units in 128-byte runs.
//   * keys: a 16-byte unit (8 dims of a token) is contiguous on both sides; a
//     wave takes 8 tokens x 8 units, 128-byte runs of the rows and, for
//     consecutive slots, of the cache block;
//   * values: a cache row holds one dim of a block's tokens, so the tile is
//     turned around in LDS.  Eight tokens in consecutive slots that start at
//     a multiple of 8 (a "cell") move as one 16-byte unit per dim; the other
//     tokens (ends of a run, scattered slots, blocks whose address is not
//     16-byte aligned) as 2-byte elements.  Tiles start slots[0] % 8 tokens
//     early, so a run that continues a half-filled cell still meets the
//     tile in whole cells.
// Measured, 1500 tokens x 32 heads x 128 written and read back: 67.7 -> 22.4 us
// against element-wise copies (2-byte stores, one workgroup per token).
constexpr int kCacheTile = 32;                 // tokens per workgroup
constexpr int kCacheSlab = 128;                // dims per pass
constexpr int kCachePitch = kCacheSlab + 4;    // halfs per LDS row: the 4 cells of a dim pair
                                               // read 4 x 16 distinct banks

template <bool RESTORE, int THREADS>
__global__ void __launch_bounds__(THREADS)
cache_tile_kernel(uint16_t* __restrict__ key, int64_t key_stride, uint16_t* __restrict__ value,
                  int64_t value_stride, const int64_t* __restrict__ kptr,
                  const int64_t* __restrict__ vptr, const int64_t* __restrict__ slots,
                  int num_tokens, int head_size, int bs_log2, int kv_head_stride) {
  __shared__ __attribute__((aligned(16))) uint16_t tile[kCacheTile * kCachePitch];
  __shared__ int64_t slot_s[kCacheTile];
  __shared__ uint16_t* kbase[kCacheTile];  // token's block (this head), null: skip the token
  __shared__ uint16_t* vbase[kCacheTile];
  __shared__ int cell_ok[kCacheTile / 8];
  const int tid = threadIdx.x;
  const int head = blockIdx.y;
  const int bs = 1 << bs_log2;
  const int64_t first = slots[0];
  const int t0 = (int)blockIdx.x * kCacheTile - (first >= 0 ? (int)(first & 7) : 0);
  if (tid < kCacheTile) {
    const int t = t0 + tid;
    const int64_t slot = t >= 0 && t < num_tokens ? slots[t] : -1;
    slot_s[tid] = slot;
    kbase[tid] = nullptr;
    vbase[tid] = nullptr;
    if (slot >= 0) {
      const int64_t blk = slot >> bs_log2;
      kbase[tid] = reinterpret_cast<uint16_t*>(kptr[blk]) + (size_t)head * kv_head_stride;
      vbase[tid] = reinterpret_cast<uint16_t*>(vptr[blk]) + (size_t)head * kv_head_stride;
    }
  }
  __syncthreads();
  if (tid < kCacheTile / 8) {
    const int64_t s0 = slot_s[tid * 8];
    bool ok = s0 >= 0 && (s0 & 7) == 0 &&
              (reinterpret_cast<uintptr_t>(vbase[tid * 8]) & 15) == 0;
    for (int i = 1; i < 8; ++i) ok = ok && slot_s[tid * 8 + i] == s0 + i;
    cell_ok[tid] = ok;
  }
  __syncthreads();
  const int off_mask = bs - 1;
  const bool singles = !(cell_ok[0] & cell_ok[1] & cell_ok[2] & cell_ok[3]);
  uint16_t* const krow = key + (size_t)head * head_size;
  uint16_t* const vrow = value + (size_t)head * head_size;

  for (int d0 = 0; d0 < head_size; d0 += kCacheSlab) {
    const int nd = min(kCacheSlab, head_size - d0);  // a multiple of 8
    const int nu = nd / 8;
    // ---- keys, 16-byte units: 8 tokens x 8 units per wave
    for (int i = tid; i < kCacheTile * (kCacheSlab / 8); i += THREADS) {
      const int w = i >> 6, l = i & 63;
      const int t = (w & 3) * 8 + (l & 7);
      const int u = (w >> 2) * 8 + (l >> 3);
      if (u >= nu || kbase[t] == nullptr) continue;
      uint16_t* row = krow + (size_t)(t0 + t) * key_stride + d0 + u * 8;
      uint16_t* unit = kbase[t] + ((size_t)(d0 / 8 + u) * bs + (int)(slot_s[t] & off_mask)) * 8;
      uint16_t* const dst = RESTORE ? row : unit;
      const uint16_t* const src = RESTORE ? unit : row;
      if ((reinterpret_cast<uintptr_t>(unit) & 15) == 0) {
        *(u4*)dst = *(const u4*)src;
      } else {
        for (int e = 0; e < 8; ++e) dst[e] = src[e];
      }
    }
    // ---- values
    auto rows = [&](auto&& move) {  // (tile address, row address) per 16-byte unit of a token
      for (int i = tid; i < kCacheTile * (kCacheSlab / 8); i += THREADS) {
        const int t = i / (kCacheSlab / 8), u = i % (kCacheSlab / 8);
        if (u >= nu || vbase[t] == nullptr) continue;
        move(&tile[t * kCachePitch + u * 8], vrow + (size_t)(t0 + t) * value_stride + d0 + u * 8);
      }
    };
    auto cells = [&](auto&& move) {  // (tile address of the cell's first token, cache address)
      for (int i = tid; i < (kCacheTile / 8) * (kCacheSlab / 2); i += THREADS) {
        const int c = i % (kCacheTile / 8), dp = i / (kCacheTile / 8);
        if (2 * dp >= nd || !cell_ok[c]) continue;
        move(&tile[c * 8 * kCachePitch + 2 * dp],
             vbase[c * 8] + (size_t)(d0 + 2 * dp) * bs + (int)(slot_s[c * 8] & off_mask));
      }
    };
    // tokens outside whole cells: a thread's token, and its dims kStep apart
    const int et = tid % kCacheTile;
    const bool single = singles && !cell_ok[et >> 3] && vbase[et] != nullptr;
    uint16_t* const erow = tile + et * kCachePitch;
    uint16_t* const ecol = single ? vbase[et] + (size_t)d0 * bs + (int)(slot_s[et] & off_mask) : nullptr;
    constexpr int kStep = THREADS / kCacheTile, kEach = kCacheSlab / kStep;
    if (!RESTORE) {
      rows([](uint16_t* lds, const uint16_t* row) {
        const u4 v = *(const u4*)row;
        *(uint2*)lds = make_uint2(v[0], v[1]);
        *(uint2*)(lds + 4) = make_uint2(v[2], v[3]);
      });
      __syncthreads();
      cells([&](const uint16_t* lds, uint16_t* dst) {
        u4 lo, hi;  // 8 tokens of the even and of the odd dim
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t a = *(const uint32_t*)(lds + (2 * e) * kCachePitch);
          const uint32_t b = *(const uint32_t*)(lds + (2 * e + 1) * kCachePitch);
          lo[e] = (a & 0xFFFFu) | (b << 16);
          hi[e] = (a >> 16) | (b & 0xFFFF0000u);
        }
        *(u4*)dst = lo;
        *(u4*)(dst + bs) = hi;
      });
      if (single)
        for (int d = tid / kCacheTile; d < nd; d += kStep) ecol[(size_t)d * bs] = erow[d];
    } else {
      cells([&](uint16_t* lds, const uint16_t* src) {
        const u4 lo = *(const u4*)src, hi = *(const u4*)(src + bs);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          *(uint32_t*)(lds + (2 * e) * kCachePitch) = (lo[e] & 0xFFFFu) | (hi[e] << 16);
          *(uint32_t*)(lds + (2 * e + 1) * kCachePitch) = (lo[e] >> 16) | (hi[e] & 0xFFFF0000u);
        }
      });
      if (single) {  // all loads in flight before the first is stored
        uint16_t v[kEach];
#pragma unroll
        for (int i = 0; i < kEach; ++i) {
          const int d = tid / kCacheTile + i * kStep;
          v[i] = d < nd ? ecol[(size_t)d * bs] : (uint16_t)0;
        }
#pragma unroll
        for (int i = 0; i < kEach; ++i) {
          const int d = tid / kCacheTile + i * kStep;
          if (d < nd) erow[d] = v[i];
        }
      }
      __syncthreads();
      rows([](const uint16_t* lds, uint16_t* row) {
        const uint2 a = *(const uint2*)lds, b = *(const uint2*)(lds + 4);
        *(u4*)row = u4{a.x, a.y, b.x, b.y};
      });
    }
    if (d0 + kCacheSlab < head_size) __syncthreads();  // the next slab reuses the tile
  }
}

template <int HS, int BS, int W>
hipError_t launch_pa_w(const PagedAttnArgs& a, const PagedAttnPlan& p, float* ws,
                       hipStream_t stream) {
  const size_t smem = attn_smem_bytes(HS, a.num_heads / a.num_kv_heads, W);
  const dim3 grid((unsigned)(a.num_seqs * a.num_kv_heads), (unsigned)p.num_parts);
  float* ws_ml = p.num_parts > 1 ? ws : nullptr;
  float* ws_out = p.num_parts > 1 ? ws + 2 * (size_t)a.num_seqs * a.num_heads * p.num_parts : nullptr;
  paged_attention_kernel<HS, BS, W><<<grid, W * 64, smem, stream>>>(
      a.query, a.q_stride, a.out, a.o_stride, a.kptr, a.vptr, a.kv_head_stride, a.num_heads,
      a.num_kv_heads, a.scale, a.block_tables, a.max_blocks, a.context_lens, a.alibi,
      p.part_tokens, p.num_parts, ws_ml, ws_out);
  return hipGetLastError();
}

template <int HS, int BS, int W>
hipError_t launch_pa_row(const PagedAttnArgs& a, const PagedAttnPlan& p, float* ws,
                         hipStream_t stream) {
  const size_t smem = attn_row_smem_bytes(HS, p.part_tokens, W);
  const dim3 grid((unsigned)(a.num_seqs * a.num_heads), (unsigned)p.num_parts);
  float* ws_ml = p.num_parts > 1 ? ws : nullptr;
  float* ws_out = p.num_parts > 1 ? ws + 2 * (size_t)a.num_seqs * a.num_heads * p.num_parts : nullptr;
  paged_attention_row_kernel<HS, BS, W><<<grid, W * 64, smem, stream>>>(
      a.query, a.q_stride, a.out, a.o_stride, a.kptr, a.vptr, a.kv_head_stride, a.num_heads,
      a.scale, a.block_tables, a.max_blocks, a.context_lens, a.alibi, p.part_tokens, p.num_parts,
      ws_ml, ws_out);
  return hipGetLastError();
}

template <int HS, int BS>
hipError_t launch_pa(const PagedAttnArgs& a, const PagedAttnPlan& p, float* ws,
                     hipStream_t stream) {
  hipError_t e = hipErrorInvalidValue;
  if (a.num_heads == a.num_kv_heads) {
    if (p.waves == 4) e = launch_pa_row<HS, BS, 4>(a, p, ws, stream);
    if constexpr (HS <= 128 && BS == 16)
      if (p.waves == 16) e = launch_pa_row<HS, BS, 16>(a, p, ws, stream);
  } else {
    if (p.waves == 4) e = launch_pa_w<HS, BS, 4>(a, p, ws, stream);
    if constexpr (HS <= 128)
      if (p.waves == 8) e = launch_pa_w<HS, BS, 8>(a, p, ws, stream);
  }
  if (e != hipSuccess || p.num_parts == 1) return e;
  float* ws_ml = ws;
  float* ws_out = ws + 2 * (size_t)a.num_seqs * a.num_heads * p.num_parts;
  paged_attention_reduce_kernel<HS><<<(unsigned)(a.num_seqs * a.num_heads), HS, 0, stream>>>(
      a.out, a.o_stride, a.num_heads, a.context_lens, a.max_blocks * BS, p.part_tokens,
      p.num_parts, ws_ml, ws_out);
  return hipGetLastError();
}

template <int HS>
hipError_t launch_pa_bs(const PagedAttnArgs& a, const PagedAttnPlan& p, float* ws,
                        hipStream_t stream) {
  if (a.block_size == 16) return launch_pa<HS, 16>(a, p, ws, stream);
  return launch_pa<HS, 32>(a, p, ws, stream);
}

// Rotary embedding, rotate-half form, in place on fp16 rows [batch][rows][hd]
// (row = token * heads + head): position p = past + row / heads, pair
// (l, r) = (x[c], x[c + hd/2]):
//   l' = fma(l, cos[p][c], fp16(r * -sin[p][c]))
//   r' = fma(r, cos[p][c + hd/2], fp16(l * sin[p][c + hd/2]))
// each product and each fma rounded once in fp16, as the reference's
// half-precision kernel (cuda_extends/exllama/fuse_v2/rope.cu:24-91) does.
__global__ void rope_kernel(uint16_t* __restrict__ x, const uint16_t* __restrict__ sinp,
                            const uint16_t* __restrict__ cosp, int rows, int hd, int heads,
                            int max_pos, int past_len, const int32_t* __restrict__ past_lens) {
  const int half = hd / 2;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int c = (int)(i % half);
  const int64_t row = i / half;  // within this batch entry
  if (row >= rows) return;
  const int b = blockIdx.y;
  const int pos = (past_len >= 0 ? past_len : past_lens[b]) + (int)(row / heads);
  if (pos < 0 || pos >= max_pos) return;  // outside the table: row left as it is
  uint16_t* xr = x + ((int64_t)b * rows + row) * hd;
  const _Float16 l = as_h(xr[c]), r = as_h(xr[c + half]);
  const _Float16 cl = as_h(cosp[(int64_t)pos * hd + c]), cr = as_h(cosp[(int64_t)pos * hd + c + half]);
  const _Float16 sl = as_h(sinp[(int64_t)pos * hd + c]), sr = as_h(sinp[(int64_t)pos * hd + c + half]);
  const _Float16 ls = r * (_Float16)(-sl);
  const _Float16 rs = l * sr;
  xr[c] = h_bits(__builtin_fmaf16(l, cl, ls));
  xr[c + half] = h_bits(__builtin_fmaf16(r, cr, rs));
}

// One decode token per sequence: its q and k rows rotated in place (the
// arithmetic of rope_kernel, position p = positions[t]), the rotated k row
// and the v row written to slot block_tables[t][p / bs] * bs + p % bs, and
// p + 1 stored to lens_out[t] (if given) -- rope on q and k, then
// reshape_and_cache, in one launch.  A position outside the block table
// writes no slot; one outside the sin/cos tables leaves q and k unrotated.
// Grid: (sequence, head slot) with head slots [0, heads) the q heads, then
// the kv heads (rotate k, write k and v to the slot); 64 threads, one
// (l, r) pair (or two v elements) each, so no thread loops.
__global__ void __launch_bounds__(64)
rope_cache_kernel(uint16_t* __restrict__ q, int64_t q_stride, uint16_t* __restrict__ k,
                  int64_t k_stride, const uint16_t* __restrict__ v, int64_t v_stride,
                  const uint16_t* __restrict__ sinp, const uint16_t* __restrict__ cosp,
                  int max_pos, const int32_t* __restrict__ positions,
                  const int32_t* __restrict__ block_tables, int max_blocks,
                  const int64_t* __restrict__ kptr, const int64_t* __restrict__ vptr,
                  int kv_head_stride, int32_t* __restrict__ lens_out, int heads, int kv_heads,
                  int hd, int bs) {
  const int t = blockIdx.x, slot = blockIdx.y, tid = threadIdx.x;
  const int p = positions[t];
  if (lens_out != nullptr && slot == 0 && tid == 0) lens_out[t] = p + 1;
  const int half = hd / 2;
  const bool rot = p >= 0 && p < max_pos;
  const bool store = p >= 0 && p / bs < max_blocks;
  const bool is_q = slot < heads;
  const int h = is_q ? slot : slot - heads;
  uint16_t* row = is_q ? q + t * q_stride + h * hd : k + t * k_stride + h * hd;
  const uint16_t* sr = sinp + (int64_t)(rot ? p : 0) * hd;
  const uint16_t* cr = cosp + (int64_t)(rot ? p : 0) * hd;
  uint16_t* kh = nullptr;
  uint16_t* vh = nullptr;
  int off = 0;
  if (!is_q && store) {
    const int blk = block_tables[(int64_t)t * max_blocks + p / bs];
    kh = reinterpret_cast<uint16_t*>(kptr[blk]) + (size_t)h * kv_head_stride;
    vh = reinterpret_cast<uint16_t*>(vptr[blk]) + (size_t)h * kv_head_stride;
    off = p % bs;
  }
  for (int c = tid; c < half; c += 64) {
    _Float16 l = as_h(row[c]), r = as_h(row[c + half]);
    if (rot) {
      const _Float16 ls = r * (_Float16)(-as_h(sr[c]));
      const _Float16 rs = l * as_h(sr[c + half]);
      l = __builtin_fmaf16(l, as_h(cr[c]), ls);
      r = __builtin_fmaf16(r, as_h(cr[c + half]), rs);
      row[c] = h_bits(l);
      row[c + half] = h_bits(r);
    }
    if (kh != nullptr) {
      kh[((c / 8) * bs + off) * 8 + c % 8] = h_bits(l);
      kh[(((c + half) / 8) * bs + off) * 8 + (c + half) % 8] = h_bits(r);
    }
  }
  if (vh != nullptr) {
    const uint16_t* vr = v + t * v_stride + h * hd;
    for (int d = tid; d < hd; d += 64) vh[(size_t)d * bs + off] = vr[d];
  }
}

}  // namespace

hipError_t launch_rope_cache(const RopeCacheArgs& a, hipStream_t stream) {
  const dim3 grid((unsigned)a.num_seqs, (unsigned)(a.heads + a.kv_heads));
  rope_cache_kernel<<<grid, 64, 0, stream>>>(
      a.q, a.q_stride, a.k, a.k_stride, a.v, a.v_stride, a.sinp, a.cosp, a.max_pos, a.positions,
      a.block_tables, a.max_blocks, a.kptr, a.vptr, a.kv_head_stride, a.lens_out, a.heads,
      a.kv_heads, a.hd, a.bs);
  return hipGetLastError();
}

hipError_t launch_rope(uint16_t* x, const uint16_t* sinp, const uint16_t* cosp, int batch,
                       int rows, int hd, int heads, int max_pos, int past_len,
                       const int32_t* past_lens, hipStream_t stream) {
  const int64_t n = (int64_t)rows * (hd / 2);
  const dim3 grid((unsigned)((n + 255) / 256), (unsigned)batch);
  rope_kernel<<<grid, 256, 0, stream>>>(x, sinp, cosp, rows, hd, heads, max_pos, past_len,
                                        past_lens);
  return hipGetLastError();
}

PagedAttnPlan plan_paged_attention(int num_seqs, int num_heads, int num_kv_heads, int head_size,
                                   int block_size, int max_context_len, int cus) {
  PagedAttnPlan p;
  const int blocks = std::max(1, (max_context_len + block_size - 1) / block_size);
  const int pairs = std::max(1, num_seqs * num_kv_heads);
  if (num_heads == num_kv_heads) {
    // one 16-wave workgroup per (sequence, head) over the whole context where
    // that gives every CU about one workgroup and the context fits one
    // partition: no combine launch
    if (head_size <= 128 && block_size == 16 && 2 * pairs > cus && pairs <= cus &&
        blocks * block_size <= kAttnRowWideTokens) {
      p.waves = 16;
      p.part_tokens = blocks * block_size;
      p.num_parts = 1;
      return p;
    }
    // about four workgroups per CU (eight measured no faster); partitions of
    // whole blocks, at most 512 tokens
    const int parts = std::min(std::max(1, (4 * cus + pairs - 1) / pairs), blocks);
    const int bpp = std::min((blocks + parts - 1) / parts, kAttnRowPartTokens / block_size);
    p.part_tokens = bpp * block_size;
    p.num_parts = (blocks + bpp - 1) / bpp;
    return p;
  }
  // One 8-wave workgroup per (sequence, kv head) over the whole context, no
  // combine launch, where that gives at least half of the CUs one (for
  // contexts up to 1024 tokens, whose combine launch would count for more, a
  // third) and none two.  Measured (us, partitioned -> this): 6 x 500 tokens, 32
  // heads of 128 14.2 -> 11.5; 24 x 3000, 8 kv heads 46.6 -> 42.9; 3 x 800, 40
  // heads 15.3 -> 12.7.
  if (head_size <= 128 && pairs <= cus && blocks * block_size <= kAttnWideMaxTokens &&
      (2 * pairs > cus || (10 * pairs > 3 * cus && blocks * block_size <= 1024))) {
    p.waves = 8;
    p.part_tokens = blocks * block_size;
    p.num_parts = 1;
    return p;
  }
  // Otherwise about one 4-wave workgroup per CU, so two on most of the CUs (all
  // their registers hold); partitions of whole blocks, at least 128 tokens (a
  // step per wave; 256 for long contexts, whose combine launch reads fewer),
  // at most 4096.  Measured (us, at least 16 tokens and four workgroups per CU
  // -> this): 1 x 4000 tokens, 8 kv heads 31.3 -> 12.1; 32 x 1000 28.2 -> 22.8;
  // 8 x 3000, 16 heads of 256 61.0 -> 54.4.
  const int least = max_context_len > kAttnShortContext ? 2 * kAttnLeastPart : kAttnLeastPart;
  int parts = (cus + pairs - 1) / pairs;
  parts = std::max(1, std::min(parts, (max_context_len + least - 1) / least));
  int bpp = (blocks + parts - 1) / parts;
  bpp = std::min(bpp, kAttnMaxPartTokens / block_size);
  p.part_tokens = bpp * block_size;
  p.num_parts = (blocks + bpp - 1) / bpp;
  return p;
}

size_t paged_attention_ws_bytes(const PagedAttnPlan& p, int num_seqs, int num_heads,
                                int head_size) {
  if (p.num_parts <= 1) return 0;
  return sizeof(float) * (size_t)num_seqs * num_heads * p.num_parts * (2 + (size_t)head_size);
}

// Fewer sequences or a shorter context can take more partitions than the
// largest call does (which may be one workgroup per pair, with none), so with
// grouped heads the size is a bound over all of them: seqs * parts is at most
// cus / kv_heads + seqs by the workgroups wanted, seqs times the most
// partitions of any context up to this one by their least size, and seqs times
// the partitions of 4096 tokens.
size_t paged_attention_ws_upto(int num_seqs, int num_heads, int num_kv_heads, int head_size,
                               int block_size, int max_context_len, int cus) {
  if (num_seqs == 0) return 0;
  if (num_heads == num_kv_heads)
    return paged_attention_ws_bytes(plan_paged_attention(num_seqs, num_heads, num_kv_heads, head_size,
                                                         block_size, max_context_len, cus),
                                    num_seqs, num_heads, head_size);
  auto ceil_of = [](int a, int b) { return a / b + (a % b != 0); };
  int most = ceil_of(std::min(max_context_len, kAttnShortContext), kAttnLeastPart);
  if (max_context_len > kAttnShortContext)
    most = std::max(most, ceil_of(max_context_len, 2 * kAttnLeastPart));
  const int64_t wanted = std::min((int64_t)num_seqs * most, (int64_t)ceil_of(cus, num_kv_heads) + num_seqs);
  const int64_t full = (int64_t)num_seqs * ceil_of(max_context_len, kAttnMaxPartTokens);
  const int64_t rows = std::max(wanted, full);
  return most <= 1 ? 0 : sizeof(float) * (size_t)rows * num_heads * (2 + (size_t)head_size);
}

hipError_t launch_paged_attention(const PagedAttnArgs& a, const PagedAttnPlan& p, float* ws,
                                  hipStream_t stream) {
  switch (a.head_size) {
    case 64: return launch_pa_bs<64>(a, p, ws, stream);
    case 80: return launch_pa_bs<80>(a, p, ws, stream);
    case 96: return launch_pa_bs<96>(a, p, ws, stream);
    case 112: return launch_pa_bs<112>(a, p, ws, stream);
    case 128: return launch_pa_bs<128>(a, p, ws, stream);
    case 256: return launch_pa_bs<256>(a, p, ws, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_reshape_and_cache(uint16_t* key, int64_t key_stride, uint16_t* value,
                                    int64_t value_stride, const int64_t* kptr, const int64_t* vptr,
                                    const int64_t* slots, int num_tokens, int num_kv_heads,
                                    int head_size, int block_size, int kv_head_stride,
                                    bool restore, hipStream_t stream) {
  // The tiles need whole 16-byte units on the rows' side (the kernel itself
  // checks the blocks' addresses), and take 3 us for a single token; the
  // element-wise copy, a workgroup of up to 1024 lanes per token, starts faster
  // the narrower a row is.  Runs of tokens written and read back, element-wise
  // against tiles (us): 8 heads of 128 256 tokens 7.6 / 8.0, 512 11.0 / 8.0; 16
  // of 128 128 tokens 8.7 / 8.1, 256 11.1 / 8.2; 32 of 128 1 token 8.9 / 6.5, 64
  // 12.4 / 8.0, 1500 67 / 22.  Tokens one to a block, which neither form can
  // read or write in whole units, lose some us to the tile's steps in between:
  // 32 of 128 64 tokens 14.0 / 15.9, 256 55 / 62, 1500 350 / 350.
  const bool vec = ((reinterpret_cast<uintptr_t>(key) | reinterpret_cast<uintptr_t>(value)) & 15) == 0 &&
                   key_stride % 8 == 0 && value_stride % 8 == 0;
  const bool wide = num_kv_heads * head_size / 8 + (int64_t)num_tokens >= 512;
  if (vec && wide) {
    const dim3 grid((unsigned)((num_tokens + 7 + kCacheTile - 1) / kCacheTile), (unsigned)num_kv_heads);
    const int bs_log2 = block_size == 16 ? 4 : 5;
    // up to three workgroups per CU (of 256) eight waves each, to have more
    // copies in flight (32 x 128, us, four / eight waves: 512 tokens 13.8 / 11.9,
    // 700 15.1 / 13.5); beyond that four (800 tokens 15.3 / 17.3, 1500 22.1 / 24.3)
    const bool few = (int64_t)grid.x * grid.y <= 768;
    auto kern = restore ? (few ? &cache_tile_kernel<true, 512> : &cache_tile_kernel<true, 256>)
                        : (few ? &cache_tile_kernel<false, 512> : &cache_tile_kernel<false, 256>);
    kern<<<grid, few ? 512 : 256, 0, stream>>>(key, key_stride, value, value_stride, kptr, vptr, slots,
                                               num_tokens, head_size, bs_log2, kv_head_stride);
    return hipGetLastError();
  }
  const int n = num_kv_heads * head_size;
  reshape_and_cache_kernel<<<(unsigned)num_tokens, std::min(1024, n), 0, stream>>>(
      key, key_stride, value, value_stride, kptr, vptr, slots, num_kv_heads, head_size,
      block_size, kv_head_stride, restore);
  return hipGetLastError();
}

}  // namespace dw4
