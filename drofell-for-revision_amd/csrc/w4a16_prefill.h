// Internal interface of the grouped prefill launches (w4a16_prefill.hip,
// w4a16_kslice.hip) for the C ABI (w4a16_capi.hip).  Not installed; the
// public ABI is include/drofell_w4a16.h.
#pragma once

#include "w4a16_device.h"
#include "w4a16_internal.h"

namespace dw4 {

// Several matrices of equal K, N and group size that share x (no act-order
// permutation) in one launch of the LDS-streamed prefill kernel: the plan's
// column tiles of every matrix, each matrix writing its own output (+ its
// bias, + its residual).  Unsplit plans only (splits == 1) for more than one
// matrix.
hipError_t launch_prefill2_group(const GroupArgs& a, const PrefillPlan& plan, void* ws,
                                 hipStream_t stream);
// The same on the K-sliced kernel (plan.kslice).
hipError_t launch_kslice_group(const GroupArgs& a, const PrefillPlan& plan, void* ws,
                               hipStream_t stream);

// Matrices of one launch: equal K, N and group size, each with its own
// packed buffers, bias, output and residual.  Column tile t of the launch
// belongs to matrix t / ntiles_item (tiles never straddle two matrices).
struct P2Items {
  const u4* pq[kGroupMax];
  const uint32_t* pz[kGroupMax];
  const uint32_t* ps[kGroupMax];
  const uint16_t* bias[kGroupMax];
  uint16_t* y[kGroupMax];
  int64_t ldy[kGroupMax];
  const uint16_t* res[kGroupMax];
  int64_t ldres[kGroupMax];
  int ntiles_item;
};

inline P2Items prefill_items(const GroupArgs& g, int bn) {
  P2Items it{};
  it.ntiles_item = (g.a[0].N + bn - 1) / bn;
  for (int i = 0; i < kGroupMax; ++i) {
    const GemmArgs& b = g.a[i < g.count ? i : 0];
    it.pq[i] = reinterpret_cast<const u4*>(b.pq);
    it.pz[i] = b.pz;
    it.ps[i] = reinterpret_cast<const uint32_t*>(b.ps);
    it.bias[i] = b.bias;
    it.y[i] = b.y;
    it.ldy[i] = b.ldy;
    it.res[i] = b.res;
    it.ldres[i] = b.ldres;
  }
  return it;
}

// x must already be in packed row order; one x, K, N and group size
inline bool same_x_shape(const GroupArgs& g) {
  if (g.count < 1 || g.count > kGroupMax) return false;
  for (int i = 0; i < g.count; ++i) {
    const GemmArgs& b = g.a[i];
    if (b.perm != nullptr || b.x != g.a[0].x || b.ldx != g.a[0].ldx || b.M != g.a[0].M ||
        b.K != g.a[0].K || b.N != g.a[0].N || b.gs != g.a[0].gs)
      return false;
  }
  return true;
}

// The prefill kernels address a row tile's activations by 32-bit byte offsets
// from its first row (at most 128 rows of 2 ldx bytes), so they take row
// strides up to this; wider ones keep the kernels with 64-bit addresses.
constexpr int64_t kPrefillMaxLdx = int64_t{1} << 22;
inline bool prefill_x_fits(int64_t ldx) { return ldx <= kPrefillMaxLdx; }

// ceil(2^32 / (chunks per group)), 0 where a chunk holds one group or more:
// the group of chunk c is then umulhi(c, magic) (exact while c times the
// chunks per group stays below 2^32).
inline uint32_t group_magic(int gs) {
  const uint64_t d = gs > kChunkK ? (uint64_t)(gs / kChunkK) : 1;
  return d <= 1 ? 0u : (uint32_t)(((1ull << 32) + d - 1) / d);
}

// XCD-aware workgroup order of the prefill kernels.  The (row tile, unit)
// pairs of a launch, a unit being a (column tile, K split) u = split * ntiles +
// ntile, run row tile first within a unit, in groups of group_m row tiles (a
// group's row tiles of unit 0, of unit 1, ..., then the next group's).
// Workgroup b runs on XCD b % 8 and takes pair b / 8 of the XCD's eighth of
// that sequence, so the workgroups an XCD runs at once share both their
// units' weights and the group's activation rows in its L2, and every XCD
// gets the same number of them.  (Dealing whole units to the XCDs instead
// left some with a unit more: 5120^2, M=700 in 64 x 256 tiles, 33 workgroups
// on four XCDs' 32 CUs, ran a second round: 90.0 us against 53.6.)
__device__ __forceinline__ bool tile_of(int b, int mtiles, int units, int group_m, int& mtile,
                                        int& unit) {
  const int total = mtiles * units;
  const int per = (total + 7) >> 3;
  const int p = (b & 7) * per + (b >> 3);
  if (p >= total) return false;
  const int grp = mtiles <= group_m ? 0 : p / (group_m * units);
  const int first_m = grp * group_m;
  const int gsz = min(mtiles - first_m, group_m);
  const int jj = p - first_m * units;
  unit = jj / gsz;
  mtile = first_m + jj - unit * gsz;
  return true;
}

// Row tiles per group: all of them up to 8 (a unit's weights then come into
// an XCD's L2 once), groups of 8 above.
constexpr int kPrefillGroupM = 8;
inline int prefill_group_m(int mtiles) { return mtiles <= kPrefillGroupM ? mtiles : kPrefillGroupM; }

}  // namespace dw4
