// Which neighbour positions a seed row keeps: the "dgs-philox-1" contract shared by the
// per-hop sampler (sample.hip), the fused sampler (pipeline.hip) and the CPU oracle.
#ifndef DGS_CSRC_PICKS_H_
#define DGS_CSRC_PICKS_H_

#include "common.h"

namespace dgs {

__host__ __device__ inline int64_t pick_count(int64_t deg, int64_t k, bool replace) {
  if (replace) return deg == 0 ? 0 : k;
  return deg < k ? deg : k;
}

// Whether a lower lane of the caller's G-lane group (of the `used` first lanes) holds the same value.
// No lane waits for what another one found, and no value makes a trip through LDS: within 16 lanes the
// values move as data-parallel-primitive operands, beyond that they are read into scalars.
template <int G>
__device__ __forceinline__ bool held_by_lower_lane(uint32_t v, int l, int used) {
  bool held = false;
  if constexpr (G <= 16) {
    // row_shr:r = the value r lanes below; lanes without one (and inactive ones) see ~v
#define DGS_LOWER(r) \
  if (r < G) held |= uint32_t(__builtin_amdgcn_update_dpp(int(~v), int(v), 0x110 + (r & 15), 0xf, 0xf, false)) == v && l >= r;
    DGS_LOWER(1) DGS_LOWER(2) DGS_LOWER(3) DGS_LOWER(4) DGS_LOWER(5) DGS_LOWER(6) DGS_LOWER(7)
    if constexpr (G == 16) {
      DGS_LOWER(8) DGS_LOWER(9) DGS_LOWER(10) DGS_LOWER(11) DGS_LOWER(12) DGS_LOWER(13) DGS_LOWER(14) DGS_LOWER(15)
    }
#undef DGS_LOWER
  } else {
    for (int s = 0; s + 1 < used; ++s) {
      uint32_t c = uint32_t(__builtin_amdgcn_readlane(int(v), s));
      if constexpr (G == 32) {
        const uint32_t upper = uint32_t(__builtin_amdgcn_readlane(int(v), 32 + s));
        c = (threadIdx.x & 32) ? upper : c;
      }
      held |= c == v && l > s;
    }
  }
  return held;
}

// Position inside the row for output slot l (0 <= l < G, k <= G) of a row of degree deg.
// All G lanes of the group call this together (G consecutive lanes of one wave, the first
// being lane group_lane0 of the wave); returns false when the slot holds no pick.
//   replacement:        slot l holds draw l reduced to [0, deg)
//   deg <= k:           the whole row, slot l = position l
//   deg >  k (Floyd):   slot s draws t in [0, deg-k+s] and keeps it unless a lower slot
//                       already kept t, in which case it keeps deg-k+s (which no lower slot
//                       can hold).
// Floyd's rule needs no walk over the slots.  A lower slot has kept t exactly if one of them drew t
// (the first that did kept it, or found it kept), or if t = deg-k+j for a lower slot j that kept its
// substitute deg-k+j: the first is a comparison of all pairs, the second a single link from a slot to
// a lower one, followed until nothing changes (once or twice as a rule: a chain of links needs a
// substitute drawn again).  Resolving slot after slot instead (a cross-lane read, a ballot and a
// dependent compare each) took a batch of 1024 seeds over fanouts [5,10,15], features and all, from
// 217 to 224 us.
// `words` is the Philox block of draw l of the row (philox_draw_words), which the caller may have
// computed before the degree was known.
template <int G>
__device__ __forceinline__ bool pick_position(uint32_t deg, int k, bool replace, int l, int group_lane0,
                                              const PhiloxWords& words, uint32_t* pos) {
  if (replace) {
    if (deg == 0 || l >= k) return false;
    *pos = philox_reduce(words, deg);
    return true;
  }
  if (deg <= uint32_t(k)) {
    *pos = uint32_t(l);
    return uint32_t(l) < deg;
  }
  const uint32_t top = deg - uint32_t(k) + uint32_t(l);
  uint32_t cand = 0xffffffffu;  // drawn by no slot
  if (l < k) cand = philox_reduce(words, top + 1u);
  const uint32_t link = cand - (deg - uint32_t(k));  // the slot whose substitute this candidate is (if below l)
  const bool linked = link < uint32_t(l) && l < k;
  const bool drawn_before = held_by_lower_lane<G>(cand, l, k);
  bool taken = drawn_before;
  uint64_t all = __ballot(taken);  // by lanes of the wave, every group's
  for (;;) {
    taken = drawn_before || (linked && ((all >> (uint32_t(group_lane0) + (linked ? link : 0u))) & 1) != 0);
    const uint64_t now = __ballot(taken);
    if (now == all) break;  // marks are only ever added: at most k rounds
    all = now;
  }
  *pos = taken ? top : cand;
  return l < k;
}

template <int G>
__device__ __forceinline__ bool pick_position(uint32_t deg, int k, bool replace, int l, int group_lane0,
                                              uint64_t rng_seed, uint32_t rng_stream, int64_t row,
                                              uint32_t* pos) {
  return pick_position<G>(deg, k, replace, l, group_lane0, philox_draw_words(rng_seed, rng_stream, row, uint32_t(l)),
                          pos);
}

}  // namespace dgs
#endif
