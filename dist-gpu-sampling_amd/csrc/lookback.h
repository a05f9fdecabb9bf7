// Exclusive prefix over the tiles of a launch inside that launch, after Merrill and Garland's single-pass
// scan with decoupled look-back: every tile's block publishes its count and adds up what the tiles before
// it published, so that counting, scanning and compacting a
// list take one launch instead of two or three (5 us of launch floor each on a short list).
//
// A tile's state word says how far it is: 0 nothing yet, kTileCount its own count, kTilePrefix the sum
// over all tiles up to and including it.  The words are the only thing that passes between blocks of
// the launch (relaxed agent-scope stores and loads of whole words: no other memory is ordered by
// them, so no fence), and must be zero when the launch begins.
//
// No block depends on another one's being scheduled: a word that stays zero for kLookbackPolls reads
// is replaced by a count of that tile done here (`recount`), so every wait ends whatever shares the
// GPU.  In practice blocks start in order and the words of earlier tiles are there at the first or
// second read.
#ifndef DGS_CSRC_LOOKBACK_H_
#define DGS_CSRC_LOOKBACK_H_

#include "common.h"

namespace dgs {

typedef unsigned long long tile_state;
constexpr tile_state kTileCount = 1ull << 62;
constexpr tile_state kTilePrefix = 2ull << 62;
constexpr int kTileFlagShift = 48;  // a word is status (2 bits), flags (8 bits, or-ed), sum (48 bits, added)
constexpr tile_state kTileSumMask = (1ull << kTileFlagShift) - 1;
constexpr int kLookbackPolls = 256;
// (test hook: n > 0 makes it n - 1, so that 1 has every prefix counted afresh; n < 0 makes it negative,
// which withholds the prefixes, so that every block reads its way back to the first tile)
inline int32_t lookback_polls() {
  const int64_t forced = debug_option(DGS_DEBUG_LOOKBACK_POLLS);
  return forced > 0 ? int32_t(forced - 1) : forced < 0 ? -kLookbackPolls : kLookbackPolls;
}

__host__ __device__ __forceinline__ tile_state tile_word(int64_t sum, uint32_t flags = 0) {
  return tile_state(sum) | (tile_state(flags) << kTileFlagShift);
}
__host__ __device__ __forceinline__ int64_t tile_sum_of(tile_state w) { return int64_t(w & kTileSumMask); }
__host__ __device__ __forceinline__ uint32_t tile_flags_of(tile_state w) { return uint32_t(w >> kTileFlagShift) & 0xffu; }
__device__ __forceinline__ tile_state tile_add(tile_state a, tile_state b) {  // of two words without status
  return tile_word(tile_sum_of(a) + tile_sum_of(b), tile_flags_of(a) | tile_flags_of(b));
}

template <int NT>
struct LookbackLds {
  tile_state part[NT / kWave];
  int found[NT / kWave];
  tile_state one;
};

// Called by all NT threads of the block of tile `tile` with the tile's own word (no status) and
// lookback_polls(), the number of times a word is read before it is counted instead; returns
// the combined word of the tiles before it.  `recount(t)` is called by the whole block and returns
// tile t's own word.  FLAGS: the words carry flags.
template <int NT, bool FLAGS, typename Recount>
__device__ __forceinline__ tile_state tile_exclusive_prefix(tile_state* state, int64_t tile, tile_state own,
                                                            int32_t max_polls, LookbackLds<NT>& lds, Recount recount) {
  constexpr int kItems = 1024 / NT;            // words a thread reads at a time: 1024 by the block
  constexpr int64_t kPerWave = kWave * kItems; // a wave reads consecutive words, the nearest ones wave 0
  constexpr tile_state kStatus = 3ull << 62;
  const int wave = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  if (threadIdx.x == 0)
    __hip_atomic_store(state + tile, own | (tile == 0 ? kTilePrefix : kTileCount), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int32_t reads = max_polls < 0 ? -max_polls : max_polls;
  tile_state before = 0;
  for (int64_t hi = tile; hi > 0;) {
    tile_state v[kItems];
    bool missing = true;
#pragma unroll
    for (int j = 0; j < kItems; ++j) v[j] = 0;
    for (int polls = 0; missing && polls < reads; ++polls) {
      missing = false;
#pragma unroll
      for (int j = 0; j < kItems; ++j) {
        const int64_t t = hi - 1 - (wave * kPerWave + j * kWave + lane);
        if (t >= 0 && v[j] == 0) v[j] = __hip_atomic_load(state + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        missing |= t >= 0 && v[j] == 0;
      }
      if (missing) __builtin_amdgcn_s_sleep(1);
    }
    if (__syncthreads_or(missing)) {  // somebody has not started: walk back word by word, counting where there is none
      for (int64_t t = hi - 1; t >= 0; --t) {
        __syncthreads();
        if (threadIdx.x == 0) lds.one = __hip_atomic_load(state + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        tile_state w = lds.one;
        if ((w & kStatus) == 0) w = recount(t) | kTileCount;
        before = tile_add(before, w & ~kStatus);
        if (w & kTilePrefix) break;
      }
      break;
    }
    // the nearest prefix among the wave's words, and the sum from there on (all of them if there is none)
    bool found = false;
    tile_state part = 0;
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const uint64_t at = __ballot((v[j] & kTilePrefix) != 0);
      const bool take = !found && (at == 0 || lane <= __builtin_ctzll(at));
      if (take) part = tile_add(part, v[j] & ~kStatus);
      found |= at != 0;
    }
    int64_t sum = tile_sum_of(part);
    uint32_t flags = tile_flags_of(part);
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) {
      sum += __shfl_xor(sum, d, kWave);
      if (FLAGS) flags |= __shfl_xor(flags, d, kWave);
    }
    if (lane == 0) {
      lds.part[wave] = tile_word(sum, flags);
      lds.found[wave] = found;
    }
    __syncthreads();
    bool done = false;
#pragma unroll
    for (int w = 0; w < NT / kWave; ++w) {
      if (!done) before = tile_add(before, lds.part[w]);
      done |= lds.found[w] != 0;
    }
    __syncthreads();  // the arrays are rewritten by the next round
    if (done) break;
    hi -= kPerWave * (NT / kWave);
  }
  if (threadIdx.x == 0 && tile != 0 && max_polls >= 0)
    __hip_atomic_store(state + tile, tile_add(before, own) | kTilePrefix, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return before;
}

}  // namespace dgs
#endif
