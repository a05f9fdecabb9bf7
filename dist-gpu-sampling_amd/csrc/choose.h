// Weighted picks: the rules of race.h for the fused sampler, laid out so that lanes belong to weights and draws.
// In a large hop many rows share a block (race_rows, draw_rows): half of all rows have a few dozen neighbours,
// and a wave for each leaves most of its lanes idle.  In a small one, where nothing but latency counts, every
// row has a wave that does it all without a barrier (race_by_wave, draw_by_wave).  Long rows have a block each
// (race_long, draw_long).
//
// Without replacement the race runs on 32-bit floats first.  An approximate key is off by less than half of what
// surely_less asks for, so entries that it orders are ordered as the 64-bit keys are; where the num_picks + 1
// smallest of a row are not all surely ordered (one row in some thousands), 64-bit keys settle it (race.h).  Rows
// of up to kShortRow positions: four positions to a lane, which is one Philox block, and then every position
// counts the smaller ones of its row.  Longer ones: a wave, or the waves of a block, that keep what is below a
// bar in an LDS list and lower the bar when the list fills.
//
// Measured, before (a wave per row, sorts, three passes over the weights) and with this: the hops of a batch of
// 1024 seeds, fanouts [5,10,15], rows of mean degree 50 up to 17 000, 28 / 36 / 84 us and 32 for the long rows'
// launch -> 27 / 28 / 63; 512 seeds with replacement 26 / 28 / 69 + 28 -> 18 / 19 / 31.  The whole batches
// 328 -> 274 and 214 -> 140 us.  Bound now: without replacement the atomics of the picks (31 us of the widest
// hop), then Philox and the counting; in a small hop the chain of waits (7 us for a wave's row) and its longest
// row (17 000 positions by one block: 21 us).
//
// Any weight above 0 has a float key.  Where one weight outside 2^-120 .. 2^90 sent its row to 64-bit keys, by
// one wave: 256 rows of 17 000 with one infinite weight each 171 us a call and now 68 (without it 67), two rows of
// 10^6 6.7 ms and 0.8, 1024 seeds, fanouts [5,10,10], rows of 60 with a fifth of the weights infinite 288 and 130.
//
// With replacement the shares of many rows are summed up in one scan over LDS, and every draw is a lane of its
// own that searches its row's part of it (draw_rows; draw_by_wave: the sums of a row's quads).
#ifndef DGS_CSRC_CHOOSE_H_
#define DGS_CSRC_CHOOSE_H_

#include <type_traits>

#include "race.h"

namespace dgs {

// positions that are ranked by counting (64: the same batch 277 us for 274; 21 k rows of 100, 64 picks 172 for 146)
constexpr uint32_t kShortRow = 128;
constexpr uint32_t kOutOfRace = 0xffffffffu;     // key bits of no position
constexpr uint32_t kLeastKey = 0x01000000u;      // 2^-125; below it: positions of infinite weights, in their order
constexpr uint32_t kLargestKey = 0x7e000000u;    // 2^125
constexpr uint32_t kUnusableKey = 0x7e800000u;   // from here on: positions of weights that are not > 0, in their order
constexpr float kSureRatio = 1.0f + 0x1p-19f;

// -ln((x + 0.5) / 2^32) to 2.9e-7 of its value (all 2^32 words tried).  Below u = 1/2 by the hardware logarithm, above by
// 2 atanh(v / (2 - v)) of v = 1 - u, which the integer gives exactly.
__device__ __forceinline__ float approx_neg_log_u32(uint32_t x) {
  const float u = (float(x) + 0.5f) * 0x1p-32f;
  const float low = -0.693147181f * __builtin_amdgcn_logf(u);  // (a base-2 logarithm)
  const float v = (float(~x) + 0.5f) * 0x1p-32f;
  const float t = v * __builtin_amdgcn_rcpf(2.0f - v);  // at most 1/3 where it is used
  const float z = t * t;
  float p = 0.0769230769f;
  p = __builtin_fmaf(p, z, 0.0909090909f);
  p = __builtin_fmaf(p, z, 0.111111111f);
  p = __builtin_fmaf(p, z, 0.142857143f);
  p = __builtin_fmaf(p, z, 0.2f);
  p = __builtin_fmaf(p, z, 0.333333333f);
  const float high = 2.0f * __builtin_fmaf(p * z, t, t);
  return x & 0x80000000u ? high : low;
}

// Race keys are the bits of positive floats (they order like the values).  A plain weight has its key by one
// reciprocal.  The others have keys too: one that leaves the range from kLeastKey to kLargestKey is set to
// the end that it left by, which surely_less orders against the keys inside as it orders the true one, and leaves
// open against its like.
__device__ __forceinline__ bool plain_weight(float w) { return w >= 0x1p-120f && w <= 0x1p90f; }
__device__ __forceinline__ uint32_t uncommon_key(float e, float w, uint32_t p) {
  const uint32_t in_order = p < 0xfffffeu ? p : 0xfffffeu;
  if (!(w > 0.0f)) return kUnusableKey + in_order;
  if (w > 3.4028234663852886e38f) return 1u + in_order;  // (the 64-bit keys are all 0)
  const float scale = w < 1.0f ? 0x1p64f : 0x1p-64f;     // the reciprocal is of a number far from either end
  const float key = e * __builtin_amdgcn_rcpf(w * scale) * scale;
  return __float_as_uint(fminf(fmaxf(key, __uint_as_float(kLeastKey)), __uint_as_float(kLargestKey)));
}

// Whether the 64-bit key behind `a` is smaller than the one behind `b` for sure.
__device__ __forceinline__ bool surely_less(uint32_t a, uint32_t b) {
  return __uint_as_float(b) > __uint_as_float(a) * kSureRatio || ((a >= kUnusableKey || a < kLeastKey) && b > a);
}

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Weights of positions [p, p + 4) of the row of `deg` positions that begins at edge `begin`; 0 beyond it.
typedef float float4_anywhere __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ float4_anywhere weight_quad(const TierView<float>& probs, int64_t begin, uint32_t p, uint32_t deg) {
  const int64_t at = begin + int64_t(p);
  if (p < deg && deg - p >= 4u && at + 4 <= probs.thr) return *reinterpret_cast<const float4_anywhere*>(probs.dev + at);
  float4_anywhere w = float4_anywhere(0.0f);
#pragma unroll
  for (int c = 0; c < 4; ++c)
    if (p < deg && deg - p > uint32_t(c)) w[c] = probs.at(at + c);
  return w;
}

// Approximate keys of positions [p, p + 4) (p a multiple of 4) of a row, of weights w (0 beyond it); kOutOfRace
// beyond it.
__device__ __forceinline__ uint4 approx_key_quad(float4_anywhere w, uint32_t p, uint32_t deg, uint64_t rng_seed,
                                                 uint32_t rng_stream, int64_t row) {
  const PhiloxWords x = philox4x32_10(0x80000000u | (p >> 2), rng_stream, uint32_t(uint64_t(row)),
                                      uint32_t(uint64_t(row) >> 32), uint32_t(rng_seed), uint32_t(rng_seed >> 32));
  float e[4];  // 2^-33 to 23
  uint32_t key[4];
  bool plain = true;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    e[c] = approx_neg_log_u32(x.w[c]);
    key[c] = __float_as_uint(e[c] * __builtin_amdgcn_rcpf(w[c]));
    plain &= plain_weight(w[c]);
  }
  if (!plain) {  // (one branch for all four, and for positions beyond the row: a branch for each is 5 % of a long row's time)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (!(p < deg && deg - p > uint32_t(c))) key[c] = kOutOfRace;
      else if (!plain_weight(w[c])) key[c] = uncommon_key(e[c], w[c], p + c);
    }
  }
  return make_uint4(key[0], key[1], key[2], key[3]);
}

// ---- a row raced by one wave ----

constexpr int kHeldQuads = 4;   // stretches whose weights are requested at a time
constexpr int kListRoom = 192;
constexpr int kListSlack = 16;  // a lowered bar keeps num_picks to num_picks + kListSlack entries
struct WaveList {
  uint32_t key[kListRoom + 4];  // (whole quads are read)
  uint32_t pos[kListRoom + 4];
};

// Every position that has not been entered into the list, or has been taken out again, is at or above
// `bar`; `dropped` is the lane's smallest key among them.  (A bar taken over from another wave may lie
// below some entries.)
struct ListRace {
  int n = 0;
  uint32_t bar = kOutOfRace;
  uint32_t dropped = kOutOfRace;
  bool open = false;  // only 64-bit keys of the whole row settle it
};

// Lowers the bar so that num_picks to num_picks + kListSlack entries stay.  (Equal keys may make that
// impossible: the race is left open then.)
__device__ __forceinline__ void list_tighten(WaveList& list, ListRace& r, int k) {
  constexpr int kEach = kListRoom / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  wave_lds_fence();
  uint32_t key[kEach], pos[kEach];
#pragma unroll
  for (int u = 0; u < kEach; ++u) {
    const int e = u * kWave + lane;
    key[u] = e < r.n ? list.key[e] : kOutOfRace;
    pos[u] = e < r.n ? list.pos[e] : kNoPos;
  }
  uint32_t lo = 0, hi = r.bar - 1;  // fewer than k entries are at or below lo (0 is no key)
  int kept = 0;
#pragma unroll
  for (int u = 0; u < kEach; ++u) kept += __builtin_popcountll(__ballot(key[u] <= hi));
  while (kept > k + kListSlack && hi - lo > 1) {
    const uint32_t mid = lo + ((hi - lo) >> 1);
    int c = 0;
#pragma unroll
    for (int u = 0; u < kEach; ++u) c += __builtin_popcountll(__ballot(key[u] <= mid));
    if (c < k) {
      lo = mid;
    } else {
      hi = mid;
      kept = c;
    }
  }
  const bool stuck = kept > k + kListSlack;
  r.open |= stuck;
  wave_lds_fence();
  int at = 0;
#pragma unroll
  for (int u = 0; u < kEach; ++u) {
    const bool stays = key[u] <= hi && (!stuck || at + lane < k);
    const uint64_t who = __ballot(stays);
    if (stays) {
      const int to = at + __builtin_popcountll(who & ((uint64_t(1) << lane) - 1));
      list.key[to] = key[u];
      list.pos[to] = pos[u];
    } else if (key[u] < r.dropped) {
      r.dropped = key[u];
    }
    at += __builtin_popcountll(who);
  }
  r.n = at;
  r.bar = hi + 1;
  wave_lds_fence();
}

// One candidate per lane (kOutOfRace: none).
__device__ __forceinline__ void list_enter(WaveList& list, ListRace& r, uint32_t key, uint32_t pos, int k) {
  if (r.n > kListRoom - kWave) list_tighten(list, r, k);
  const int lane = threadIdx.x & (kWave - 1);
  const bool in = key < r.bar;
  const uint64_t who = __ballot(in);
  if (in) {
    const int to = r.n + __builtin_popcountll(who & ((uint64_t(1) << lane) - 1));
    list.key[to] = key;
    list.pos[to] = pos;
  } else if (key < r.dropped) {
    r.dropped = key;
  }
  r.n += __builtin_popcountll(who);
}

__device__ __forceinline__ void list_enter_quad(WaveList& list, ListRace& r, uint4 key, uint32_t pos, int k) {
  list_enter(list, r, key.x, pos, k);
  list_enter(list, r, key.y, pos + 1, k);
  list_enter(list, r, key.z, pos + 2, k);
  list_enter(list, r, key.w, pos + 3, k);
}

__device__ __forceinline__ uint32_t wave_min(uint32_t v) {
#pragma unroll
  for (int d = kWave / 2; d > 0; d >>= 1) {
    const uint32_t o = lane_xor(v, d);
    v = o < v ? o : v;
  }
  return v;
}

// The picks in order: entry_pos[0 .. k), with entry_key[0 .. k] for scratch.  The row has more than k
// positions.  Returns false (in every lane) if 64-bit keys of the whole row have to settle it: otherwise an
// unsure order is settled by the 64-bit keys of the entries, which are all that could be picked.
__device__ __forceinline__ bool list_finish(WaveList& list, ListRace& r, int k, uint32_t* entry_key, uint32_t* entry_pos,
                                            const TierView<float>& probs, int64_t begin, uint64_t rng_seed,
                                            uint32_t rng_stream, int64_t row) {
  const int lane = threadIdx.x & (kWave - 1);
  if (r.n > 2 * kWave) list_tighten(list, r, k);
  if (lane < 4) list.key[r.n + lane] = kOutOfRace;
  for (int e = lane; e <= k; e += kWave) entry_key[e] = 0;  // stays where two keys share a rank: unsure
  const uint32_t next = wave_min(r.dropped);
  wave_lds_fence();
  uint32_t key[2], pos[2];
  int rank[2] = {0, 0};
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int e = u * kWave + lane;
    key[u] = e < r.n ? list.key[e] : kOutOfRace;
    pos[u] = e < r.n ? list.pos[e] : kNoPos;
  }
  for (int j = 0; j < r.n; j += 4) {
    const uint4 o = *reinterpret_cast<const uint4*>(&list.key[j]);
#pragma unroll
    for (int u = 0; u < 2; ++u)
      rank[u] += int(o.x < key[u]) + int(o.y < key[u]) + int(o.z < key[u]) + int(o.w < key[u]);
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    if (key[u] != kOutOfRace && rank[u] <= k) {
      entry_key[rank[u]] = key[u];
      entry_pos[rank[u]] = pos[u];
    }
  }
  wave_lds_fence();
  if (lane == 0 && (r.n <= k || next < entry_key[k])) entry_key[k] = next;
  wave_lds_fence();
  const bool unsure = lane < k && !surely_less(entry_key[lane], entry_key[lane + 1]);
  if (__ballot(r.open) != 0) return false;
  if (__ballot(unsure) == 0) return true;
  const uint32_t last = entry_key[k - 1];
  if (last == 0 || !surely_less(last, next)) return false;
  uint64_t exact[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    exact[u] = kNoKey;
    rank[u] = 0;
    if (pos[u] == kNoPos) continue;
    const PhiloxWords x = philox4x32_10(0x80000000u | (pos[u] >> 2), rng_stream, uint32_t(uint64_t(row)),
                                        uint32_t(uint64_t(row) >> 32), uint32_t(rng_seed), uint32_t(rng_seed >> 32));
    const uint32_t word = pos[u] & 2 ? (pos[u] & 1 ? x.w[3] : x.w[2]) : (pos[u] & 1 ? x.w[1] : x.w[0]);
    exact[u] = race_key(word, probs.at(begin + int64_t(pos[u])), pos[u]);
  }
#pragma unroll
  for (int v = 0; v < 2; ++v) {
    for (int j = 0; j < kWave && v * kWave + j < r.n; ++j) {
      const uint64_t ok = lane_read(exact[v], j);
      const uint32_t op = lane_read(pos[v], j);
#pragma unroll
      for (int u = 0; u < 2; ++u) rank[u] += race_less(ok, op, exact[u], pos[u]);
    }
  }
#pragma unroll
  for (int u = 0; u < 2; ++u)
    if (pos[u] != kNoPos && rank[u] < k) entry_pos[rank[u]] = pos[u];
  wave_lds_fence();
  return true;
}

// A row of up to kShortRow positions: every position counts the smaller ones.  Returns as list_finish does.
__device__ __forceinline__ bool race_short(uint32_t* keys, uint32_t* entry_key, uint32_t* entry_pos, int k,
                                           const TierView<float>& probs, int64_t begin, uint32_t deg, uint64_t rng_seed,
                                           uint32_t rng_stream, int64_t row) {
  static_assert(kShortRow == 2 * kWave, "two positions to a lane at most");
  const uint32_t lane = threadIdx.x & (kWave - 1);
  if (4 * lane < deg)
    *reinterpret_cast<uint4*>(&keys[4 * lane]) =
        approx_key_quad(weight_quad(probs, begin, 4 * lane, deg), 4 * lane, deg, rng_seed, rng_stream, row);
  for (int e = int(lane); e <= k; e += kWave) entry_key[e] = 0;  // stays where two keys share a rank: unsure
  wave_lds_fence();
  const auto enter = [&](uint32_t key, int rank, uint32_t pos) {
    if (key == kOutOfRace || rank > k) return;
    entry_key[rank] = key;
    entry_pos[rank] = pos;
  };
  const uint32_t own = lane < deg ? keys[lane] : kOutOfRace;
  int rank = 0;
  if (deg <= kWave) {
#pragma unroll 4
    for (uint32_t j = 0; j < deg; j += 4) {
      const uint4 o = *reinterpret_cast<const uint4*>(&keys[j]);
      rank += int(o.x < own) + int(o.y < own) + int(o.z < own) + int(o.w < own);
    }
  } else {
    const uint32_t own1 = lane + kWave < deg ? keys[lane + kWave] : kOutOfRace;
    int rank1 = 0;
#pragma unroll 4
    for (uint32_t j = 0; j < deg; j += 4) {
      const uint4 o = *reinterpret_cast<const uint4*>(&keys[j]);
      rank += int(o.x < own) + int(o.y < own) + int(o.z < own) + int(o.w < own);
      rank1 += int(o.x < own1) + int(o.y < own1) + int(o.z < own1) + int(o.w < own1);
    }
    enter(own1, rank1, lane + kWave);
  }
  enter(own, rank, lane);
  wave_lds_fence();
  return __ballot(int(lane) < k && !surely_less(entry_key[lane], entry_key[lane + 1])) == 0;
}

// A row of more than k positions by one wave: its picks in order into entry_pos[0 .. k] (the last one for
// scratch, and entry_key[0 .. k]).  `floats`: not raced on them before.
template <bool SHORT>
__device__ __forceinline__ void race_by_wave(WaveList& list, uint32_t* entry_key, uint32_t* entry_pos, bool floats, int k,
                                             const TierView<float>& probs, int64_t begin, uint32_t deg, uint64_t rng_seed,
                                             uint32_t rng_stream, int64_t row) {
  const int lane = threadIdx.x & (kWave - 1);
  bool settled = false;
  if (SHORT && deg <= kShortRow) {
    settled = race_short(list.key, entry_key, entry_pos, k, probs, begin, deg, rng_seed, rng_stream, row);
  } else if (floats) {
    ListRace race;
    constexpr uint32_t kStretch = 4 * kWave;
    for (uint32_t p0 = 0; p0 < deg; p0 += kHeldQuads * kStretch) {
      float4_anywhere held[kHeldQuads];
#pragma unroll
      for (int u = 0; u < kHeldQuads; ++u) held[u] = weight_quad(probs, begin, p0 + u * kStretch + 4u * uint32_t(lane), deg);
#pragma unroll
      for (int u = 0; u < kHeldQuads; ++u) {
        if (p0 + u * kStretch >= deg) break;
        const uint32_t p = p0 + u * kStretch + 4u * uint32_t(lane);
        list_enter_quad(list, race, approx_key_quad(held[u], p, deg, rng_seed, rng_stream, row), p, k);
      }
    }
    settled = list_finish(list, race, k, entry_key, entry_pos, probs, begin, rng_seed, rng_stream, row);
  }
  if (!settled) {
    const Group<kWave> g;
    const uint32_t pos = race_row<kWave>(g, probs, begin, deg, k, rng_seed, rng_stream, row);
    if (lane < k) entry_pos[lane] = pos;
  }
  wave_lds_fence();
}

// ---- many rows raced by one block ----

constexpr int kChooseRows = 32;       // rows of a block at most ...
constexpr int kChooseEntries = 1056;  // ... and rows * (num_picks + 1)
inline int choose_rows(int64_t k) { return k <= 32 ? kChooseRows : kChooseRows / 2; }

template <int NT>
struct RaceRowsLds {
  int64_t begin[kChooseRows];   // first edge, seed id and degree of every row
  int64_t row[kChooseRows];
  uint32_t deg[kChooseRows];    // (0: not raced here)
  int quad0[kChooseRows + 1];   // short rows: first quad of the row's positions
  uint32_t open[kChooseRows];   // the row is on the list already
  int listed[kChooseRows];      // rows that a wave takes
  int n_listed, next;
  uint32_t entry_key[kChooseEntries];  // row r's from r * (k + 1) on
  uint32_t entry_pos[kChooseEntries];
  union __align__(16) {
    uint32_t key[kChooseRows * kShortRow];
    WaveList list[NT / kWave];
  };
};

// The row whose quads quad `q` is among.
__device__ __forceinline__ int row_of_quad(const int (&quad0)[kChooseRows + 1], int q) {
  int r = 0;
#pragma unroll
  for (int step = kChooseRows / 2; step > 0; step >>= 1)
    if (quad0[r + step] <= q) r += step;
  return r;
}

// quad0[] of the rows' quads, one wave's work (`quads`: those of the lane's row).
__device__ __forceinline__ void scan_quads(int (&quad0)[kChooseRows + 1], int quads) {
  const int lane = threadIdx.x & (kWave - 1);
  int upto = lane < kChooseRows ? quads : 0;
#pragma unroll
  for (int d = 1; d < kChooseRows; d <<= 1) {
    const int t = __shfl_up(upto, d, kWave);
    if (lane >= d) upto += t;
  }
  if (lane < kChooseRows) quad0[lane + 1] = upto;
  if (lane == 0) quad0[0] = 0;
}

// What race_rows and draw_rows begin with, in two halves in front of one barrier: the first wave's, whose
// lanes bring a row each, and the whole block's.
template <int NT>
__device__ __forceinline__ void set_row(RaceRowsLds<NT>& lds, int64_t begin, int64_t row, uint32_t deg) {
  const int lane = threadIdx.x;
  if (lane < kChooseRows) {
    lds.begin[lane] = begin;
    lds.row[lane] = row;
    lds.deg[lane] = deg;
    lds.open[lane] = 0;
  }
  scan_quads(lds.quad0, deg <= kShortRow ? int(deg + 3) / 4 : 0);
  const uint64_t who = __ballot(deg > kShortRow);
  if (deg > kShortRow) lds.listed[__builtin_popcountll(who & ((uint64_t(1) << lane) - 1))] = lane;
  if (lane == 0) {
    lds.n_listed = __builtin_popcountll(who);
    lds.next = 0;
  }
}
template <int NT>
__device__ __forceinline__ void clear_entries(RaceRowsLds<NT>& lds, int rows, int k) {
  for (int e = threadIdx.x; e < rows * (k + 1); e += NT) lds.entry_key[e] = 0;
}

// Called by the whole block behind that barrier.  Afterwards (behind another) entry_pos holds the picks of
// every row with deg > 0, which are rows of more than k positions.
template <int NT>
__device__ __forceinline__ void race_rows(RaceRowsLds<NT>& lds, int rows, int k, const TierView<float>& probs,
                                          uint64_t rng_seed, uint32_t rng_stream) {
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int each = k + 1;
  const int quads = lds.quad0[kChooseRows];
  for (int q = threadIdx.x; q < quads; q += NT) {
    const int r = row_of_quad(lds.quad0, q);
    const uint32_t p = 4u * uint32_t(q - lds.quad0[r]), deg = lds.deg[r];
    const uint4 key = approx_key_quad(weight_quad(probs, lds.begin[r], p, deg), p, deg, rng_seed, rng_stream, lds.row[r]);
    *reinterpret_cast<uint4*>(&lds.key[4 * q]) = key;
  }
  __syncthreads();
  // A position counts the smaller ones of its row; where the block has threads for all positions, each by
  // itself, else four to a thread, which reads every other quad once for all of them.
  const auto enter = [&](int r, uint32_t key, int rank, int pos) {
    if (key == kOutOfRace || rank > k) return;
    lds.entry_key[r * each + rank] = key;
    lds.entry_pos[r * each + rank] = uint32_t(pos);
  };
  if (4 * quads <= NT) {
    const int e = threadIdx.x;
    if (e < 4 * quads) {
      const int r = row_of_quad(lds.quad0, e >> 2);
      const int q0 = lds.quad0[r], q1 = lds.quad0[r + 1];
      const uint32_t own = lds.key[e];
      int rank = 0;
#pragma unroll 4
      for (int j = q0; j < q1; ++j) {
        const uint4 o = *reinterpret_cast<const uint4*>(&lds.key[4 * j]);
        rank += int(o.x < own) + int(o.y < own) + int(o.z < own) + int(o.w < own);
      }
      enter(r, own, rank, e - 4 * q0);
    }
  } else {
    for (int q = threadIdx.x; q < quads; q += NT) {
      const int r = row_of_quad(lds.quad0, q);
      const uint4 mine = *reinterpret_cast<const uint4*>(&lds.key[4 * q]);
      const uint32_t own[4] = {mine.x, mine.y, mine.z, mine.w};
      int rank[4] = {0, 0, 0, 0};
      const int q0 = lds.quad0[r], q1 = lds.quad0[r + 1];
#pragma unroll 2
      for (int j = q0; j < q1; ++j) {
        const uint4 o = *reinterpret_cast<const uint4*>(&lds.key[4 * j]);
#pragma unroll
        for (int c = 0; c < 4; ++c) rank[c] += int(o.x < own[c]) + int(o.y < own[c]) + int(o.z < own[c]) + int(o.w < own[c]);
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) enter(r, own[c], rank[c], 4 * (q - q0) + c);
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < rows * each; e += NT) {
    const int r = e / each;
    const uint32_t deg = lds.deg[r];
    if (deg == 0 || deg > kShortRow || e - r * each == k) continue;
    if (!surely_less(lds.entry_key[e], lds.entry_key[e + 1]) && atomicExch(&lds.open[r], 1u) == 0u)
      lds.listed[atomicAdd(&lds.n_listed, 1)] = r;
  }
  __syncthreads();
  if (lds.n_listed == 0) return;
  for (;;) {
    int t = 0;
    if (lane == 0) t = atomicAdd(&lds.next, 1);
    t = int(wave_uniform(uint32_t(t)));
    if (t >= lds.n_listed) break;
    const int r = int(wave_uniform(uint32_t(lds.listed[t])));
    const int64_t begin = wave_uniform(lds.begin[r]), row = wave_uniform(lds.row[r]);
    const uint32_t deg = wave_uniform(lds.deg[r]);
    race_by_wave<false>(lds.list[wave], lds.entry_key + r * each, lds.entry_pos + r * each, deg > kShortRow, k, probs, begin, deg, rng_seed,
                 rng_stream, row);
  }
  __syncthreads();
}

// A long row raced by a whole block of NT threads (every thread must call it): returns, in lane l < k of
// wave 0, the position of the l-th winner.  Every wave races an interleaved share; the lowest bar that any
// of them has reached holds for all, and wave 0 enters what the others kept into its list.
template <int NT>
struct RaceLongLds {
  union __align__(16) {
    WaveList list[NT / kWave];
    FullRaceLds<NT> full;
  };
  int kept[NT / kWave];
  uint32_t entry_key[kMaxWeightedPicks + 1];
  uint32_t entry_pos[kMaxWeightedPicks + 1];
  uint32_t bar, dropped;
  int open;
};

template <int NT>
__device__ __forceinline__ uint32_t race_long(RaceLongLds<NT>& lds, const TierView<float>& probs, int64_t begin, uint32_t deg,
                                              int k, uint64_t rng_seed, uint32_t rng_stream, int64_t row) {
  constexpr int kWaves = NT / kWave;
  constexpr int kHeld = NT == kLongBlock ? 5 : kHeldQuads;  // (rows of up to 20480 positions in one go)
  constexpr uint64_t kStretch = 4 * kWave;
  const int lane = threadIdx.x & (kWave - 1), wave = int(wave_uniform(uint32_t(threadIdx.x / kWave)));
  if (threadIdx.x == 0) {
    lds.bar = lds.dropped = kOutOfRace;
    lds.open = 0;
  }
  __syncthreads();
  WaveList& list = lds.list[wave];
  ListRace race;
  for (uint64_t p0 = kStretch * uint32_t(wave); p0 < deg; p0 += kStretch * kWaves * kHeld) {
    const auto quad_begin = [&](int u) {  // (a position that does not exist where the row has none there)
      const uint64_t p = p0 + uint64_t(u) * kStretch * kWaves + 4u * uint32_t(lane);
      return p < deg ? uint32_t(p) : deg;
    };
    float4_anywhere held[kHeld];
#pragma unroll
    for (int u = 0; u < kHeld; ++u) held[u] = weight_quad(probs, begin, quad_begin(u), deg);
#pragma unroll
    for (int u = 0; u < kHeld; ++u) {
      if (p0 + uint64_t(u) * kStretch * kWaves >= deg) break;
      const uint32_t published = wave_uniform(__atomic_load_n(&lds.bar, __ATOMIC_RELAXED));
      if (published < race.bar) race.bar = published;  // (entries at or above it do no harm)
      const uint32_t before = race.bar, p = quad_begin(u);
      list_enter_quad(list, race, approx_key_quad(held[u], p, deg, rng_seed, rng_stream, row), p, k);
      if (race.bar < before && lane == 0) atomicMin(&lds.bar, race.bar);
    }
  }
  if (wave != 0 && race.n > k + kListSlack) {
    list_tighten(list, race, k);
    if (lane == 0) atomicMin(&lds.bar, race.bar);
  }
  const uint32_t least = wave_min(race.dropped);
  if (lane == 0) {
    if (wave != 0) atomicMin(&lds.dropped, least);
    lds.kept[wave] = race.n;
  }
  if (race.open && lane == 0) lds.open = 1;  // (the same in every lane)
  __syncthreads();
  uint32_t pos = kNoPos;
  if (wave == 0) {
    if (lds.dropped < race.dropped) race.dropped = lds.dropped;
    if (lds.bar < race.bar) race.bar = lds.bar;
    race.open |= lds.open != 0;
    // (a lane for every entry of the others: 64 at a time, and not one list after the other)
    int upto = lane > 0 && lane < kWaves ? lds.kept[lane] : 0;
#pragma unroll
    for (int d = 1; d < kWaves; d <<= 1) {
      const int o = __shfl_up(upto, d, kWave);
      if (lane >= d) upto += o;
    }
    const int total = int(lane_read(uint32_t(upto), kWaves - 1));
    for (int e0 = 0; e0 < total; e0 += kWave) {
      const int e = e0 + lane;
      int w = 1, from = 0;
#pragma unroll
      for (int v = 1; v < kWaves - 1; ++v) {
        const int end = int(lane_read(uint32_t(upto), v));
        if (e >= end) {
          w = v + 1;
          from = end;
        }
      }
      list_enter(list, race, e < total ? lds.list[w].key[e - from] : kOutOfRace, e < total ? lds.list[w].pos[e - from] : kNoPos, k);
    }
    if (list_finish(list, race, k, lds.entry_key, lds.entry_pos, probs, begin, rng_seed, rng_stream, row)) {
      if (lane < k) pos = lds.entry_pos[lane];
    } else if (lane == 0) {
      lds.open = 1;
    }
  }
  __syncthreads();
  if (lds.open != 0) {
    Race full;
    race_long_row_full<NT>(full, lds.full, probs, begin, deg, k, rng_seed, rng_stream, row);
    pos = wave == 0 ? full.pos : kNoPos;
  }
  __syncthreads();  // lds is reused by the block's next row
  return pos;
}

// ---- draws with replacement ----

// Quads of positions whose sums LDS holds at a time: no fewer than a row has here.  (16 384 rows of 1000
// neighbours, 10 draws each, us a call: 512 quads for a block of 256 threads 153, 1024 133.)
constexpr int kDrawQuads = 1024;
constexpr uint32_t kDrawRow = 4 * kDrawQuads;

template <int NT>
struct DrawRowsLds {
  int64_t begin[kChooseRows];   // as in RaceRowsLds; at most kDrawRow positions a row
  int64_t row[kChooseRows];
  uint32_t deg[kChooseRows];
  int quad0[kChooseRows + 1];
  uint32_t max[kChooseRows];    // largest weight, as the bits of a float
  uint64_t part[NT / kWave];
  uint64_t running[4 * kDrawQuads];  // shares up to and including a position, over the rows of a pass
};

__device__ __forceinline__ float quad_max(float4_anywhere w) {
  float m = 0.0f;
#pragma unroll
  for (int c = 0; c < 4; ++c) m = w[c] > m ? w[c] : m;
  return m;
}

template <int NT>
__device__ __forceinline__ void set_row(DrawRowsLds<NT>& lds, int64_t begin, int64_t row, uint32_t deg) {
  const int lane = threadIdx.x;
  if (lane < kChooseRows) {
    lds.begin[lane] = begin;
    lds.row[lane] = row;
    lds.deg[lane] = deg;
    lds.max[lane] = 0;
  }
  scan_quads(lds.quad0, int((deg + 3) / 4));
}
template <int NT>
__device__ __forceinline__ void clear_entries(DrawRowsLds<NT>&, int, int) {}

// Called by the whole block behind the barrier.  emit(r, j, position) is called for every draw j of every
// row with deg > 0, by some thread.  A row without a positive share keeps its last neighbour.
template <int NT, typename Emit>
__device__ __forceinline__ void draw_rows(DrawRowsLds<NT>& lds, int rows, int k, const TierView<float>& probs,
                                          uint64_t rng_seed, uint32_t rng_stream, Emit emit) {
  constexpr int kEach = kDrawQuads / NT;
  const int lane = threadIdx.x & (kWave - 1);
  for (int r0 = 0; r0 < rows;) {
    const int q0 = lds.quad0[r0];
    const bool fits = lane >= r0 && lane < rows && lds.quad0[lane + 1] - q0 <= kDrawQuads;
    const int r1 = r0 + __builtin_popcountll(__ballot(fits));  // one row always fits
    const int quads = lds.quad0[r1] - q0;
    float4_anywhere w[kEach];
    int row[kEach];
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
      const int q = i * NT + int(threadIdx.x);
      row[i] = row_of_quad(lds.quad0, q0 + q);
      w[i] = float4_anywhere(0.0f);
      if (q < quads) {
        w[i] = weight_quad(probs, lds.begin[row[i]], 4u * uint32_t(q0 + q - lds.quad0[row[i]]), lds.deg[row[i]]);
        const float m = quad_max(w[i]);
        if (m > 0.0f) atomicMax(&lds.max[row[i]], __float_as_uint(m));
      }
    }
    __syncthreads();
    uint64_t before = 0;
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
      if (i * NT >= quads) break;  // (the same for every thread)
      const int q = i * NT + int(threadIdx.x);
      const QuantumScale scale = quantum_scale(__uint_as_float(q < quads ? lds.max[row[i]] : 0u));
      uint64_t upto[4], sum = 0;
#pragma unroll
      for (int c = 0; c < 4; ++c) upto[c] = sum += weight_quantum(w[i][c], scale);
      uint64_t total;
      const uint64_t at = before + block_exclusive_scan<NT, uint64_t>(sum, &total, lds.part);
      if (q < quads) {
#pragma unroll
        for (int c = 0; c < 4; ++c) lds.running[4 * q + c] = at + upto[c];
      }
      before += total;
    }
    __syncthreads();
    int r = r0 + int(threadIdx.x) / k, j = int(threadIdx.x) % k;
    while (r < r1) {
      const int deg = int(lds.deg[r]);
      if (deg > 0) {
        const uint64_t* running = lds.running + 4 * (lds.quad0[r] - q0);
        const uint64_t base = lds.quad0[r] > q0 ? running[-1] : 0;
        const uint64_t total = running[deg - 1] - base;
        int lo = deg - 1;
        if (total > 0) {
          const uint64_t want = base + philox_bounded64(rng_seed, rng_stream, lds.row[r], uint32_t(j), total);
          int hi = deg - 1;  // the first position whose sum is beyond it
          for (lo = 0; lo < hi;) {
            const int mid = (lo + hi) >> 1;
            if (running[mid] > want) hi = mid; else lo = mid + 1;
          }
        }
        emit(r, j, uint32_t(lo));
      }
      r += NT / k;
      j += NT % k;
      if (j >= k) {
        j -= k;
        ++r;
      }
    }
    __syncthreads();
    r0 = r1;
  }
}

// A row of up to kWaveDrawRow positions drawn from by one wave: lane j < k returns the position of draw j (k at
// most 64).
constexpr int kWaveDrawQuads = 8;  // quads a lane holds
constexpr uint32_t kWaveDrawRow = 4 * kWave * kWaveDrawQuads;
struct WaveDrawLds {
  uint64_t upto[kWave * kWaveDrawQuads];  // shares up to and including a quad
};
__device__ __forceinline__ uint32_t draw_by_wave(WaveDrawLds& lds, const TierView<float>& probs, int64_t begin, uint32_t deg, int k,
                                                 uint64_t rng_seed, uint32_t rng_stream, int64_t row) {
  constexpr uint32_t kStretch = 4 * kWave;
  const int lane = threadIdx.x & (kWave - 1);
  float4_anywhere w[kWaveDrawQuads];
  float most = 0.0f;
#pragma unroll
  for (int u = 0; u < kWaveDrawQuads; ++u) w[u] = weight_quad(probs, begin, u * kStretch + 4u * uint32_t(lane), deg);
#pragma unroll
  for (int u = 0; u < kWaveDrawQuads; ++u) {
    if (u * kStretch >= deg) break;
    const float m = quad_max(w[u]);
    most = m > most ? m : most;
  }
  const QuantumScale scale = quantum_scale(__uint_as_float(~wave_min(~__float_as_uint(most))));
  uint64_t total = 0;
#pragma unroll
  for (int u = 0; u < kWaveDrawQuads; ++u) {
    if (u * kStretch >= deg) break;
    uint64_t sum = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) sum += weight_quantum(w[u][c], scale);
    const uint64_t upto = total + group_inclusive_sum<kWave>(sum, lane);
    lds.upto[u * kWave + lane] = upto;
    total = lane_read(upto, kWave - 1);
  }
  wave_lds_fence();
  uint32_t pos = deg - 1;  // where the row has no positive share
  if (lane < k && total > 0) {
    const uint64_t want = philox_bounded64(rng_seed, rng_stream, row, uint32_t(lane), total);
    uint32_t lo = 0, hi = (deg - 1) >> 2;  // the first quad whose sum is beyond it
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if (lds.upto[mid] > want) hi = mid; else lo = mid + 1;
    }
    uint64_t s = lo > 0 ? lds.upto[lo - 1] : 0;
    const float4_anywhere quad = weight_quad(probs, begin, 4 * lo, deg);  // (still in a cache)
    pos = 4 * lo;
    bool beyond = false;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      s += weight_quantum(quad[c], scale);
      beyond |= s > want;
      if (!beyond) ++pos;
    }
  }
  wave_lds_fence();
  return pos;
}

// A long row drawn from by a whole block of NT threads (every thread must call it): every wave owns a
// contiguous part of it, read once as far as kHeld quads a lane go, and settles the draws that fall into
// its own part.  What is beyond is read in three passes, bound by the wait for memory: several stretches ahead
// (16 384 rows, 8 of them of 10^6 positions, 10 draws, us a call: one stretch at a time 1593; four ahead in
// every pass 1117, eight in the two sums and four in the search, whose registers eight would not fit, 1057; 64
// rows of 200 000: 391, 288, 274).  Rows that end soon after the held part gain nothing: 4000 seeds, fanouts [5,10], rows of
// 6000, one stretch at a time 449; eight asked for whether or not they are there 521, those that are there 470.
template <int N> using AheadOf = std::integral_constant<int, N>;
template <int NT>
struct DrawLongLds {
  float max[NT / kWave];
  uint64_t sum[NT / kWave];
};
template <int NT, typename Emit>
__device__ __forceinline__ void draw_long(DrawLongLds<NT>& lds, const TierView<float>& probs, int64_t begin, uint32_t deg,
                                          int k, uint64_t rng_seed, uint32_t rng_stream, int64_t row, Emit emit) {
  constexpr int kWaves = NT / kWave;
  constexpr int kHeld = 5;
  constexpr uint64_t kStretch = 4 * kWave;
  const int lane = threadIdx.x & (kWave - 1), wave = int(wave_uniform(uint32_t(threadIdx.x / kWave)));
  begin = wave_uniform(begin);
  deg = wave_uniform(deg);
  const uint64_t part = ((deg + uint64_t(kWaves) - 1) / kWaves + kStretch - 1) / kStretch * kStretch;
  const uint64_t lo = part * uint32_t(wave) < deg ? part * uint32_t(wave) : deg;
  const uint64_t hi = lo + part < deg ? lo + part : deg;
  const auto quad_at = [&](uint64_t p0) {
    const uint64_t p = p0 + 4u * uint32_t(lane);
    return weight_quad(probs, begin, p < hi ? uint32_t(p) : deg, deg);
  };
  float4_anywhere held[kHeld];
#pragma unroll
  for (int u = 0; u < kHeld; ++u) held[u] = quad_at(lo + u * kStretch);
  const auto every_stretch = [&](auto ahead, auto each) {  // each(p0, quad) returns whether to go on
    constexpr int kAhead = decltype(ahead)::value;
    bool on = true;
#pragma unroll
    for (int u = 0; u < kHeld; ++u)
      if (on && lo + u * kStretch < hi) on = each(lo + u * kStretch, held[u]);
    for (uint64_t p0 = lo + kHeld * kStretch; on && p0 < hi; p0 += kAhead * kStretch) {
      float4_anywhere next[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u)  // (the last stretches are few: none is asked for beyond them)
        next[u] = p0 + u * kStretch < hi ? quad_at(p0 + u * kStretch) : float4_anywhere(0.0f);
#pragma unroll
      for (int u = 0; u < kAhead; ++u)
        if (on && p0 + u * kStretch < hi) on = each(p0 + u * kStretch, next[u]);
    }
  };
  float most = 0.0f;
  every_stretch(AheadOf<8>(), [&](uint64_t, float4_anywhere w) {
    const float m = quad_max(w);
    most = m > most ? m : most;
    return true;
  });
  most = group_max<kWave>(most);
  if (lane == 0) lds.max[wave] = most;
  __syncthreads();
  for (int w = 0; w < kWaves; ++w) most = lds.max[w] > most ? lds.max[w] : most;
  const QuantumScale scale = quantum_scale(most);
  const auto share = [&](float4_anywhere w) {
    uint64_t sum = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) sum += weight_quantum(w[c], scale);
    return sum;
  };
  uint64_t mine = 0;
  every_stretch(AheadOf<8>(), [&](uint64_t, float4_anywhere w) {
    mine += share(w);
    return true;
  });
  mine = group_sum<kWave>(mine);
  if (lane == 0) lds.sum[wave] = mine;
  __syncthreads();
  uint64_t before = 0, total = 0;
  for (int w = 0; w < kWaves; ++w) {
    if (w < wave) before += lds.sum[w];
    total += lds.sum[w];
  }
  for (int first = 0; first < k; first += kWave) {
    const int j = first + lane;
    if (total == 0) {
      if (wave == 0 && j < k) emit(j, deg - 1);
      continue;
    }
    uint64_t want = 0;
    if (j < k) want = philox_bounded64(rng_seed, rng_stream, row, uint32_t(j), total);
    const bool here = j < k && want >= before && want < before + mine;
    uint64_t pending = __ballot(here);
    if (pending == 0) continue;
    uint32_t pick = deg - 1;
    uint64_t at = before;
    every_stretch(AheadOf<4>(), [&](uint64_t p0, float4_anywhere w) {
      const uint64_t sum = share(w);
      const uint64_t upto = at + group_inclusive_sum<kWave>(sum, lane);
      const uint64_t after = lane_read(upto, kWave - 1);
      uint64_t found = pending & __ballot(here && want < after);
      pending &= ~found;
      at = after;
      while (found) {
        const int b = __builtin_ctzll(found);
        found &= found - 1;
        const uint64_t wanted = lane_read(want, b);
        const int src = __builtin_ctzll(__ballot(upto > wanted));  // the lane whose quad it falls into
        uint64_t s = upto - sum;
        uint32_t p = uint32_t(p0) + 4u * uint32_t(lane);
        bool beyond = false;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          s += weight_quantum(w[c], scale);
          beyond |= s > wanted;
          if (!beyond) ++p;
        }
        p = lane_read(p, src);
        if (lane == b) pick = p;
      }
      return pending != 0;
    });
    if (here) emit(j, pick);
  }
  __syncthreads();  // lds is reused by the block's next row
}

}  // namespace dgs
#endif
