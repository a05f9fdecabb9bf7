// First-occurrence unique + relabel of node ids.
//
// A linear-probing table in HBM (table.h: packed 64-bit slots, or id array + value array for
// 8-byte ids that may not fit 32 bits) maps each id to the smallest position at which it occurs.
// The atomic that inserts a position tells whether it is, so far, its id's smallest and which
// position it displaced (marked lost): a position is a "first occurrence" when it was smallest
// at insertion and never lost.  First occurrences are counted, ranked and compacted in input order
// (which is what makes the result independent of the table layout) by one launch whose blocks add
// up the tiles before theirs (lookback.h), and the first occurrence's word becomes the id's rank.
// Every mapping id remembers its slot, so a tensor that is both mapped and relabelled (the picked
// neighbours of the upstream sampler loop) is not probed a second time.
//
// Launches: clear -> insert -> rank -> lookup.  The caller waits for the count that the third one
// leaves, so every launch in front of it is 5 us of a short call.  Long lists of ids below 2^32 - 1 do without the
// table (buckets.h): sort -> first -> rank -> lookup.
#include "buckets.h"
#include "common.h"
#include "lookback.h"
#include "table.h"

#include <algorithm>

namespace dgs {
namespace {

constexpr int kThreads = 256;
// Positions of a rank block: kThreads x kItems (one vector load of words and one of lost marks per
// thread) x GROUPS.  One group up to 1024 tiles, which the look-back reads in one go; four beyond, where the
// line could lie higher.  us a call, one group / four: ids that are mostly new 500 k 74.3 / 76.9, 1.04 M
// 101.4 / 103.0, 1.06 M 103.9 / 105.3, 2 M 149 / 146, 4 M 268 / 251; a tenth of them new 500 k 58.0 / 64.6,
// 1.04 M 76.6 / 81.5, 1.06 M 78.2 / 82.2, 2 M 121 / 121, 4 M 234 / 223.
constexpr int kItems = 4;
constexpr int kGroupIds = kThreads * kItems;
constexpr int kLongGroups = 4;
constexpr int64_t kLongIds = int64_t(1024) * kGroupIds;
inline int rank_groups(int64_t n) { return n <= kLongIds ? 1 : kLongGroups; }
inline int64_t rank_tiles(int64_t n) {
  const int64_t tile = int64_t(kGroupIds) * rank_groups(n);
  return (n + tile - 1) / tile;
}
constexpr uint32_t kFirstBit = 0x80000000u;   // marks a first occurrence in slot[]
constexpr int64_t kMaxMappingIds = int64_t(1) << 30;
// slot[] word of a mapping id the table could not take (the call's results are void then: the
// overflow word is set).  It lies beyond the mask of every table but the largest possible one
// (2^31 slots), where it names a real slot; lookup_kernel checks a word against the mask, and what
// the slot holds against the number of positions, before either is used as an index.
constexpr uint32_t kNoSlot = 0x7fffffffu;

// Element i of the logical concatenation, or of a single array when count == 1.
template <typename IdT>
__device__ __forceinline__ IdT seg_load(const dgs_segments& s, int64_t i) {
  const IdT* p = static_cast<const IdT*>(s.ptr[0]);
  int64_t j = i;
#pragma unroll
  for (int k = 1; k < DGS_MAX_SEGMENTS; ++k) {
    if (k < s.count && i >= s.len[k - 1]) {
      i -= s.len[k - 1];
      p = static_cast<const IdT*>(s.ptr[k]);
      j = i;
    } else {
      i = -1;  // stays negative: no later segment can match
    }
  }
  return p[j];
}

// Table bytes become 0xFF (empty slots), the lost marks and the overflow word 0.
__global__ __launch_bounds__(kThreads) void clear_kernel(uint4* __restrict__ table, int64_t table16,
                                                         uint4* __restrict__ zeros, int64_t zeros16) {
  const int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  if (i < table16) table[i] = make_uint4(~0u, ~0u, ~0u, ~0u);
  else if (i - table16 < zeros16) zeros[i - table16] = make_uint4(0u, 0u, 0u, 0u);
}

// Every mapping id goes into the table with its position; the atomic that does it also tells
// whether the position is (so far) the smallest of its id and which one it displaced, so "first
// occurrence" is later decided from the two streamed arrays slot[] and lost[] without a second
// random read of the table.  An id the table cannot hold sets the overflow word.
template <typename IdT, typename TableT>
__global__ __launch_bounds__(kThreads) void insert_kernel(dgs_segments mapping, int64_t n, TableT table,
                                                          uint32_t* __restrict__ slot, uint8_t* __restrict__ lost,
                                                          int* __restrict__ overflow) {
  const int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  if (i >= n) return;
  const IdT key = seg_load<IdT>(mapping, i);
  if (!table.holds(key)) {
    *overflow = 1;
    slot[i] = kNoSlot;  // no slot, no first bit: the call's results are void, and a lookup through this word gives -1
    return;
  }
  bool first;
  uint32_t met;
  const uint32_t w = table.insert_min(key, uint32_t(i), &first, &met);
  slot[i] = first ? (w | kFirstBit) : w;
  if (first && met != kNoPosition) lost[met] = 1;
}

// First occurrences of one tile of mapping positions: counted, added to what the tiles before hold,
// compacted into unique_out; a first occurrence's word then holds its rank.  The block of the last tile
// leaves counts_dev[0] = number of distinct ids, [1] = 1 if an id did not fit the table (then everything
// else the call wrote is void), mirrored into pinned host memory when the caller gave some.
// The arrays slot[] and lost[] reach to the end of the last tile; what lies beyond n is read and
// written back but never counts.
template <typename IdT, int GROUPS>
__global__ __launch_bounds__(kThreads) void rank_kernel(dgs_segments mapping, int64_t n, uint32_t* __restrict__ slot,
                                                        const uint8_t* __restrict__ lost, tile_state* __restrict__ state,
                                                        int32_t max_polls, const int* __restrict__ overflow,
                                                        IdT* __restrict__ unique_out, int64_t* __restrict__ counts_dev,
                                                        int64_t* __restrict__ counts_host) {
  typedef uint32_t words __attribute__((ext_vector_type(kItems)));
  constexpr int kWaves = kThreads / kWave;
  constexpr int64_t kTileIds = int64_t(kGroupIds) * GROUPS;
  __shared__ LookbackLds<kThreads> look;
  __shared__ int wave_count[GROUPS * kWaves];
  __shared__ int lds[kWaves];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int64_t tile = blockIdx.x;
  const int64_t base = tile * kTileIds + threadIdx.x * kItems;
  const bool last = (tile + 1) * kTileIds >= n;
  const int64_t bad = last ? int64_t(*overflow != 0) : 0;
  words word[GROUPS];
  uint32_t marks[GROUPS];
#pragma unroll
  for (int g = 0; g < GROUPS; ++g) {
    word[g] = *reinterpret_cast<const words*>(slot + base + g * kGroupIds);
    marks[g] = *reinterpret_cast<const uint32_t*>(lost + base + g * kGroupIds);
  }
  uint32_t first[GROUPS];   // bit j: position j of the group's is its id's first
  int lane_before[GROUPS];  // first positions in the lanes below, then in all of the tile before
#pragma unroll
  for (int g = 0; g < GROUPS; ++g) {
    first[g] = 0;
#pragma unroll
    for (int j = 0; j < kItems; ++j)
      if (base + g * kGroupIds + j < n && (word[g][j] & kFirstBit) != 0 && ((marks[g] >> (8 * j)) & 0xffu) == 0) first[g] |= 1u << j;
    const int c = __builtin_popcount(first[g]);  // its bits are summed over the lanes by ballots
    lane_before[g] = 0;
    int sum = 0;
#pragma unroll
    for (int bit = 0; (1 << bit) <= kItems; ++bit) {
      const uint64_t at = __ballot((c >> bit) & 1);
      lane_before[g] += __builtin_popcountll(at & ((uint64_t(1) << lane) - 1)) << bit;
      sum += __builtin_popcountll(at) << bit;
    }
    if (lane == 0) wave_count[g * kWaves + wave] = sum;
  }
  __syncthreads();
  int total = 0;
#pragma unroll
  for (int q = 0; q < GROUPS * kWaves; ++q) {
    if (q % kWaves == wave) lane_before[q / kWaves] += total;
    total += wave_count[q];
  }
  const tile_state before = tile_exclusive_prefix<kThreads, false>(state, tile, tile_word(total), max_polls, look, [&](int64_t t) {
    int c = 0;  // (a tile before this one is full; a word counts the same before and after its block has rewritten it)
    for (int j = 0; j < GROUPS * kItems; ++j) {
      const int64_t p = t * kTileIds + int64_t(j) * kThreads + threadIdx.x;
      c += (slot[p] & kFirstBit) != 0 && lost[p] == 0;
    }
    int sum;
    block_exclusive_scan<kThreads, int>(c, &sum, lds);
    return tile_word(sum);
  });
  const int64_t rank0 = tile_sum_of(before);
  if (last && threadIdx.x == 0) {
    counts_dev[0] = rank0 + total;
    counts_dev[1] = bad;
    if (counts_host) {
      mirror_to_host(counts_host, rank0 + total);
      mirror_to_host(counts_host + 1, bad);
    }
  }
#pragma unroll
  for (int g = 0; g < GROUPS; ++g) {
    const int64_t p = base + g * kGroupIds;
    uint32_t rank = uint32_t(rank0) + uint32_t(lane_before[g]);
    bool changed = false;
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      if ((first[g] >> j) & 1) {
        unique_out[rank] = seg_load<IdT>(mapping, p + j);
        word[g][j] = rank | kFirstBit;
        ++rank;
        changed = true;
      } else if (((marks[g] >> (8 * j)) & 0xffu) != 0) {
        word[g][j] &= ~kFirstBit;
        changed = true;
      }
    }
    if (changed) *reinterpret_cast<words*>(slot + p) = word[g];
  }
}

// Where element i of a segment list lives: its segment and its offset inside it.
__device__ __forceinline__ void seg_locate(const dgs_segments& s, int64_t i, int* seg, int64_t* off) {
  int k = 0;
  while (k + 1 < s.count && i >= s.len[k]) {
    i -= s.len[k];
    ++k;
  }
  *seg = k;
  *off = i;
}

// Mapping positions of the requiring segments that are mapping segments themselves (-1: not one).
struct SegmentAlias {
  int64_t mapping_begin[DGS_MAX_SEGMENTS];
};

// out[j] = rank of requiring[j], -1 when the id is not in the table.  Ranks live in the slot
// words of the first occurrences (a streamed array), the table keeps every id's smallest
// position: an element that is itself a first occurrence of the mapping list needs no random
// read at all, any other one reads the table entry and then that position's word.
// Nothing read from the table or from slot[] is used as an index before it has been checked: a
// slot word must name a slot of the table, and the position a table entry holds must be one of
// the n mapping positions (an entry that was never filled holds 0xffffffff).
template <typename IdT, typename TableT>
__global__ __launch_bounds__(kThreads) void lookup_kernel(dgs_segments requiring, int64_t m, TableT table,
                                                          const uint32_t* __restrict__ slot, int64_t n,
                                                          SegmentAlias alias, dgs_segments out) {
  const int64_t j = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  if (j >= m) return;
  int seg;
  int64_t off;
  seg_locate(requiring, j, &seg, &off);
  uint32_t s;
  bool holds_rank = false;  // s is the word of a first occurrence of the mapping list
  if (alias.mapping_begin[seg] >= 0) {
    s = slot[alias.mapping_begin[seg] + off];
    holds_rank = (s & kFirstBit) != 0;
    s &= ~kFirstBit;
  } else {
    const IdT key = static_cast<const IdT*>(requiring.ptr[seg])[off];
    s = table.holds(key) ? table.find(key) : table.mask + 1;  // an id the table cannot hold is not in it
  }
  IdT rank = IdT(-1);
  if (holds_rank) {
    rank = IdT(s);
  } else if (s <= table.mask) {
    const uint32_t first_at = table.value(s);  // smallest mapping position of the id
    if (int64_t(first_at) < n) rank = IdT(slot[first_at] & ~kFirstBit);
  }
  static_cast<IdT*>(const_cast<void*>(out.ptr[seg]))[off] = rank;
}

// ---- long lists: buckets in place of the table -----------------------------------------------
//
// An insertion into the table is a dependent load and an atomic at the memory side, and the table itself is
// cleared first; found by buckets, first occurrences cost streams.  Units are the mapping ids, tile by tile,
// then, from a tile of their own on, the requiring ids that are not mapping ids themselves: an id that is equal to
// the one in front of it is none (the rows of an edge list come in runs), so that those add little.
// Bound: the chains of waits of four launches and the hashed form's LDS work.  890 k ids, most of them new, and 832 k
// edges: sort 11.9, first 10.1, rank 12.1, lookup 11.8 us, where clearing the table took 5.4, the insertions 48.7, rank 10.8
// and lookup 13.2.
constexpr uint32_t kAbsent = kNoId;

// Where a tile of entries of a segment list lies: one after the other in one segment, as a rule.  (No segment is
// named by a number that is not a constant: the list would be copied to memory for it.)
template <typename T>
__device__ __forceinline__ T* seg_at(const dgs_segments& s, int64_t i, int* seg = nullptr) {
  T* p = static_cast<T*>(const_cast<void*>(s.ptr[0])) + i;
  if (seg) *seg = 0;
#pragma unroll
  for (int k = 1; k < DGS_MAX_SEGMENTS; ++k) {
    if (k < s.count && i >= s.len[k - 1]) {
      i -= s.len[k - 1];
      p = static_cast<T*>(const_cast<void*>(s.ptr[k])) + i;
      if (seg) *seg = k;
    } else {
      i = -1;  // stays negative: no later segment can match
    }
  }
  return p;
}
template <typename T, int TILE>
struct TileSpan {
  int64_t first;  // the tile's first entry
  uint32_t count; // its entries
  T* begin;       // where the first one lies
  bool whole;     // and all others behind it
  __device__ __forceinline__ TileSpan(const dgs_segments& s, uint32_t tile, int64_t total) {
    first = int64_t(tile) * TILE;
    count = uint32_t(total - first < TILE ? total - first : TILE);
    int from, upto;
    begin = seg_at<T>(s, first, &from);
    seg_at<T>(s, first + count - 1, &upto);
    whole = from == upto;
  }
  __device__ __forceinline__ T& at(const dgs_segments& s, uint32_t e) const { return whole ? nth(begin, e) : *seg_at<T>(s, first + e); }
};

// Units that sort_tile has folded: (place of the one before it that it is equal to, its own place) each, from the end of the tile's
// items downwards, which that many units less leave free.
using Item = BucketItem<true>::type;
template <typename Shape>
__device__ __forceinline__ Item* folded_items(const Buckets& b, uint32_t tile) {
  return static_cast<Item*>(b.items) + (size_t(tile) + 1) * Shape::kTile - 1;
}
template <typename Shape>
__device__ __forceinline__ void unfold_tile(const Buckets& b, uint32_t tile, uint32_t folds, uint32_t* into /* [kTile] in LDS */) {
  for (uint32_t e = threadIdx.x; e < folds && e < uint32_t(Shape::kTile); e += Shape::kThreads) {
    const Item it = folded_items<Shape>(b, tile)[-int64_t(e)];
    into[it.y & (Shape::kTile - 1)] = into[it.x & (Shape::kTile - 1)];
  }
  __syncthreads();
}

// The mapping ids that the table would hold as well.  notes[]: 1 if the tile has met another one, and twice its folded units.
template <typename IdT, typename Shape>
__global__ __launch_bounds__(Shape::kThreads) void bucketed_sort_kernel(dgs_segments mapping, int64_t n, uint32_t map_tiles, dgs_segments queries,
                                                                     int64_t m, Buckets b, uint32_t* __restrict__ notes) {
  __shared__ SortLds<true, Shape> lds;
  __shared__ uint32_t any_bad, folds;
  const uint32_t tile = blockIdx.x;
  if (threadIdx.x == 0) any_bad = folds = 0;
  __syncthreads();
  const bool query = tile >= map_tiles;
  IdT key[Shape::kItems], front[Shape::kItems];  // (front: of a wave's first lane, the query in front of its own)
  uint32_t count;
  const auto load = [&](const dgs_segments& list, uint32_t list_tile, int64_t total, bool fronts) {
    const TileSpan<const IdT, Shape::kTile> span(list, list_tile, total);
    count = span.count;
#pragma unroll
    for (int j = 0; j < Shape::kItems; ++j) {
      const uint32_t e = uint32_t(j * Shape::kThreads) + threadIdx.x;
      key[j] = e < count ? span.at(list, e) : IdT(-1);
      front[j] = fronts && (threadIdx.x & (kWave - 1)) == 0 && e > 0 && e < count ? span.at(list, e - 1) : IdT(-1);
    }
  };
  if (query) load(queries, tile - map_tiles, m, true);
  else load(mapping, tile, n, false);
  uint32_t id[Shape::kItems];
  bool refused = false;
#pragma unroll
  for (int j = 0; j < Shape::kItems; ++j) {
    const uint32_t e = uint32_t(j * Shape::kThreads) + threadIdx.x;
    const bool held = uint64_t(int64_t(key[j])) < 0xffffffffull;
    bool again = false;  // a query equal to the one in front of it
    if (query) {
      const IdT below = __shfl_up(key[j], 1, kWave);
      again = e > 0 && key[j] == ((threadIdx.x & (kWave - 1)) == 0 ? front[j] : below);
    }
    refused |= e < count && !held;
    id[j] = e < count && held && !again ? uint32_t(key[j]) : kNoId;
  }
  if (refused) any_bad = 1;
  sort_tile<true, Shape>(b, b.log_buckets, tile, id, lds, [&](int j, uint32_t before) {  // noted from the end of the tile's items on
    const uint64_t here = __ballot(1);
    const int lower = __builtin_popcountll(here & ((uint64_t(1) << (threadIdx.x & (kWave - 1))) - 1));
    uint32_t at = 0;
    if (lower == 0) at = atomicAdd(&folds, uint32_t(__builtin_popcountll(here)));
    at = __builtin_amdgcn_readfirstlane(at) + uint32_t(lower);
    folded_items<Shape>(b, tile)[-int64_t(at)] = Item{before, uint32_t(j * Shape::kThreads) + threadIdx.x};
  });
  if (threadIdx.x == 0) notes[tile] = any_bad | folds << 1;  // (sort_tile has barriers)
}

__global__ __launch_bounds__(kBucketBlock) void bucketed_first_kernel(Buckets b, uint32_t tiles) {
  __shared__ HashedLds lds;
  clear_counts(lds.counts, tiles);
  first_of_bucket_hashed(b, b.log_buckets, bucket_in_turn(blockIdx.x, b.log_buckets), tiles, 0, lds);
  add_counts(b, lds.counts, tiles);
}

// rank_kernel's work on one tile of the mapping list.
template <typename IdT, typename Shape>
__global__ __launch_bounds__(Shape::kThreads) void bucketed_rank_kernel(dgs_segments mapping, int64_t n, uint32_t map_tiles, Buckets b,
                                                                     const uint32_t* __restrict__ notes, uint32_t* __restrict__ slot,
                                                                     IdT* __restrict__ unique_out, int64_t* __restrict__ counts_dev,
                                                                     int64_t* __restrict__ counts_host) {
  typedef uint32_t words __attribute__((ext_vector_type(kItems)));
  constexpr int kGroups = Shape::kItems / kItems, kWaves = Shape::kThreads / kWave;
  constexpr uint32_t kGroup = Shape::kThreads * kItems;
  __shared__ __align__(16) uint32_t least_of[Shape::kTile];
  __shared__ uint32_t wave_before[kWaves];
  __shared__ int wave_count[kGroups * kWaves];
  __shared__ int any_bad;
  const uint32_t tile = blockIdx.x, first_unit = tile * Shape::kTile, at = threadIdx.x * kItems;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const bool last = tile + 1 == map_tiles;
  const TileSpan<const IdT, Shape::kTile> span(mapping, tile, n);
  uint32_t before = firsts_before<Shape::kThreads>(b, tile);
  uint32_t refused = 0;
  for (uint32_t t = threadIdx.x; last && t < map_tiles; t += Shape::kThreads) refused |= notes[t] & 1;
  const uint32_t folds = notes[tile] >> 1;
#pragma unroll
  for (int g = 0; g < kGroups; ++g) *reinterpret_cast<words*>(least_of + g * kGroup + at) = words(kAbsent);  // (ids that are no units)
  if (threadIdx.x == 0) any_bad = 0;
  __syncthreads();
  unsort_tile<true, Shape>(b, b.log_buckets, tile, least_of);
  if (refused != 0) any_bad = 1;
#pragma unroll
  for (int d = kWave / 2; d > 0; d >>= 1) before += __shfl_xor(before, d, kWave);
  if (lane == 0) wave_before[wave] = before;
  __syncthreads();
  if (folds != 0) unfold_tile<Shape>(b, tile, folds, least_of);
  words word[kGroups];
  uint32_t first[kGroups];  // bit j: position j of the group's is its id's first
  int lane_before[kGroups];
#pragma unroll
  for (int g = 0; g < kGroups; ++g) {
    first[g] = 0;
    const uint32_t u = first_unit + g * kGroup + at;
    word[g] = *reinterpret_cast<const words*>(least_of + g * kGroup + at);
#pragma unroll
    for (int j = 0; j < kItems; ++j)
      if (int64_t(u + j) < n && word[g][j] == u + j) first[g] |= 1u << j;
    const int c = __builtin_popcount(first[g]);  // its bits are summed over the lanes by ballots
    lane_before[g] = 0;
    int sum = 0;
#pragma unroll
    for (int bit = 0; (1 << bit) <= kItems; ++bit) {
      const uint64_t mask = __ballot((c >> bit) & 1);
      lane_before[g] += __builtin_popcountll(mask & ((uint64_t(1) << lane) - 1)) << bit;
      sum += __builtin_popcountll(mask) << bit;
    }
    if (lane == 0) wave_count[g * kWaves + wave] = sum;
  }
  __syncthreads();
  // the groups' and waves' counts, in the order of the positions: one a lane, summed over the lanes
  static_assert(kGroups * kWaves <= kWave, "a count per lane");
  const int own = lane < kGroups * kWaves ? wave_count[lane] : 0;
  int upto = own;
#pragma unroll
  for (int d = 1; d < kGroups * kWaves; d <<= 1) {
    const int lower = __shfl_up(upto, d, kWave);
    if (lane >= d) upto += lower;
  }
  uint32_t rank0 = wave_before[lane & (kWaves - 1)];
#pragma unroll
  for (int d = kWaves / 2; d > 0; d >>= 1) rank0 += __shfl_xor(rank0, d, kWave);
  if (last && threadIdx.x == kGroups * kWaves - 1) {
    counts_dev[0] = int64_t(rank0) + upto;
    counts_dev[1] = any_bad;
    if (counts_host) {
      mirror_to_host(counts_host, int64_t(rank0) + upto);
      mirror_to_host(counts_host + 1, any_bad);
    }
  }
#pragma unroll
  for (int g = 0; g < kGroups; ++g) {
    const uint32_t u = first_unit + g * kGroup + at;
    uint32_t rank = rank0 + uint32_t(lane_before[g] + __shfl(upto - own, g * kWaves + wave, kWave));
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      if ((first[g] >> j) & 1) {
        unique_out[rank] = span.at(mapping, u + j - first_unit);
        word[g][j] = rank | kFirstBit;
        ++rank;
      } else if (word[g][j] >= u + j) {
        word[g][j] = kNoSlot;  // no unit (or not one that the launches before have left)
      }
    }
    *reinterpret_cast<words*>(slot + u) = word[g];  // (the array holds whole tiles)
  }
}

// Blocks [0, query_tiles): a tile of the queries each, whose ids have their smallest units at the first of every run;
// then blocks of Shape::kTile requiring ids that are mapping ids, given by their words.
template <typename IdT, typename Shape>
__global__ __launch_bounds__(Shape::kThreads) void bucketed_lookup_kernel(dgs_segments queries, int64_t m, uint32_t map_tiles, uint32_t query_tiles,
                                                                       Buckets b, const uint32_t* __restrict__ notes,
                                                                       const uint32_t* __restrict__ slot, int64_t n, dgs_segments query_out,
                                                                       dgs_segments words, int64_t n_words, dgs_segments words_out) {
  __shared__ uint32_t least_of[Shape::kTile];
  __shared__ uint16_t head[Shape::kTile];  // where the run begins that an id belongs to
  __shared__ int wave_head[Shape::kThreads / kWave];
  if (blockIdx.x >= query_tiles) {
    const TileSpan<const uint32_t, Shape::kTile> in(words, blockIdx.x - query_tiles, n_words);
    const TileSpan<IdT, Shape::kTile> to(words_out, blockIdx.x - query_tiles, n_words);
    uint32_t word[Shape::kItems];
#pragma unroll
    for (int j = 0; j < Shape::kItems; ++j) {
      const uint32_t e = uint32_t(j * Shape::kThreads) + threadIdx.x;
      word[j] = e < in.count ? in.at(words, e) : kNoSlot;
    }
#pragma unroll
    for (int j = 0; j < Shape::kItems; ++j)
      if ((word[j] & kFirstBit) == 0) word[j] = int64_t(word[j]) < n ? slot[word[j]] : kNoSlot;
#pragma unroll
    for (int j = 0; j < Shape::kItems; ++j) {
      const uint32_t e = uint32_t(j * Shape::kThreads) + threadIdx.x;
      if (e < in.count) to.at(words_out, e) = (word[j] & kFirstBit) != 0 ? IdT(word[j] & ~kFirstBit) : IdT(-1);
    }
    return;
  }
  const uint32_t tile = map_tiles + blockIdx.x;
  const TileSpan<IdT, Shape::kTile> to(query_out, blockIdx.x, m);
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const bool odd_ones = (notes[tile] & 1) != 0;
  const uint32_t folds = notes[tile] >> 1;
  for (int e = threadIdx.x; e < Shape::kTile; e += Shape::kThreads) least_of[e] = kAbsent;
  __syncthreads();
  unsort_tile<true, Shape>(b, b.log_buckets, tile, least_of);
  __syncthreads();
  if (folds != 0) unfold_tile<Shape>(b, tile, folds, least_of);
  // a thread has eight ids in a row: where the last run begins that does so before or at each
  int own[Shape::kItems], latest = -1;
#pragma unroll
  for (int j = 0; j < Shape::kItems; ++j) {
    const int e = int(threadIdx.x) * Shape::kItems + j;
    if (least_of[e] != kAbsent) latest = e;
    own[j] = latest;
  }
  int upto = latest;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int lower = __shfl_up(upto, d, kWave);
    if (lane >= d && lower > upto) upto = lower;
  }
  if (lane == kWave - 1) wave_head[wave] = upto;
  int prior = __shfl_up(upto, 1, kWave);
  if (lane == 0) prior = -1;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < Shape::kThreads / kWave; ++w)
    if (w < wave && wave_head[w] > prior) prior = wave_head[w];
#pragma unroll
  for (int j = 0; j < Shape::kItems; ++j) {
    const int h = own[j] >= 0 ? own[j] : prior;
    head[int(threadIdx.x) * Shape::kItems + j] = uint16_t(h >= 0 ? h : 0);  // (the first id of a tile is a head, or no id)
  }
  __syncthreads();
  uint32_t word[Shape::kItems];
#pragma unroll
  for (int j = 0; j < Shape::kItems; ++j) {
    const uint32_t least = least_of[head[j * Shape::kThreads + threadIdx.x]];
    word[j] = int64_t(least) < n ? slot[least] : kNoSlot;  // (one of the queries: the id is not in the mapping list)
  }
#pragma unroll
  for (int j = 0; j < Shape::kItems; ++j) {
    const uint32_t e = uint32_t(j * Shape::kThreads) + threadIdx.x;
    if (e >= to.count) continue;
    IdT rank = (word[j] & kFirstBit) != 0 ? IdT(word[j] & ~kFirstBit) : IdT(-1);
    if (odd_ones && uint64_t(int64_t(*seg_at<const IdT>(queries, to.first + e))) >= 0xffffffffull) rank = IdT(-1);  // (in no run)
    to.at(query_out, e) = rank;
  }
}

// ---- small inputs: one block, the table in LDS -----------------------------------------------
//
// Up to kSmallIds mapping ids are handled by a single 1024-thread block whose hash table lives in
// LDS: one launch instead of four, LDS atomics instead of memory-side ones.  One block is one CU,
// though: its probe chains run at one CU's pace (kernel time on 8-byte ids, 6144 ids 43 us, 10240 ids
// 84 us).  us a call with the wait for its count, the block / the launches: 2040 ids 28.6 / 42.1 (mostly new)
// and 27.3 / 35.4 (a tenth new); with four ids a thread in place of two, 3000 ids 32.5 / 39.0 and 29.4 / 34.9,
// 4090 ids 36.4 / 42.2 and 30.7 / 34.9, but every shorter list takes 1.1 us more (512 ids 26.4 -> 27.5).
// Slots are packed words (id in the high half, position / rank in the low half), so an id
// of 2^32 - 1 or more sets the overflow word like the packed table in HBM does.
constexpr int kSmallThreads = 1024;
constexpr int kSmallSlots = 8192;                        // 64 KB of the CU's 160 KB
constexpr int64_t kSmallIds = 2048;                      // load factor <= 0.25: short probe chains
constexpr int kSmallPerThread = int(kSmallIds / kSmallThreads);
constexpr int64_t kSmallRequiring = int64_t(1) << 17;    // ids relabelled by the one block

template <typename IdT>
__global__ __launch_bounds__(kSmallThreads) void small_relabel_kernel(dgs_segments mapping, int64_t n,
                                                                      dgs_segments requiring, int64_t m,
                                                                      IdT* __restrict__ unique_out,
                                                                      int64_t* __restrict__ counts_dev,
                                                                      int64_t* __restrict__ counts_host,
                                                                      dgs_segments out) {
  __shared__ unsigned long long table[kSmallSlots];
  __shared__ int lds[kSmallThreads / kWave];
  __shared__ int overflow;
  constexpr unsigned long long kEmpty = ~0ull;
  constexpr uint32_t kMask = kSmallSlots - 1;
  for (int i = threadIdx.x; i < kSmallSlots; i += kSmallThreads) table[i] = kEmpty;
  if (threadIdx.x == 0) overflow = 0;
  __syncthreads();
  // insert: position i of the mapping list belongs to thread i % 1024, round i / 1024
  // (one block has one CU's worth of memory parallelism: a thread asks for all its ids at once)
  IdT key[kSmallPerThread];
  uint32_t slot[kSmallPerThread];
#pragma unroll
  for (int r = 0; r < kSmallPerThread; ++r) {
    const int64_t i = int64_t(r) * kSmallThreads + threadIdx.x;
    key[r] = i < n ? seg_load<IdT>(mapping, i) : IdT(0);
  }
#pragma unroll
  for (int r = 0; r < kSmallPerThread; ++r) {
    const int64_t i = int64_t(r) * kSmallThreads + threadIdx.x;
    slot[r] = kSmallSlots;  // none
    if (i >= n) continue;
    if (uint64_t(int64_t(key[r])) >= 0xffffffffull) {
      overflow = 1;
      continue;
    }
    const unsigned long long packed = (static_cast<unsigned long long>(uint32_t(key[r])) << 32) | uint32_t(i);
    uint32_t pos = hash_id(uint32_t(key[r])) & kMask;
    for (;;) {
      unsigned long long cur = table[pos];
      if (cur == kEmpty) {
        cur = atomicCAS(&table[pos], kEmpty, packed);
        if (cur == kEmpty) break;
      }
      if (uint32_t(cur >> 32) == uint32_t(key[r])) {
        atomicMin(&table[pos], packed);
        break;
      }
      pos = (pos + 1) & kMask;
    }
    slot[r] = pos;
  }
  __syncthreads();
  // first occurrences: the positions the table kept.  All of them are read before any slot is
  // rewritten with a rank.
  bool first[kSmallPerThread];
#pragma unroll
  for (int r = 0; r < kSmallPerThread; ++r)
    first[r] = slot[r] < kSmallSlots && uint32_t(table[slot[r]]) == uint32_t(r * kSmallThreads + threadIdx.x);
  __syncthreads();
  int base = 0;
#pragma unroll
  for (int r = 0; r < kSmallPerThread; ++r) {  // round by round: ranks follow the order of positions
    int total;
    const int ex = block_exclusive_scan<kSmallThreads, int>(first[r] ? 1 : 0, &total, lds);
    if (first[r]) {
      const uint32_t rank = uint32_t(base + ex);
      unique_out[rank] = key[r];
      table[slot[r]] = (static_cast<unsigned long long>(uint32_t(key[r])) << 32) | rank;
    }
    base += total;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    counts_dev[0] = base;
    counts_dev[1] = overflow;
    if (counts_host) {
      mirror_to_host(counts_host, base);
      mirror_to_host(counts_host + 1, overflow);
    }
  }
  // relabel: rank of every requiring id, -1 when it is not in the table; eight ids a thread at a time
  constexpr int kBatch = 8;
  for (int64_t j0 = 0; j0 < m; j0 += int64_t(kSmallThreads) * kBatch) {
    IdT id[kBatch];
    IdT* dst[kBatch];
#pragma unroll
    for (int b = 0; b < kBatch; ++b) {
      const int64_t j = j0 + int64_t(b) * kSmallThreads + threadIdx.x;
      dst[b] = nullptr;
      id[b] = IdT(-1);
      if (j < m) {
        int seg;
        int64_t off;
        seg_locate(requiring, j, &seg, &off);
        id[b] = static_cast<const IdT*>(requiring.ptr[seg])[off];
        dst[b] = static_cast<IdT*>(const_cast<void*>(out.ptr[seg])) + off;
      }
    }
#pragma unroll
    for (int b = 0; b < kBatch; ++b) {
      if (dst[b] == nullptr) continue;
      IdT rank = IdT(-1);
      if (uint64_t(int64_t(id[b])) < 0xffffffffull) {
        uint32_t pos = hash_id(uint32_t(id[b])) & kMask;
        for (;;) {
          const unsigned long long cur = table[pos];
          if (cur == kEmpty) break;
          if (uint32_t(cur >> 32) == uint32_t(id[b])) {
            rank = IdT(uint32_t(cur));
            break;
          }
          pos = (pos + 1) & kMask;
        }
      }
      *dst[b] = rank;
    }
  }
}

struct UniqueWorkspace {
  void* table;       // capacity slots of the table layout in use
  uint8_t* lost;     // [padded to whole rank tiles], then the rank tiles' states and the overflow word: one region to zero
  tile_state* state;
  int* overflow;
  uint32_t* slot;    // [padded to whole rank tiles, and bucket tiles]
  Buckets buckets;   // of lists that may be bucketed: room for the mapping ids and as many queries
  uint32_t* notes;   // [bucket tiles]
  uint32_t capacity;
  size_t table_bytes;  // multiple of 16 (sized for the larger layout)
  size_t zero_bytes;   // multiple of 16
};

// Lists that may go by buckets: long enough for the table's atomics to cost more than the chains of waits, and short enough
// for the tiles that a block has room to count.  us a call with the wait for its count, table / buckets, of ids mostly new and of
// a tenth new: 131 k 44 / 33, 35 / 33; 180 k 67 / 34, 37 / 35; 250 k of a tenth new 39 / 35; 400 k 56 / 38, 46 / 38; 890 k 83 / 50,
// 65 / 47; 4 M 262 / 213, 239 / 199.
// Short lists have smaller tiles, which are more blocks and less of a chain each.  Tiles of 8192 / 2048 units: 131 k 38 / 33, 41 / 33;
// 180 k 39 / 34, 42 / 35; 400 k 42 / 38, 45 / 38, 890 k 50 / 60 (of 4096, by 512 or 1024 threads, 34 / 35, 36 / 36, 38 / 39, 53; of
// 2048 by 256 threads 35, 36, 40, 60; of 1024 35, 37, 47).
using LongLists = BucketShape;
using ShortLists = TileShape<512, 4>;
constexpr int64_t kBucketedMinIds = int64_t(1) << 17, kShortListIds = int64_t(1) << 19;
inline int64_t bucket_tile(int64_t n) { return n <= kShortListIds ? ShortLists::kTile : LongLists::kTile; }
inline int64_t bucket_tiles(int64_t ids, int64_t tile) { return (ids + tile - 1) / tile; }
constexpr int64_t kBucketedMaxTiles = kMaxBucketTiles / 2;  // of mapping ids (as many of queries)
constexpr int64_t kBucketedMaxIds = kBucketedMaxTiles * LongLists::kTile;
static_assert(kShortListIds / ShortLists::kTile <= kBucketedMaxTiles, "room to count them");
inline bool may_be_bucketed(int64_t n) { return n >= kBucketedMinIds && n <= kBucketedMaxIds; }

// packed 64-bit slots, or id array + value array (the larger: what the workspace is sized for)
size_t slot_bytes(int32_t id_bytes, bool packed) { return packed ? 8 : size_t(id_bytes) + 4; }

void take_buckets(Carver* c, int64_t n, UniqueWorkspace* t) {
  const int64_t tile = bucket_tile(n);
  Buckets& b = t->buckets;
  b.hashed = 1;
  b.hash_slots = kHashSlots;
  b.log_tile = __builtin_ctzll(uint64_t(tile));
  b.tiles_max = int32_t(2 * bucket_tiles(n, tile));
  b.items = c->take<uint2>(size_t(b.tiles_max) * size_t(tile));
  b.least = c->take<uint32_t>(size_t(b.tiles_max) * size_t(tile));
  b.piece = c->take<uint16_t>(size_t(b.tiles_max) * (kMaxBuckets + 1));
  b.firsts = c->take<uint32_t>(kCounters * kMaxBucketTiles);
  t->notes = c->take<uint32_t>(size_t(b.tiles_max));
}

// The slot words, then either the table with its marks or the buckets: an attempt uses one of them, and the one that follows a
// void attempt comes behind it on the stream.  The size never falls as lists grow (a caller sizes one workspace for its longest
// list): lists beyond those that go by buckets have the room of the longest one that does, and those of large tiles that of the
// longest one of small tiles.
size_t unique_workspace_layout(int64_t n, int32_t id_bytes, void* base, UniqueWorkspace* w) {
  if (n < 0) n = 0;
  if (n > kMaxMappingIds) n = kMaxMappingIds;
  const size_t tiles = size_t(n > 0 ? rank_tiles(n) : 1);  // (an empty list has its counts written too)
  const size_t padded = tiles * size_t(kGroupIds) * rank_groups(n);
  UniqueWorkspace t{};
  Carver c(base);
  t.slot = c.take<uint32_t>(std::max(padded, may_be_bucketed(n) ? size_t(bucket_tiles(n, bucket_tile(n)) * bucket_tile(n)) : 0));
  Carver buckets = c;
  t.capacity = table_capacity(n);
  t.table_bytes = size_t(t.capacity) * slot_bytes(id_bytes, id_bytes == 4);
  t.table = c.take<char>(t.table_bytes);
  t.zero_bytes = (padded + tiles * sizeof(tile_state) + sizeof(int) + 15) / 16 * 16;
  t.lost = c.take<uint8_t>(t.zero_bytes);
  t.state = reinterpret_cast<tile_state*>(t.lost + padded);
  t.overflow = reinterpret_cast<int*>(t.state + tiles);
  size_t used = c.used;
  if (n >= kBucketedMinIds) {
    for (const int64_t ids : {std::min(n, kShortListIds), std::min(n, kBucketedMaxIds)}) {
      c = buckets;
      take_buckets(&c, ids, &t);
      used = std::max(used, c.used);
    }
  }
  if (w) *w = t;
  return used + 256;
}

int64_t seg_total(const dgs_segments& s) {
  int64_t t = 0;
  for (int k = 0; k < s.count; ++k) t += s.len[k];
  return t;
}

template <typename IdT, typename TableT>
dgs_status run_unique_relabel(const dgs_segments& mapping, int64_t n, const dgs_segments& requiring,
                              int64_t m, void* unique_out, int64_t* counts_dev, int64_t* counts_host,
                              void** ticket, const dgs_segments& out, const UniqueWorkspace& w, size_t table_bytes,
                              hipStream_t st) {
  const TableT table(w.table, w.capacity);
  const int64_t table16 = int64_t(table_bytes / 16), zeros16 = int64_t(w.zero_bytes / 16);
  hipLaunchKernelGGL(clear_kernel, dim3(uint32_t((table16 + zeros16 + kThreads - 1) / kThreads)), dim3(kThreads), 0,
                     st, static_cast<uint4*>(w.table), table16, reinterpret_cast<uint4*>(w.lost), zeros16);
  DGS_LAUNCH_CHECK();
  if (n > 0) {
    hipLaunchKernelGGL((insert_kernel<IdT, TableT>), dim3(uint32_t((n + kThreads - 1) / kThreads)), dim3(kThreads),
                       0, st, mapping, n, table, w.slot, w.lost, w.overflow);
    DGS_LAUNCH_CHECK();
  }
  const dim3 tiles(uint32_t(n > 0 ? rank_tiles(n) : 1));
  if (rank_groups(n) == 1)
    hipLaunchKernelGGL((rank_kernel<IdT, 1>), tiles, dim3(kThreads), 0, st, mapping, n, w.slot, w.lost, w.state,
                       lookback_polls(), w.overflow, static_cast<IdT*>(unique_out), counts_dev, counts_host);
  else
    hipLaunchKernelGGL((rank_kernel<IdT, kLongGroups>), tiles, dim3(kThreads), 0, st, mapping, n, w.slot, w.lost, w.state,
                       lookback_polls(), w.overflow, static_cast<IdT*>(unique_out), counts_dev, counts_host);
  DGS_LAUNCH_CHECK();
  // the counts are final here: mark the point the caller may wait for
  if (ticket) {
    const dgs_status ts = dgs_ticket_record(st, ticket);
    if (ts != DGS_OK) return ts;
  }
  if (m > 0) {
    SegmentAlias alias;
    for (int r = 0; r < DGS_MAX_SEGMENTS; ++r) {
      alias.mapping_begin[r] = -1;
      int64_t begin = 0;
      for (int k = 0; k < mapping.count && r < requiring.count; ++k) {
        if (requiring.len[r] > 0 && mapping.ptr[k] == requiring.ptr[r] && mapping.len[k] == requiring.len[r])
          alias.mapping_begin[r] = begin;
        begin += mapping.len[k];
      }
    }
    hipLaunchKernelGGL((lookup_kernel<IdT, TableT>), dim3(uint32_t((m + kThreads - 1) / kThreads)), dim3(kThreads),
                       0, st, requiring, m, table, w.slot, n, alias, out);
    DGS_LAUNCH_CHECK();
  }
  return DGS_OK;
}

// The requiring segments that are mapping segments themselves, as segments of slot words, and the others (queries).
struct SplitRequiring {
  dgs_segments queries{}, query_out{}, words{}, words_out{};
};
SplitRequiring split_requiring(const dgs_segments& mapping, const dgs_segments& requiring, const dgs_segments& out, const uint32_t* slot) {
  SplitRequiring r;
  for (int q = 0; q < requiring.count; ++q) {
    if (requiring.len[q] == 0) continue;
    int64_t begin = 0, at = -1;
    for (int k = 0; k < mapping.count; ++k) {
      if (mapping.ptr[k] == requiring.ptr[q] && mapping.len[k] == requiring.len[q]) at = begin;
      begin += mapping.len[k];
    }
    dgs_segments& in = at >= 0 ? r.words : r.queries;
    dgs_segments& to = at >= 0 ? r.words_out : r.query_out;
    in.ptr[in.count] = at >= 0 ? static_cast<const void*>(slot + at) : requiring.ptr[q];
    to.ptr[to.count] = out.ptr[q];
    in.len[in.count++] = to.len[to.count++] = requiring.len[q];
  }
  return r;
}
template <typename IdT, typename Shape>
dgs_status run_bucketed_relabel(const dgs_segments& mapping, int64_t n, const SplitRequiring& r, void* unique_out,
                                int64_t* counts_dev, int64_t* counts_host, void** ticket, const UniqueWorkspace& w, hipStream_t st) {
  const int64_t m = seg_total(r.queries), n_words = seg_total(r.words);
  const uint32_t map_tiles = uint32_t(bucket_tiles(n, Shape::kTile)), query_tiles = uint32_t(bucket_tiles(m, Shape::kTile)), tiles = map_tiles + query_tiles;
  Buckets b = w.buckets;
  b.log_buckets = kMinLogBuckets;
  while (b.log_buckets < kMaxLogBuckets && (int64_t(kHashSlots / 2) << b.log_buckets) < n + m) ++b.log_buckets;
  hipLaunchKernelGGL((bucketed_sort_kernel<IdT, Shape>), dim3(tiles), dim3(Shape::kThreads), 0, st, mapping, n, map_tiles, r.queries, m, b, w.notes);
  DGS_LAUNCH_CHECK();
  hipLaunchKernelGGL(bucketed_first_kernel, dim3(1u << b.log_buckets), dim3(kBucketBlock), 0, st, b, tiles);
  DGS_LAUNCH_CHECK();
  hipLaunchKernelGGL((bucketed_rank_kernel<IdT, Shape>), dim3(map_tiles), dim3(Shape::kThreads), 0, st, mapping, n, map_tiles, b, w.notes, w.slot,
                     static_cast<IdT*>(unique_out), counts_dev, counts_host);
  DGS_LAUNCH_CHECK();
  // the counts are final here: mark the point the caller may wait for
  if (ticket) {
    const dgs_status ts = dgs_ticket_record(st, ticket);
    if (ts != DGS_OK) return ts;
  }
  const uint32_t blocks = query_tiles + uint32_t(bucket_tiles(n_words, Shape::kTile));
  if (blocks > 0)
    hipLaunchKernelGGL((bucketed_lookup_kernel<IdT, Shape>), dim3(blocks), dim3(Shape::kThreads), 0, st, r.queries, m, map_tiles, query_tiles, b,
                       w.notes, w.slot, n, r.query_out, r.words, n_words, r.words_out);
  DGS_LAUNCH_CHECK();
  return DGS_OK;
}

// Whether the current device lets one block have the LDS the small kernel declares (checked once
// per process; a device that does not takes the general path).
bool small_path_fits() {
  static const bool fits = [] {
    int dev = 0, lds_per_block = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    if (hipDeviceGetAttribute(&lds_per_block, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    return size_t(lds_per_block) >= sizeof(unsigned long long) * kSmallSlots + 1024;
  }();
  return fits;
}

}  // namespace
}  // namespace dgs

DGS_API size_t dgs_unique_relabel_workspace_bytes(int64_t n_mapping, int32_t id_bytes) {
  if (!dgs::width_ok(id_bytes)) id_bytes = 8;
  return dgs::unique_workspace_layout(n_mapping, id_bytes, nullptr, nullptr);
}

DGS_API dgs_status dgs_unique_relabel(dgs_segments mapping, dgs_segments requiring, int32_t id_bytes,
                                      int32_t packed_table, void* unique_out, int64_t* counts_dev,
                                      int64_t* counts_host, void** counts_ticket, dgs_segments out, void* workspace,
                                      size_t workspace_bytes, void* stream) {
  using namespace dgs;
  DGS_REQUIRE(width_ok(id_bytes), DGS_ERR_INVALID, "relabel: id width %d is not 4 or 8", id_bytes);
  DGS_REQUIRE(mapping.count >= 0 && mapping.count <= DGS_MAX_SEGMENTS && requiring.count >= 0 &&
                  requiring.count <= DGS_MAX_SEGMENTS,
              DGS_ERR_INVALID, "relabel: segment count out of range");
  DGS_REQUIRE(out.count == requiring.count, DGS_ERR_INVALID, "relabel: %d outputs for %d inputs", out.count,
              requiring.count);
  for (int k = 0; k < mapping.count; ++k)
    DGS_REQUIRE(mapping.len[k] >= 0 && (mapping.len[k] == 0 || mapping.ptr[k]), DGS_ERR_INVALID,
                "relabel: bad mapping segment %d", k);
  for (int k = 0; k < requiring.count; ++k)
    DGS_REQUIRE(requiring.len[k] >= 0 && out.len[k] == requiring.len[k] &&
                    (requiring.len[k] == 0 || (requiring.ptr[k] && out.ptr[k])),
                DGS_ERR_INVALID, "relabel: bad requiring/output segment %d", k);
  DGS_REQUIRE(counts_dev != nullptr, DGS_ERR_INVALID, "relabel: null counts_dev");
  DGS_REQUIRE(counts_ticket == nullptr || counts_host != nullptr, DGS_ERR_INVALID,
              "relabel: a counts_ticket needs counts_host");
  const int64_t n = seg_total(mapping);
  const int64_t m = seg_total(requiring);
  DGS_REQUIRE(n <= kMaxMappingIds, DGS_ERR_UNSUPPORTED, "relabel: %lld mapping ids exceed 2^30", (long long)n);
  DGS_REQUIRE(m <= int64_t(0x7fffffff) * kThreads, DGS_ERR_UNSUPPORTED, "relabel: too many ids to relabel");
  DGS_REQUIRE(n == 0 || unique_out != nullptr, DGS_ERR_INVALID, "relabel: null unique_out");
  DGS_REQUIRE(workspace != nullptr && workspace_bytes >= dgs_unique_relabel_workspace_bytes(n, id_bytes),
              DGS_ERR_WORKSPACE, "relabel: workspace of %zu B, need %zu", workspace_bytes,
              dgs_unique_relabel_workspace_bytes(n, id_bytes));
  DGS_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 255) == 0, DGS_ERR_WORKSPACE,
              "relabel: workspace must be 256-byte aligned");
  UniqueWorkspace w;
  unique_workspace_layout(n, id_bytes, workspace, &w);
  hipStream_t st = static_cast<hipStream_t>(stream);
  // small inputs with packable ids: the one-block kernel with its table in LDS
  if (n <= kSmallIds && m <= kSmallRequiring && (id_bytes == 4 || packed_table != 0) && small_path_fits()) {
    if (id_bytes == 4)
      hipLaunchKernelGGL(small_relabel_kernel<int32_t>, dim3(1), dim3(kSmallThreads), 0, st, mapping, n, requiring, m,
                         static_cast<int32_t*>(unique_out), counts_dev, counts_host, out);
    else
      hipLaunchKernelGGL(small_relabel_kernel<int64_t>, dim3(1), dim3(kSmallThreads), 0, st, mapping, n, requiring, m,
                         static_cast<int64_t*>(unique_out), counts_dev, counts_host, out);
    DGS_LAUNCH_CHECK();
    return counts_ticket ? dgs_ticket_record(st, counts_ticket) : DGS_OK;
  }
  // (an attempt that packed_table asks for: ids that do not fit a word void it)
  if (packed_table != 0 && may_be_bucketed(n) && lookback_polls() == kLookbackPolls) {  // (test hook of the launches that it replaces)
    const SplitRequiring r = split_requiring(mapping, requiring, out, w.slot);
    const int64_t tile = bucket_tile(n);
    if (bucket_tiles(seg_total(r.queries), tile) <= bucket_tiles(n, tile)) {
      const auto run = [&](auto id, auto shape) {
        return run_bucketed_relabel<decltype(id), decltype(shape)>(mapping, n, r, unique_out, counts_dev, counts_host, counts_ticket, w, st);
      };
      if (tile == ShortLists::kTile) return id_bytes == 4 ? run(int32_t(0), ShortLists{}) : run(int64_t(0), ShortLists{});
      return id_bytes == 4 ? run(int32_t(0), LongLists{}) : run(int64_t(0), LongLists{});
    }
  }
  if (id_bytes == 4)
    return run_unique_relabel<int32_t, Table<int32_t, true>>(mapping, n, requiring, m, unique_out, counts_dev,
                                                             counts_host, counts_ticket, out, w, w.table_bytes, st);
  if (packed_table != 0)  // 8-byte ids in 8-byte slots: ids of 2^32 - 1 or more set the overflow word
    return run_unique_relabel<int64_t, Table<int64_t, true>>(mapping, n, requiring, m, unique_out, counts_dev,
                                                             counts_host, counts_ticket, out, w,
                                                             size_t(w.capacity) * 8, st);
  return run_unique_relabel<int64_t, Table<int64_t, false>>(mapping, n, requiring, m, unique_out, counts_dev,
                                                            counts_host, counts_ticket, out, w, w.table_bytes, st);
}
