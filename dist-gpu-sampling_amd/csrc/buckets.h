// First occurrences of a long list of ids without memory-side atomics: the list is cut into tiles, a block
// puts its tile's units in bucket order, and then a block per bucket finds the smallest unit of every id in
// LDS.
//
// A unit is an entry of the list; its number is its order.  Three launches:
//   sort     a block per tile of kBucketTile units: counted by bucket, placed and staged in LDS, written as
//            one contiguous run of items; piece[tile][b] says where bucket b's piece begins in the run;
//   first    a block per bucket: its pieces in all tiles are read by 16 lanes each, the smallest unit of every
//            id is found in LDS, and least[] gets it for every unit, at the unit's place in the sorted run; the
//            tiles' first occurrences are counted;
//   the caller's launch that goes over a tile again reads the tile's run of items and least[] as streams
//            and puts them back in the order of the units in LDS (unsort_tile).
// All of it is streams and LDS work: what is read or written out of order are pieces of some 32 items.  Bound: the
// chain of waits of each launch (its length, then what hangs on it, then the LDS work between barriers), for which
// there is little to do but to keep it short: 1024 threads with eight units each, every load asked for at once.
// us a launch, 1024 seeds, fanouts [5,10,15], 832 k picks in 109 tiles, 256 buckets: sort 7.9, first 6.8, the compact
// launch behind them 10.4; before (256 threads with 16 units and items of two words; a block of 256 threads that
// searched the pieces for its units; repeats' slot words stored at random) 11.5, 16.2 and 9.9, and 204 -> 191 for the
// batch with its features.  The three together with 512 threads and 8 / 16 units, 256 and 16: 25.7, 28.2,
// 35.2 (25.9 with 1024; 512 buckets).  8 batches through the loader, of 1024 / 2048 seeds: 1354 / 2195, with 512 threads and 8 units
// 1356 / 2214, 16 1366 / 2200, 256 and 8 1370 / 2232, 16 1358 / 2197, the pass before 1355 / 2290; sort and compact held to 64
// registers, which spills, 1387.
//
// Two forms.  Direct: bucket = low bits of the id, and the high bits index an array of kBucketRange entries;
// items are one word (the high bits and the unit's place in its tile).  Hashed, for any number of ids:
// bucket = low bits of a hash that takes no two ids to one value, hashes are told apart in an open-addressing table of
// packed words (hash, unit), items are the hash and the unit.  A bucket whose ids do not fit that table is gone over
// again in parts, by other bits of the hash, one table's worth at a time; a part whose ids crowd it all the same (not by
// chance) in ranges of its hashes, each of which a table takes whatever the ids (in_parts).
#ifndef DGS_CSRC_BUCKETS_H_
#define DGS_CSRC_BUCKETS_H_

#include <type_traits>

#include "common.h"
#include "table.h"

namespace dgs {

constexpr int kBucketBlock = 1024;                   // threads of the launch that finds the first ones
template <int THREADS, int ITEMS> struct TileShape {  // of the launches that go over tiles: a block's threads, units a thread takes
  static constexpr int kThreads = THREADS, kItems = ITEMS, kTile = THREADS * ITEMS;
};
using BucketShape = TileShape<1024, 8>;
constexpr int kBucketTile = BucketShape::kTile;      // units of a tile, at most
constexpr int kLocalBits = 13;
static_assert(1 << kLocalBits == kBucketTile, "a unit's place in its tile");
constexpr int kMaxBucketTiles = 8388608 / kBucketTile;  // 8.4 M units
constexpr int kMinLogBuckets = 8, kMaxLogBuckets = 10;
constexpr int kMaxBuckets = 1 << kMaxLogBuckets;
constexpr int kBucketRange = 16384;                  // direct: ids per bucket at most, 64 KB of LDS
constexpr int64_t kDirectMaxIds = int64_t(kMaxBuckets) * kBucketRange;
constexpr int kHashSlots = 16384;                    // hashed: entries of a bucket's table, 128 KB of LDS
constexpr int kFewProbes = 64;                       // ... of which an id sees this many at first
static_assert(int64_t(kHashSlots / 2) * kMaxBuckets >= int64_t(kMaxBucketTiles) * kBucketTile, "half full, were all units' ids different");

// A tile's first occurrences are counted by the blocks of all buckets, each of which adds its counts of all tiles with a
// few atomics of whole lines (one for every piece took 44 us); several counters, so that few blocks meet at one.  The
// compact launch adds them up where it would have to look back at the tiles before: 10.5 us against 13.9.
constexpr int kCounters = 8;

struct Buckets {
  void* items;         // [tiles_max][kBucketTile] one word or two (hashed) each
  uint32_t* least;     // [tiles_max][kBucketTile] smallest unit of the item's id
  uint16_t* piece;     // [tiles_max][buckets + 1]; the last one: units of the tile
  uint32_t* firsts;    // [kCounters][kMaxBucketTiles] units that are their ids' smallest (of those that count, see below)
  int* overflow;       // the sampler's: a bucket was not answered
  int32_t tiles_max;
  int32_t log_buckets; // hashed: at most
  int32_t log_tile;    // units of a tile
  uint32_t n_ids;      // direct: ids are below it
  int32_t hashed;
  int32_t hash_slots;  // kHashSlots (a test hook makes it small, so that small inputs fill it)
};

constexpr uint32_t kNoId = 0xffffffffu;              // an entry of the list that holds none

// Element i of an array of less than 4 GB: a scalar base and one register of offset.
template <typename T>
__device__ __forceinline__ T& nth(T* base, uint32_t i) {
  return *reinterpret_cast<T*>(reinterpret_cast<char*>(const_cast<std::remove_const_t<T>*>(base)) + uint32_t(i * uint32_t(sizeof(T))));
}

// Buckets of a list of that many units.  Direct: by the number of ids.  Hashed: as few as leave a bucket's table a
// quarter empty on average were all its units' ids different (R-MAT, 3.1 M units: 45 us for the launch with 256, 49 with 512).
__device__ __forceinline__ int log_buckets_of(const Buckets& b, uint32_t units) {
  if (!b.hashed) return b.log_buckets;
  int lb = kMinLogBuckets;
  while (lb < b.log_buckets && (uint32_t(b.hash_slots / 4 * 3) << lb) < units) ++lb;
  return lb;
}
// Bucket number i of a launch.  Blocks go to the 8 XCDs in turn: buckets whose pieces lie side by side go to one of
// them, whose L2 then reads the lines that they share once and puts their stores together.  The launch with neighbours
// on different XCDs / on the same one: direct 7.6 / 5.9 us, hashed with pieces of 8 items 130 / 50.
__device__ __forceinline__ int bucket_in_turn(int i, int log_buckets) { return (i & 7) << (log_buckets - 3) | i >> 3; }

template <bool HASHED> struct BucketItem;
template <> struct BucketItem<false> {
  using type = uint32_t;
  static __device__ __forceinline__ uint32_t bucket(uint32_t id, int log_buckets) { return id & ((1u << log_buckets) - 1); }
  static __device__ __forceinline__ type make(uint32_t id, int log_buckets, uint32_t local) { return id >> log_buckets << kLocalBits | local; }
  static __device__ __forceinline__ uint32_t local(type item) { return item & (kBucketTile - 1); }
};
template <> struct BucketItem<true> {
  typedef uint32_t type __attribute__((ext_vector_type(2)));
  static __device__ __forceinline__ uint32_t bucket(uint32_t id, int log_buckets) { return hash_id(id) & ((1u << log_buckets) - 1); }
  static __device__ __forceinline__ type make(uint32_t id, int, uint32_t local) { return type{hash_id(id), local}; }
  static __device__ __forceinline__ uint32_t local(type item) { return item.y; }
};

template <bool HASHED, typename Shape>
struct SortLds {
  int count[kMaxBuckets];  // units of every bucket, then where its piece begins
  __align__(8) typename BucketItem<HASHED>::type stage[Shape::kTile];
  int scan[Shape::kThreads / kWave];
  int hot;
};
// A piece of that many units (four times the average, or more) is one id's or a few ids', as a rule.
template <typename Shape> constexpr int kHotPiece = Shape::kTile / 64;

// The units in hot buckets whose id has one before them in the tile are none: folded(j, place of that one in the tile).  An entry of
// the filter goes to the smallest of the ids that meet there, and to its smallest unit; the others stay as they are.
template <bool HASHED, typename Shape, typename Folded>
__device__ __forceinline__ void fold_tile(int log_buckets, uint32_t (&id)[Shape::kItems], SortLds<HASHED, Shape>& lds, Folded folded) {
  using Item = BucketItem<HASHED>;
  constexpr int NT = Shape::kThreads, ITEMS = Shape::kItems;
  constexpr int kEntries = sizeof(lds.stage) / sizeof(unsigned long long), kLogEntries = __builtin_ctz(kEntries);
  unsigned long long* filter = reinterpret_cast<unsigned long long*>(lds.stage);
  for (int j = threadIdx.x; j < kEntries; j += NT) filter[j] = ~0ull;
  __syncthreads();
  const auto packed = [&](int j) { return (static_cast<unsigned long long>(id[j]) << 32) | (uint32_t(j * NT) + threadIdx.x); };
  const auto hot = [&](int j) { return id[j] != kNoId && lds.count[Item::bucket(id[j], log_buckets)] > kHotPiece<Shape>; };
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    if (!hot(j)) continue;
    unsigned long long* entry = filter + (hash_id(id[j]) >> (32 - kLogEntries));
    if (*entry > packed(j)) atomicMin(entry, packed(j));
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    if (!hot(j)) continue;
    const unsigned long long held = filter[hash_id(id[j]) >> (32 - kLogEntries)];
    if (uint32_t(held >> 32) != id[j] || held == packed(j)) continue;
    folded(j, uint32_t(held));
    id[j] = kNoId;
  }
  __syncthreads();
}

// The tile's units in bucket order.  id[j] is that of unit tile * kTile + j * kThreads + thread, or kNoId.  A bucket's units
// are one block's work in the launch behind this one, and meet at one word of LDS if they are one id's: a tile that an id comes up
// in again and again hands on the first one alone (fold_tile).  us a relabel call, without / with it: 4 M ids, one different
// 4630 / 175, ten 625 / 178, a fifth of them one id 1133 / 246; 890 k 1150 / 50, 157 / 49, 221 / 58; without any such id 211 / 213
// and 49.8 / 49.6.  A batch of 4096 seeds, [5,10,15], 2.4 M nodes of 50 neighbours, one node on 5 / 20 / 50 % of the edges: 576
// / 845 / 1035 -> 389 / 253 / 234, none 255 / 254.
template <bool HASHED, typename Shape, typename Folded>
__device__ __forceinline__ void sort_tile(const Buckets& b, int log_buckets, uint32_t tile, uint32_t (&id)[Shape::kItems],
                                         SortLds<HASHED, Shape>& lds, Folded folded) {
  using Item = BucketItem<HASHED>;
  constexpr int NT = Shape::kThreads, ITEMS = Shape::kItems;
  const int buckets = 1 << log_buckets;
  constexpr int kMine = (kMaxBuckets + NT - 1) / NT;  // consecutive buckets of a thread, at most
  const int mine = buckets > NT ? buckets / NT : 1, b0 = int(threadIdx.x) * mine;
  int before[ITEMS];      // units of its bucket that were counted before it
  const auto count = [&] {
    for (int j = threadIdx.x; j < buckets; j += NT) lds.count[j] = 0;
    if (threadIdx.x == 0) lds.hot = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      before[j] = 0;
      if (id[j] != kNoId) before[j] = atomicAdd(&lds.count[Item::bucket(id[j], log_buckets)], 1);
    }
    int most = 0;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) most = before[j] > most ? before[j] : most;
    if (most >= kHotPiece<Shape>) lds.hot = 1;
    __syncthreads();
  };
  count();
  if (lds.hot != 0) {
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) asm volatile("" : "+v"(id[j]));  // (what hangs on them is worked out anew, not kept: 47 registers, 85)
    fold_tile<HASHED, Shape>(log_buckets, id, lds, folded);
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) asm volatile("" : "+v"(id[j]));
    count();
  }
  int own[kMine], sum = 0;
#pragma unroll
  for (int j = 0; j < kMine; ++j) {
    own[j] = j < mine && b0 + j < buckets ? lds.count[b0 + j] : 0;
    sum += own[j];
  }
  int all;
  int at = block_exclusive_scan<NT, int>(sum, &all, lds.scan);  // (has barriers)
  uint16_t* piece = b.piece + size_t(tile) * (buckets + 1);
#pragma unroll
  for (int j = 0; j < kMine; ++j) {
    if (j < mine && b0 + j < buckets) {
      lds.count[b0 + j] = at;
      piece[b0 + j] = uint16_t(at);
      at += own[j];
    }
  }
  if (threadIdx.x == 0) piece[buckets] = uint16_t(all);
  if (threadIdx.x < kCounters) b.firsts[threadIdx.x * kMaxBucketTiles + tile] = 0;  // (for the launch behind this one)
  __syncthreads();
#pragma unroll
  for (int j = 0; j < ITEMS; ++j)
    if (id[j] != kNoId)
      lds.stage[lds.count[Item::bucket(id[j], log_buckets)] + before[j]] =
          Item::make(id[j], log_buckets, uint32_t(j * NT) + threadIdx.x);
  __syncthreads();
  typename Item::type* items = static_cast<typename Item::type*>(b.items) + size_t(tile) * Shape::kTile;
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const int e = j * NT + int(threadIdx.x);
    if (e < all) nth(items, uint32_t(e)) = lds.stage[e];
  }
}

// A bucket's units, as the threads of its block come by them: 16 lanes have a piece, four or six pieces at a time,
// of each of which the first 48 units are read at once.
constexpr int kPieceLanes = 16, kPieceGroups = kBucketBlock / kPieceLanes;
constexpr int kPieceChunks = 3;

template <bool HASHED>
struct PieceRound {
  using Item = BucketItem<HASHED>;
  static constexpr int kPieces = HASHED ? 6 : 4;
  static constexpr uint32_t kTiles = kPieceGroups * kPieces;  // of a round
  uint32_t at[kPieces];   // the lane's first item
  uint32_t end[kPieces];  // the piece's end
  typename Item::type item[kPieces][kPieceChunks];

  __device__ __forceinline__ const typename Item::type* items(const Buckets& b) const { return static_cast<const typename Item::type*>(b.items); }
  __device__ __forceinline__ void load(const Buckets& b, int log_buckets, int bucket, uint32_t first_tile, uint32_t tiles) {
    const uint32_t buckets = 1u << log_buckets;
    uint32_t from[kPieces], upto[kPieces];
#pragma unroll
    for (int q = 0; q < kPieces; ++q) {
      const uint32_t tile = first_tile + uint32_t(q * kPieceGroups) + threadIdx.x / kPieceLanes;
      from[q] = upto[q] = 0;
      if (tile < tiles) {
        from[q] = nth(b.piece + bucket, tile * (buckets + 1));
        upto[q] = nth(b.piece + bucket + 1, tile * (buckets + 1));
      }
    }
#pragma unroll
    for (int q = 0; q < kPieces; ++q) {
      const uint32_t tile = first_tile + uint32_t(q * kPieceGroups) + threadIdx.x / kPieceLanes;
      if (upto[q] > 1u << b.log_tile) upto[q] = 1u << b.log_tile;  // (sizes that no tile has are not followed)
      at[q] = (tile << b.log_tile) + from[q] + (threadIdx.x & (kPieceLanes - 1));
      end[q] = (tile << b.log_tile) + upto[q];
    }
#pragma unroll
    for (int q = 0; q < kPieces; ++q)
#pragma unroll
      for (int c = 0; c < kPieceChunks; ++c)
        if (at[q] + c * kPieceLanes < end[q]) item[q][c] = nth(items(b), at[q] + c * kPieceLanes);
  }
  // units of the round's pieces that the lane's group has, counted once (by its first lane)
  __device__ __forceinline__ int units() const {
    int n = 0;
    if ((threadIdx.x & (kPieceLanes - 1)) == 0) {
#pragma unroll
      for (int q = 0; q < kPieces; ++q) n += end[q] > at[q] ? int(end[q] - at[q]) : 0;
    }
    return n;
  }
  // see(place, item, unit) of every unit; `count` is given, tile by tile, for how many it was true.
  template <typename See, typename Count>
  __device__ __forceinline__ void each(const Buckets& b, See see, Count count) const {
    const int group = int(threadIdx.x & (kWave - 1)) / kPieceLanes * kPieceLanes;
#pragma unroll
    for (int q = 0; q < kPieces; ++q) {
      const uint32_t tile = at[q] >> b.log_tile;  // (an item's place is in its tile)
      int n = 0;
      const auto one = [&](uint32_t e, typename Item::type it) {
        const bool yes = see(e, it, (tile << b.log_tile) + Item::local(it));
        // (the group's first lane is there as long as any of its lanes is)
        n += __builtin_popcountll((__ballot(yes) >> group) & ((1u << kPieceLanes) - 1));
      };
#pragma unroll
      for (int c = 0; c < kPieceChunks; ++c)
        if (at[q] + c * kPieceLanes < end[q]) one(at[q] + c * kPieceLanes, item[q][c]);
      // (longer pieces: of ids that come up again and again, four more at a time)
      for (uint32_t e = at[q] + kPieceChunks * kPieceLanes; e < end[q]; e += 4 * kPieceLanes) {
        typename Item::type more[4];
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (e + c * kPieceLanes < end[q]) more[c] = nth(items(b), e + c * kPieceLanes);
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (e + c * kPieceLanes < end[q]) one(e + c * kPieceLanes, more[c]);
      }
      if (n > 0 && (threadIdx.x & (kPieceLanes - 1)) == 0) count(tile, uint32_t(n));
    }
  }
  template <typename See>
  __device__ __forceinline__ void each(const Buckets& b, See see) const {
    each(b, [&](uint32_t e, typename Item::type it, uint32_t unit) { see(e, it, unit); return false; }, [](uint32_t, uint32_t) {});
  }
};

// The block's counts of first occurrences, tile by tile, go to the launch's.
__device__ __forceinline__ void clear_counts(uint32_t* counts /* [kMaxBucketTiles] in LDS */, uint32_t tiles) {
  for (uint32_t t = threadIdx.x; t < tiles; t += kBucketBlock) counts[t] = 0;
}
__device__ __forceinline__ void add_counts(const Buckets& b, const uint32_t* counts, uint32_t tiles) {
  for (uint32_t t = threadIdx.x; t < tiles; t += kBucketBlock)
    if (counts[t] != 0) atomicAdd(b.firsts + (blockIdx.x / 8 % kCounters) * kMaxBucketTiles + t, counts[t]);
}

// least[] of the bucket's units from `first_unit` on, which are also those that count (units before it take part, but
// nobody asks for theirs).
__device__ __forceinline__ void first_of_bucket_direct(const Buckets& b, int bucket, uint32_t tiles, uint32_t first_unit,
                                                       uint32_t* best /* [kBucketRange] in LDS */, uint32_t* counts) {
  const uint32_t range = (b.n_ids + (1u << b.log_buckets) - 1) >> b.log_buckets;  // <= kBucketRange by the plan
  PieceRound<false> round;
  round.load(b, b.log_buckets, bucket, 0, tiles);
  for (uint32_t j = threadIdx.x * 4; j < range && j < uint32_t(kBucketRange); j += kBucketBlock * 4)
    *reinterpret_cast<uint4*>(best + j) = make_uint4(~0u, ~0u, ~0u, ~0u);
  __syncthreads();
  for (uint32_t t0 = 0; t0 < tiles; t0 += PieceRound<false>::kTiles) {
    if (t0 > 0) round.load(b, b.log_buckets, bucket, t0, tiles);
    round.each(b, [&](uint32_t, uint32_t item, uint32_t unit) {
      const uint32_t at = item >> kLocalBits;
      if (at < uint32_t(kBucketRange)) atomicMin(&best[at], unit);
    });
  }
  __syncthreads();
  for (uint32_t t0 = 0; t0 < tiles; t0 += PieceRound<false>::kTiles) {
    if (tiles > PieceRound<false>::kTiles) round.load(b, b.log_buckets, bucket, t0, tiles);  // (a single round is in registers still)
    round.each(b, [&](uint32_t e, uint32_t item, uint32_t unit) {
      const uint32_t at = item >> kLocalBits;
      if (unit < first_unit || at >= uint32_t(kBucketRange)) return false;
      const uint32_t least = best[at];
      nth(b.least, e) = least;
      return least == unit;
    }, [&](uint32_t tile, uint32_t n) { counts[tile] += n; });  // (nobody else has the tile's piece of this bucket)
  }
  __syncthreads();  // best[] is rewritten by the block's next bucket
}

struct HashedLds {
  __align__(16) unsigned long long table[kHashSlots];  // hash << 32 | smallest unit; all ones: empty
  uint32_t counts[kMaxBucketTiles];
  int units;
  int overflow;
};
// Part `part` of `parts` of a bucket, by bits of the hash that did not choose the bucket, and of it the hashes whose other
// bits are `span` numbers from `lo` on.
struct HashPart {
  int part, parts;
  uint32_t lo, span;
};
constexpr int kPartBit = 23, kPartValues = 1 << (32 - kPartBit);  // what the choice of a part looks at
// Goes over a bucket of so many units in parts that fill half a table, were all units' ids different; a part that
// `attempt` says its table has not taken, value by value of the bits that chose the part, in ranges of as many hashes as
// a table has slots: no two ids have one hash, so each is taken whatever the ids are.  A sweep reads the
// whole bucket, and there are no more than kPartValues for the parts and as many (256 buckets: twice as many) for the ranges.
// 2 M ids that were made for one of 256 buckets: 244 + 226 sweeps.  A relabel call of such ids, by far the longest that there is:
// 131 k 17 ms, 262 k 31, 1 M 240, 2 M 613 (on the table, where they meet too, 0.7 to 1.3).
template <typename Attempt>
__device__ __forceinline__ bool in_parts(int units, int slots, int log_buckets, Attempt attempt) {
  const int half_tables = (units + slots / 2 - 1) / (slots / 2), parts = half_tables < kPartValues ? half_tables : kPartValues;
  const uint32_t hashes = 1u << (kPartBit - log_buckets), span = hashes < uint32_t(kHashSlots) ? hashes : uint32_t(kHashSlots);  // of a value; of a range
  bool took = true;
  for (int part = 0; part < parts; ++part) {
    bool fits = attempt(HashPart{part, parts, 0u, ~0u});
    if (!fits && slots == kHashSlots) {
      fits = true;
      for (uint32_t value = part; value < uint32_t(kPartValues); value += parts)
        for (uint32_t lo = value * hashes; lo < (value + 1) * hashes; lo += span) fits &= attempt(HashPart{part, parts, lo, span});
    }
    took &= fits;
  }
  return took;
}
// All units of the bucket, or (PARTS) of a part of it; returns whether the table took them (the same in all threads),
// within max_probes probes each.
template <bool PARTS>
__device__ __forceinline__ bool first_of_part_hashed(const Buckets& b, int log_buckets, int bucket, uint32_t tiles, uint32_t first_unit,
                                                     HashPart part, int max_probes, HashedLds& lds) {
  using ItemT = BucketItem<true>::type;
  const int slots = b.hash_slots;
  const uint32_t mask = uint32_t(slots - 1);
  const auto elsewhere = [&](uint32_t hash) {
    return PARTS && (int((hash >> kPartBit) % uint32_t(part.parts)) != part.part || (hash >> log_buckets) - part.lo >= part.span);
  };
  PieceRound<true> round;
  round.load(b, log_buckets, bucket, 0, tiles);
  for (int j = threadIdx.x; j < slots / 2; j += kBucketBlock) reinterpret_cast<uint4*>(lds.table)[j] = make_uint4(~0u, ~0u, ~0u, ~0u);
  if (threadIdx.x == 0) lds.overflow = 0;
  __syncthreads();
  for (uint32_t t0 = 0; t0 < tiles; t0 += PieceRound<true>::kTiles) {
    if (t0 > 0) round.load(b, log_buckets, bucket, t0, tiles);
    round.each(b, [&](uint32_t, ItemT item, uint32_t unit) {
      if (elsewhere(item.x)) return;
      if (PARTS && *const_cast<volatile int*>(&lds.overflow) != 0) return;  // (a full table is searched to its end by whoever comes too late)
      const unsigned long long packed = (static_cast<unsigned long long>(item.x) << 32) | unit;
      uint32_t slot = (item.x >> log_buckets) & mask;
      bool placed = false;
      for (int probes = 0; probes < max_probes && !placed; ++probes) {
        unsigned long long cur = lds.table[slot];
        if (cur == ~0ull) cur = atomicCAS(&lds.table[slot], ~0ull, packed);
        placed = cur == ~0ull || uint32_t(cur >> 32) == item.x;
        if (placed && cur > packed && cur != ~0ull) atomicMin(&lds.table[slot], packed);
        slot = (slot + 1) & mask;
      }
      if (!placed) lds.overflow = 1;
    });
  }
  __syncthreads();
  const bool took = lds.overflow == 0;
  if (took) {
    for (uint32_t t0 = 0; t0 < tiles; t0 += PieceRound<true>::kTiles) {
      if (tiles > PieceRound<true>::kTiles) round.load(b, log_buckets, bucket, t0, tiles);  // (a single round is in registers still)
      round.each(b, [&](uint32_t e, ItemT item, uint32_t unit) {
        if (unit < first_unit) return false;
        if (elsewhere(item.x)) return false;
        uint32_t slot = (item.x >> log_buckets) & mask;
        unsigned long long held = lds.table[slot];
        for (int probes = 0; probes < slots && uint32_t(held >> 32) != item.x; ++probes) {
          slot = (slot + 1) & mask;
          held = lds.table[slot];
        }
        nth(b.least, e) = uint32_t(held);
        return uint32_t(held) == unit;
      }, [&](uint32_t tile, uint32_t n) { lds.counts[tile] += n; });  // (nobody else has the tile's piece of this bucket)
    }
  }
  __syncthreads();  // the table is rewritten
  return took;
}
// A bucket of many units may be one of few ids: it is gone over in parts only where the table has not taken them all.  Returns
// whether it was answered: it is, but for one that crowds a part of it where a test hook has made the tables small.
__device__ __forceinline__ bool first_of_bucket_hashed(const Buckets& b, int log_buckets, int bucket, uint32_t tiles,
                                                       uint32_t first_unit, HashedLds& lds) {
  const int few = kFewProbes < b.hash_slots ? kFewProbes : b.hash_slots;
  if (first_of_part_hashed<false>(b, log_buckets, bucket, tiles, first_unit, HashPart{0, 1, 0u, ~0u}, few, lds)) return true;
  if (threadIdx.x == 0) lds.units = 0;
  __syncthreads();
  int n = 0;
  for (uint32_t t0 = 0; t0 < tiles; t0 += PieceRound<true>::kTiles) {
    PieceRound<true> round;
    round.load(b, log_buckets, bucket, t0, tiles);
    n += round.units();
  }
  if (n > 0) atomicAdd(&lds.units, n);
  __syncthreads();
  return in_parts(lds.units, b.hash_slots, log_buckets, [&](HashPart part) {
    // (a part that would take longer searches is gone over in ranges, whose hashes all begin at slots of their own)
    const int probes = part.span == ~0u && b.hash_slots == kHashSlots ? kFewProbes : b.hash_slots;
    return first_of_part_hashed<true>(b, log_buckets, bucket, tiles, first_unit, part, probes, lds);
  });
}

// into[place of a unit in the tile] = its id's smallest unit, for all of the tile's units.
template <bool HASHED, typename Shape>
__device__ __forceinline__ void unsort_tile(const Buckets& b, int log_buckets, uint32_t tile, uint32_t* into /* [kTile] in LDS */) {
  using Item = BucketItem<HASHED>;
  constexpr int NT = Shape::kThreads, ITEMS = Shape::kItems;
  const auto* items = static_cast<const typename Item::type*>(b.items) + size_t(tile) * Shape::kTile;
  const uint32_t* least = b.least + size_t(tile) * Shape::kTile;
  const int count = b.piece[size_t(tile) * ((1 << log_buckets) + 1) + (1 << log_buckets)];
  typename Item::type item[ITEMS];
  uint32_t value[ITEMS];
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {  // (the arrays hold whole tiles)
    item[j] = nth(items, uint32_t(j * NT) + threadIdx.x);
    value[j] = nth(least, uint32_t(j * NT) + threadIdx.x);
  }
#pragma unroll
  for (int j = 0; j < ITEMS; ++j)
    if (j * NT + int(threadIdx.x) < count) into[Item::local(item[j]) & (Shape::kTile - 1)] = value[j];
}

// First occurrences in the tiles before `tile`: the sum over the block's threads of what each is returned.
template <int NT>
__device__ __forceinline__ uint32_t firsts_before(const Buckets& b, uint32_t tile) {
  uint32_t n = 0;
  for (uint32_t t = threadIdx.x; t < tile; t += NT) {
#pragma unroll
    for (int c = 0; c < kCounters; ++c) n += b.firsts[c * kMaxBucketTiles + t];
  }
  return n;
}

}  // namespace dgs
#endif
