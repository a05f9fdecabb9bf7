// The packed edge list of one hop of the fused sampler: what the launch that writes it needs, and the work
// of one block.  It is off the critical path, so it runs as surplus blocks of another launch where there is
// one: the next hop's fill, or the gather of the feature rows behind the last hop.
#ifndef DGS_CSRC_EDGES_H_
#define DGS_CSRC_EDGES_H_

#include "common.h"

namespace dgs {

constexpr int kEdgeBlock = 256;
constexpr int kRowTile = 256;    // seed rows per tile
constexpr int kEdgeItems = 4;    // padded picks per thread
constexpr uint32_t kFirstBit = 0x80000000u;
// row_cnt markers of rows that make the call fail (bit (kBadRow - marker) of the hop's flag word)
constexpr uint32_t kBadRow = 0xffffffffu;      // degree >= 2^32, or offsets outside the edge array
constexpr uint32_t kBadSeed = 0xfffffffeu;     // the seed id is not a row of the graph
constexpr uint32_t kBadPick = 0xfffffffdu;     // a picked neighbour id is outside what the table holds
__device__ __forceinline__ bool is_bad_row(uint32_t row_cnt) { return row_cnt >= kBadPick; }

// ---- Slot words ----
//
// What the slot word of a position says when its edge is written out:
//   kFirstBit | table slot    the first occurrence of its id: its rank is at the position itself;
//   kRankBit | rank           the rank itself (bucketed hops);
//   a position                of the same id and smaller, or the position's own where it has lost its bit:
//                             the rank is there, or a link to a smaller position;
//   table slot                in hop 0, whose first occurrences are settled by asking the table.
// A pick that is not its id's first has met a smaller position of the id when it was inserted.  That one may
// itself be displaced later in the same launch: whoever does so leaves a link to its own position in rank_at,
// and positions only get smaller along the links.  What makes every position met a rank or a link: one of the same
// launch is linked when it is displaced, and one of an earlier hop is its id's smallest for good, because a hop's
// launches end before the next hop looks (see DirectTable).  Hop 0 leaves no links: its displaced positions hold
// numbers that mean nothing, and none of them may be met later.  Reading these words, a stream and some 4-byte reads near
// one another, in place of the table's entry saves a random read of a table that caches do not hold: R-MAT of
// 2^26 nodes, 3.05 M picks, two thirds of them repeats: 44 -> 25 us for the hop's edge list, 376 -> 365 for the batch.
constexpr uint32_t kRankBit = 0x40000000u;
constexpr uint32_t kLinkBit = 0x80000000u;

struct EdgeJob {
  const int64_t* n_seeds;      // device scalar: rows of the hop (used when n_seeds_host < 0)
  int64_t n_seeds_host;
  const uint32_t* row_cnt;     // [s_max] picks of every row
  const uint32_t* row_off;     // [s_max] first packed edge of the row
  const uint32_t* slot;        // [all positions]
  const uint32_t* rank_at;     // [all positions]
  void* src_local;
  void* dst_local;
  int64_t s_max;
  int64_t first;               // position of the hop's first pick
  int64_t bucket_pos_cap;      // the words are those of a bucketed hop if its padded picks are no more than this
  int64_t blocks;              // virtual blocks of the worst case (0: nothing to write)
  int32_t k;
  int32_t id_bytes;
};

// (written without a conditional so that the read is not moved behind a test)
__device__ __forceinline__ int64_t count_of(const int64_t* n_dev, int64_t n_host) {
  const int64_t on_device = *n_dev;
  const int64_t use_device = n_host >> 63;  // all ones when the count lives on the device
  return (on_device & use_device) | (n_host & ~use_device);
}

__host__ __device__ __forceinline__ int edge_groups(int k) { return (k + kEdgeItems - 1) / kEdgeItems; }
inline int64_t edge_blocks(int64_t s_max, int k) { return ((s_max + kRowTile - 1) / kRowTile) * edge_groups(k); }

// The rank that r, read at position `at`, is, or that the links from there lead to.  A link to no smaller position is
// none that a launch has left: it is not followed (rank 0).
__device__ __forceinline__ uint32_t rank_from(const uint32_t* __restrict__ rank_at, uint32_t at, uint32_t r) {
  while (r & kLinkBit) {
    const uint32_t next = r & ~kLinkBit;
    if (next >= at) return 0;
    at = next;
    r = rank_at[at];
  }
  return r;
}

// One block per (256-row tile, 4 x 256 padded picks): writes the rows' edges at their packed
// offsets; a thread handles four picks, 256 apart, so that a wave has four times the loads in
// flight and the launch a quarter of the waves.  src_local = rank of the picked id; dst_local = rank of the
// row's seed, which is the row number itself except in hop 0, whose seeds may repeat: at_of(word) is the
// position (or rank, if *known) that the word of a repeat names, dst_of(i) the row's rank.
//
// EARLY: the launch is about as large as the hop really is, so a thread requests its own elements
// together with the hop's length and tests afterwards.  Without it the launch was sized for a worst case
// that may exceed the hop many times over (and loops over its virtual blocks): the length is waited for
// first and blocks beyond it leave without having read anything.
template <typename IdT, bool EARLY, typename AtOf, typename DstOf>
__device__ __forceinline__ void edge_tile(const EdgeJob& e, int64_t b, int tid, AtOf at_of, DstOf dst_of) {
  const int k = e.k;
  if (k == 0) return;
  const int groups = edge_groups(k);
  const int64_t tile = b / groups;
  const int group = int(b - tile * groups);
  // the hop's length and this thread's own rows and picks, requested together
  const int64_t s = count_of(e.n_seeds, e.n_seeds_host);
  if (!EARLY && tile * kRowTile >= s) return;
  int64_t i[kEdgeItems], p[kEdgeItems];
  int l[kEdgeItems];
  bool mine[kEdgeItems];
  uint32_t rc[kEdgeItems], off[kEdgeItems], word[kEdgeItems];
#pragma unroll
  for (int j = 0; j < kEdgeItems; ++j) {
    const int chunk = group * kEdgeItems + j;
    const int t = chunk * kEdgeBlock + tid;  // padded pick inside the tile
    const int r = t / k;
    l[j] = t - r * k;
    i[j] = tile * kRowTile + r;
    p[j] = e.first + i[j] * k + l[j];
    mine[j] = chunk < k && i[j] < e.s_max;
    rc[j] = off[j] = word[j] = 0;
    if (mine[j]) {
      rc[j] = e.row_cnt[i[j]];
      off[j] = e.row_off[i[j]];
      word[j] = e.slot[p[j]];
    }
  }
  if (tile * kRowTile >= s) return;  // whole blocks leave together
  // Rank of a pick = rank recorded at the smallest position of its id (see Slot words).  Rounds of
  // loads, each issued for all of the thread's picks before any is used.
  bool live[kEdgeItems];
  bool known[kEdgeItems];  // the word is the rank itself
  uint32_t at[kEdgeItems];
#pragma unroll
  for (int j = 0; j < kEdgeItems; ++j) {
    live[j] = mine[j] && i[j] < s && !is_bad_row(rc[j]) && uint32_t(l[j]) < rc[j];
    at[j] = uint32_t(p[j]);
    known[j] = false;
    if (live[j] && !(word[j] & kFirstBit)) at[j] = at_of(s, word[j], &known[j]);
    if (!known[j] && at[j] > uint32_t(p[j])) at[j] = uint32_t(p[j]);  // (words name no later position: none is read by one that does)
  }
  uint32_t rank[kEdgeItems];
#pragma unroll
  for (int j = 0; j < kEdgeItems; ++j) rank[j] = !live[j] ? 0u : known[j] ? at[j] : e.rank_at[at[j]];
  static_assert(kEdgeItems == 4, "the ranks are looked over at once");
  if ((rank[0] | rank[1] | rank[2] | rank[3]) & kLinkBit) {
#pragma unroll
    for (int j = 0; j < kEdgeItems; ++j) rank[j] = rank_from(e.rank_at, at[j], rank[j]);
  }
#pragma unroll
  for (int j = 0; j < kEdgeItems; ++j) {
    if (!live[j]) continue;
    const int64_t o = int64_t(off[j]) + l[j];
    static_cast<IdT*>(e.src_local)[o] = IdT(rank[j]);
    static_cast<IdT*>(e.dst_local)[o] = IdT(dst_of(i[j]));
  }
}

// The same for a hop after the first.
template <typename IdT, bool EARLY>
__device__ __forceinline__ void later_edge_tile(const EdgeJob& e, int64_t b, int tid) {
  edge_tile<IdT, EARLY>(
      e, b, tid,
      [&](int64_t s, uint32_t word, bool* known) {
        *known = s * e.k <= e.bucket_pos_cap && (word & kRankBit) != 0;
        return *known ? word & (kRankBit - 1) : word;
      },
      [](int64_t i) { return i; });
}

}  // namespace dgs
#endif
