// Multi-hop sampling + relabel as one stream of kernels with no host round trip.  Inside a kernel no
// block depends on another one's being scheduled: the blocks of a compact launch look for the counts of
// the tiles before theirs, and count for themselves what does not come (lookback.h).
//
// The per-hop operators (sample.hip, unique.hip) each read a length back to the host so
// that they can return exactly-sized arrays.  Here every buffer has its worst-case size
// (hop h has at most S_h = S_{h-1} (1 + k_{h-1}) seeds), lengths stay in device memory,
// grids are sized for the worst case and surplus blocks retire at once.
//
// What makes the chain short and cheap:
//   * ranks depend on the ORDER of mapping positions only, so every pick gets the padded
//     position P_h + i*k + l (hop h, row i, pick l; P_h is a host-side constant): no
//     count/scan has to run before the picks are inserted, and positions are unique over
//     the whole call;
//   * a hop's frontier is the next hop's seed list, so ONE table serves all hops, holding
//     for every id the smallest position at which it was seen; seeds are never
//     re-inserted and the frontier is a single array that grows hop by hop;
//   * the table is touched once per pick: the atomicMin that inserts a position also
//     tells whether it is (so far) the smallest of its id and which position it displaced;
//     the displaced one is marked lost.  "First occurrence" is then decided from two
//     streamed arrays, without a second random read of the table.  Random 8-byte
//     accesses are what bounds these kernels (on MI355X: loads 71 G/s, atomics 26.7 G/s, every
//     device-scope atomic being executed at the memory side), and a hop costs two of them
//     per pick: the indices read and the table atomic.
//
// A large last hop of uniform picks does without the table altogether (buckets.h): its fill records the
// picked ids, two launches group them by id and find the first position of every id in LDS, and a
// compact launch of its own leaves the slot words that relabel reads on the table path.
//
// Critical path per hop (2 launches): fill -> compact.
//   fill     G lanes per seed row (G = 8..64): indptr pair, picks by the dgs-philox-1
//            contract, one insert_min per pick.
//   compact  a block per tile of positions finalises the first-occurrence bits (hop 0, whose
//            seed list may repeat ids, asks the table; later hops look at the lost marks),
//            learns how many first occurrences lie in the tiles before (lookback.h), ranks its
//            own, appends them to the frontier and records the rank at the position.
// Off the critical path, as surplus blocks: the rows' pick counts are scanned (in the compact launch),
// and the packed edge list (src_local, dst_local) is written (in the next hop's fill; rank of a pick =
// rank recorded at its id's smallest position, which the pick met when it was inserted or finds by links:
// the table is not read again).
// A small batch is one launch of one block instead of all this (one_block.h).
//
// These kernels are chains of dependent memory accesses, so what a thread will need is requested
// as early as its address is known: a hop's length lives in device memory, but every buffer has
// its worst-case size, so a thread asks for its own elements (inside the buffer whatever the
// length turns out to be) together with the length and only then decides whether they count.
#include <string.h>

#include <algorithm>
#include <type_traits>

#include "buckets.h"
#include "choose.h"
#include "common.h"
#include "edges.h"
#include "lookback.h"
#include "one_block.h"
#include "picks.h"
#include "table.h"

namespace dgs {
namespace {

constexpr int kBlock = 256;
static_assert(kBlock == kEdgeBlock, "edge lists are written by surplus blocks of the fills");
constexpr int kRowItems = 4;                   // rows a thread of a compact block takes
// What a compact block's tile is, by the hop's worst case: NT threads x ITEMS consecutive positions x
// GROUPS.  A few hundred tiles at most for the look-back (see lookback.h), but no fewer blocks than a
// short list can use: hop 0 reads the table at random, and two CUs alone take 6 us longer over 6 k
// positions than twelve.  Blocks of four waves as far as it goes: beside other batches' gathers, which
// free a CU's wave slots four at a time, blocks of eight wait (8 batches through the loader 1394 us
// against 1433).  Beyond 1.3 M positions eight-wave blocks, since a launch that loops has 512 blocks
// whatever their size.  us a call, short / middle / long tiles, by positions of its last hop: one hop
// 100 k 50.2 / 52.1 / 59.3, 131 k 60.7 / 59.7 / 65.4, 180 k 61.5 / 57.5 / 64.0, 1.2 M 172 / 123.9 / 120.9,
// 2.1 M 274 / 186 / 182; two hops (short, middle, and the rule's own choice, which takes shorter tiles for
// the first one) 131 k 63.2 / 65.8 / 63.7, 180 k 69.1 / 69.3 / 64.6, 1.2 M 189 / 137.5 / 137.9, 2.1 M 277 /
// 182 / 179.
enum PosTile { kShortTile, kMiddleTile, kLongTile };  // NT x ITEMS x GROUPS = 256 x 1 x 1, 256 x 4 x 4, 512 x 4 x 4
inline PosTile pos_tile_kind(int64_t len_max) { return len_max <= 131072 ? kShortTile : len_max <= 1310720 ? kMiddleTile : kLongTile; }
inline int64_t pos_tile_size(int64_t len_max) {
  const PosTile t = pos_tile_kind(len_max);
  return t == kShortTile ? 256 : t == kMiddleTile ? 4096 : 8192;
}
inline int64_t row_tile_size(int64_t len_max) { return (pos_tile_kind(len_max) == kLongTile ? 512 : 256) * kRowItems; }
constexpr int kMaxPosTile = 8192;
constexpr uint32_t kInvalidSlot = 0xffffffffu; // padded position that holds no pick
constexpr int kErrBucketOverflow = 8;          // hop flag bit: the ids of a bucket of the hashed pass did not fit its LDS table
constexpr int kMaxPicks = 64;
constexpr int64_t kMaxPositions = int64_t(1) << 30;
// Launches are sized for the worst case, which can exceed the real work many times over (a hub
// graph deduplicates heavily).  Grids are capped and blocks stride over the virtual block index,
// so a mostly empty worst case costs a few loop trips instead of 10^5 empty blocks.
constexpr int64_t kGridCap = 16384;
// A launch that loops anyway is given fewer blocks than the cap: its worst case is far beyond the
// work, and blocks that find none still take a slot each from whatever else shares the GPU
// (measured with batches in flight, 1024 / 2048 / 4096 / 16384 blocks: 111 M-node graph 0.169-0.180 /
// 0.167-0.178 / 0.165-0.169 / 0.183-0.187 ms per step, R-MAT [50,50] 0.342-0.352 / 0.345-0.356 /
// 0.343-0.353 / 0.357-0.361; a batch alone is level or 2 % faster).
constexpr int64_t kLoopGrid = 4096;
// A compact launch that loops keeps to blocks that fit the GPU all at once: a tile's block waits for the
// tiles before it (a bounded wait, see lookback.h), so those should not queue behind it for a slot.
constexpr int64_t kLookbackGrid = 512;
inline int64_t grid_cap() {
  const int64_t forced = debug_option(DGS_DEBUG_SAMPLER_GRID_CAP);
  return forced > 0 ? forced : kGridCap;
}
inline uint32_t capped_grid(int64_t virtual_blocks) {
  const int64_t cap = grid_cap();
  if (virtual_blocks <= cap) return uint32_t(virtual_blocks < 1 ? 1 : virtual_blocks);
  return uint32_t(cap < kLoopGrid ? cap : kLoopGrid);  // (a forced cap below kLoopGrid is the grid itself)
}
inline bool is_capped(int64_t virtual_blocks) { return virtual_blocks > grid_cap(); }
// Kernels come in two flavours: STRIDE = false runs exactly one virtual block per block (the
// common, uncapped launch, with no loop in the instruction stream), STRIDE = true strides.
#define DGS_FOR_VIRTUAL_BLOCKS(vb, total)                                                       \
  for (int64_t vb = blockIdx.x; vb < (total); vb += STRIDE ? int64_t(gridDim.x) : (total))

struct Hop {
  const void* seeds;        // seed ids: caller's seeds (hop 0) or the frontier array
  // The three device scalars below are read without a test in front of them, so that the reads
  // leave together with a thread's first own reads: the pointers name readable words in every
  // hop, also where the value is not used (hop 0 takes its count from n_seeds_host and has no
  // previous hop).
  const int64_t* n_seeds;   // device scalar: seeds of this hop (used when n_seeds_host < 0)
  int64_t n_seeds_host;     // hop 0: the caller's count; later hops: -1
  int64_t* n_seeds_out;     // hop 0: where to publish n_seeds on the device
  const int64_t* prev_nnz;      // device scalar: edges of the previous hop
  const int64_t* prev_n_seeds;  // device scalar: seeds of the previous hop
  int64_t* n_unique;        // device scalar: frontier size after this hop
  int64_t* nnz;             // device scalar: edges of this hop
  int64_t* flags;           // device scalar: bit 0 degree, bit 1 seed id, bit 2 picked id of a bad row
  int64_t* host_sizes;      // optional pinned mirror of the whole sizes array (NULL: none)
  int32_t n_hops;           // layout of the mirror: [0..H] seeds, then H edge counts, then H flags
  int32_t look_polls;       // lookback_polls()
  uint32_t* row_cnt;        // [s_max] picks of every row (kBadRow on error)
  uint32_t* row_off;        // [s_max] first packed edge of the row
  tile_state* row_state;    // [row tiles] the tiles' edge counts, in the course of their scan
  uint32_t* slot;           // [all positions] what is known of a position's id (see edges.h)
  uint32_t* rank_at;        // [all positions] rank of the id first seen there; of a lost position: a smaller one | kLinkBit
  uint8_t* lost;            // [all positions] non-zero: a smaller position of the same id exists
  int64_t* long_rows;       // weighted only: ranks of the frontier's rows of more than kLongRow positions ...
  int64_t* long_count;      // ... and how many there are, one array for all hops but the first
  uint8_t* long_seeds;      // weighted only, hop 0: the long ones of every kSeedSegment seeds ...
  int32_t* long_seed_count; // ... and how many there are
  tile_state* pos_state;    // [position tiles of this hop] first occurrences, in the course of their scan
  void* frontier;           // growing array of distinct ids
  void* src_local;          // out [nnz]
  void* dst_local;          // out [nnz]
  int64_t s_max;
  int64_t pos_base;         // first position of this hop (P_h)
  int64_t len_max;          // positions of this hop in the worst case: (hop 0: s_max) + s_max * k
  int32_t k;
  int32_t index;            // hop number
  uint32_t rng_stream;
  int32_t bucketed;         // non-zero: first occurrences come from the bucketed pass (see below) ...
  int32_t pad1_;
  int64_t bucket_pos_cap;   // ... as long as the hop's padded positions (seeds * k) are no more than this: decided on the device
  const int* bucket_overflow;  // set by the pass when a bucket held more ids than its LDS table takes (the call fails)
  dgs_view indptr;          // weighted, where a hop follows: the offsets, for finding its long rows
  int64_t n_edges;
};

__device__ __forceinline__ int64_t seeds_of(const Hop& h) { return count_of(h.n_seeds, h.n_seeds_host); }
// Whether this hop finds its first occurrences by the bucketed pass.  Its worst case may be far
// beyond what the pass has room for (it grows with the product of the fanouts, the hop does not),
// so the host only says whether the hop is eligible and every kernel decides from the hop's real
// length, the same way.  (A bucketed hop is never hop 0: its positions are seeds * k.)
__device__ __forceinline__ bool bucketed_now(const Hop& h, int64_t s) {
  return h.bucketed != 0 && s * h.k <= h.bucket_pos_cap;
}
// the first seed_part positions of hop 0 are the caller's seeds themselves
__device__ __forceinline__ int64_t seed_part(const Hop& h, int64_t s) { return h.index == 0 ? s : 0; }
// rank of the first id this hop can add: later hops append behind their seeds
__device__ __forceinline__ int64_t first_rank(const Hop& h, int64_t s) { return h.index == 0 ? 0 : s; }
// the wave-local search for repeated draws of a row (fill_rows): entries per wave, and the longest
// row, in multiples of the fanout, that is searched (k draws from 4 k positions repeat one in nine)
constexpr int kFoldSlotBits = 7;
constexpr int kFoldSlots = 1 << kFoldSlotBits;
constexpr int kFoldMaxRowPerPick = 4;

// ---- a large last hop without memory-side atomics -------------------------------------------
// The atomicMin per pick is what a large hop costs most (every device-scope atomic executes at
// the memory side: 26.7 G/s, 31 us for the 832 k picks of a 1024 x [5,10,15] batch, and as much
// again while other batches share the GPU).  The last hop needs no table entry afterwards, so its
// first occurrences can be found without the table (buckets.h).  The hop's units are the ids the frontier
// already holds, their number rounded up to a multiple of 16, then the padded positions.  The fill leaves
// the picked ids in the slot words; the compact launch has every pick's smallest unit from the pass: its own
// (a first occurrence), that of an id the frontier held before this hop (its rank | kRankBit: final, no further
// lookup), or that of an earlier pick of this hop (whose position becomes the slot word, and whose rank
// the compaction records there).  A draw that repeats another one of its row is no unit: its slot word is that
// draw's position from the fill on, where it finds a rank, or the link to one; nor is a pick of an id that its tile holds again and
// again (sort_tile), whose slot word becomes the first one's position or rank.  Same result as the table gives.
//
// It takes two launches more than the table does, and pays where the hop is large (by its worst case: that is what the
// host knows) and the table beyond the caches.  us a batch with rows of 64 bytes, table / pass: 2.4 M nodes, fanouts
// [5,10,15], 640 seeds (0.63 M picks at most) 83 / 87, 768 85 / 88, 896 (0.89 M) 89 / 89; 4 M nodes, [5,10] from 16 384
// seeds (0.98 M) 100 / 90, [5,10,15] from 2048 (2.0 M) 127 / 112, from 4096 228 / 193; 16 M nodes 103 / 94, 135 / 120,
// 259 / 226.  Small graphs repeat their ids, and the table sits in the caches: 2048 and 4096 seeds, 100 k nodes 97 /
// 100 and 112 / 122, 250 k 106 / 103 and 133 / 135, 500 k 115 / 103 and 157 / 140.  8 batches through the loader,
// 400-byte rows, 2.4 M nodes: 512 seeds 737 / 772, 768 823 / 842, 1024 995 / 971, 2048 1679 / 1570; 20 M nodes,
// 64-byte rows, 1024 seeds 675 / 690.
// That is for graphs whose rows leave many of the positions empty, which the pass goes over all the same.  Where the mean degree is
// twice the fanout it pays earlier, the more so the wider the rows that are gathered behind it or beside it.  The same, table / the
// pass before it had tiles of 8192 units / pass: 2.4 M nodes of 50 neighbours, 400-byte rows, a batch of 640 seeds
// 136 / 140 / 133, 704 (0.7 M) 145 / 147 / 139, 896 181 / 180 / 168, 8 through the loader 1033 / 1024 / 1010, 1065 / 1066 /
// 1065, 1262 / 1233 / 1221; 512-byte rows, 704 seeds 156 / 157 / 146 and 1169 / 1098 / 1107; 64-byte rows 101 / 107 / 101;
// 8 M nodes of 50 neighbours, 256-byte rows, 704 122 / 127 / 117; 35 neighbours, 400-byte rows, 704 128 / 134 / 127; 25 108 / 117 / 111,
// 896 123 / 131 / 125; 16 M nodes of 19, 64-byte rows, 704 91 / 109 / 104; draws, 50 neighbours, 704 115 / 123 / 114.
constexpr int64_t kBucketedMinNodes = 262144, kBucketedMaxNodes = 16777216;
constexpr int64_t kBucketedMinPicks = 917504, kBucketedMinPicksFull = 655360;
static_assert(kBucketedMaxNodes <= kDirectMaxIds, "the direct form takes them");
// Larger graphs stay on the table: the hashed form (test hook) goes over every position, with a pick or without, and a
// hub's draws are one block's work.  us a batch of draws, 64-byte rows, table / hashed pass: 20 M nodes of 15 neighbours,
// fanouts [5,10,15] from 4096 seeds 225 / 212, with a node that 5 % of the edges lead to 306 / 371, 50 % 205 / 480; 60 M
// nodes, [50,50] from 8192 316 / 383; R-MAT of 2^26 nodes, [50,50] from 16 384 368 / 356.  Nothing that the host knows tells
// the last one from the others.  Without replacement, 111 M nodes, 0.94 M picks in 2.8 M positions: 215 / 216.
__host__ __device__ __forceinline__ int64_t front_units(int64_t s) { return (s + 15) / 16 * 16; }

// rank of the id at position p of hop 0, given p's slot word
template <typename TableT>
__device__ __forceinline__ uint32_t rank_of(const Hop& h, const TableT& table, int64_t p, uint32_t slot_word) {
  if (slot_word & kFirstBit) return h.rank_at[p];
  return h.rank_at[table.value(slot_word)];  // smallest position of the id: a first occurrence
}

template <int NT, typename T>
__device__ __forceinline__ T block_sum(T v, T* lds /* NT/64 */) {
#pragma unroll
  for (int d = kWave / 2; d > 0; d >>= 1) v += __shfl_xor(v, d, kWave);
  if ((threadIdx.x & (kWave - 1)) == 0) lds[threadIdx.x / kWave] = v;
  __syncthreads();
  T s = 0;
#pragma unroll
  for (int w = 0; w < NT / kWave; ++w) s += lds[w];
  __syncthreads();
  return s;
}

// ---- packed edge list of one hop (off the critical path) -----------------------------

// One block per NT * kRowItems rows: scan of the rows' pick counts.  The block of the last row publishes the
// hop's edge count and error bits; in a hop without rows (every id before it was refused) tile 0 does.
template <int NT, bool EARLY>
__device__ __forceinline__ void offsets_tile(const Hop& h, int64_t tile) {
  constexpr int64_t kRows = NT * kRowItems;
  __shared__ int lds[NT / kWave];
  __shared__ LookbackLds<NT> look;
  __shared__ int bad;
  const int64_t s = seeds_of(h);
  if (!EARLY && tile != 0 && tile * kRows >= s) return;
  const int64_t i = tile * kRows + threadIdx.x * kRowItems;
  uint32_t rc[kRowItems];
#pragma unroll
  for (int j = 0; j < kRowItems; ++j) rc[j] = i + j < h.s_max ? h.row_cnt[i + j] : 0u;  // requested together with s
  if (tile != 0 && tile * kRows >= s) return;  // whole blocks leave together
  if (threadIdx.x == 0) bad = 0;
  __syncthreads();
  int c = 0;
#pragma unroll
  for (int j = 0; j < kRowItems; ++j) {
    if (i + j >= s) rc[j] = 0;
    if (is_bad_row(rc[j])) {
      atomicOr(&bad, 1 << (kBadRow - rc[j]));
      rc[j] = 0;
    }
    c += int(rc[j]);
  }
  int total;
  const int ex = block_exclusive_scan<NT, int>(c, &total, lds);
  const tile_state own = tile_word(total, uint32_t(bad));
  const tile_state before = tile_exclusive_prefix<NT, true>(h.row_state, tile, own, h.look_polls, look, [&](int64_t t) {
    __syncthreads();
    if (threadIdx.x == 0) bad = 0;
    __syncthreads();
    int n = 0;
    for (int j = 0; j < kRowItems; ++j) {  // (a tile before this one is full)
      const uint32_t r = h.row_cnt[t * kRows + j * NT + threadIdx.x];
      if (is_bad_row(r)) atomicOr(&bad, 1 << (kBadRow - r)); else n += int(r);
    }
    const int sum = block_sum<NT, int>(n, lds);
    return tile_word(sum, uint32_t(bad));
  });
  uint32_t off = uint32_t(tile_sum_of(before)) + uint32_t(ex);
#pragma unroll
  for (int j = 0; j < kRowItems; ++j) {
    if (i + j < s) h.row_off[i + j] = off;
    off += rc[j];
  }
  if ((tile + 1) * kRows >= s && threadIdx.x == 0) {
    const tile_state all = tile_add(before, own);
    int64_t flags = tile_flags_of(all);
    if (h.bucketed != 0 && *h.bucket_overflow != 0) flags |= kErrBucketOverflow;
    *h.nnz = tile_sum_of(all);
    *h.flags = flags;
    if (h.host_sizes) {
      mirror_to_host(h.host_sizes + h.n_hops + 1 + h.index, tile_sum_of(all));
      mirror_to_host(h.host_sizes + 2 * h.n_hops + 1 + h.index, flags);
    }
  }
}

__host__ __device__ __forceinline__ EdgeJob edge_job(const Hop& h) {
  EdgeJob e{};
  e.n_seeds = h.n_seeds;
  e.n_seeds_host = h.n_seeds_host;
  e.row_cnt = h.row_cnt;
  e.row_off = h.row_off;
  e.slot = h.slot;
  e.rank_at = h.rank_at;
  e.src_local = h.src_local;
  e.dst_local = h.dst_local;
  e.s_max = h.s_max;
  e.first = h.pos_base + (h.index == 0 ? h.n_seeds_host : 0);  // (the caller's count: positions hang on no load)
  e.bucket_pos_cap = h.bucketed != 0 ? h.bucket_pos_cap : -1;
  e.k = h.k;
  return e;
}
template <typename IdT, typename TableT, bool EARLY>
__device__ __forceinline__ void relabel_tile(const Hop& h, const TableT& table, int64_t b, int tid) {
  const EdgeJob e = edge_job(h);
  if (h.index != 0) {
    later_edge_tile<IdT, EARLY>(e, b, tid);
    return;
  }
  edge_tile<IdT, EARLY>(
      e, b, tid, [&](int64_t, uint32_t word, bool*) { return table.value(word); },
      [&](int64_t i) { return rank_of(h, table, h.pos_base + i, h.slot[h.pos_base + i]); });
}

// ---- critical path ------------------------------------------------------------------------

// Marks `displaced` (a position of this hop) as no longer the smallest of its id: p is smaller.
__device__ __forceinline__ void mark_lost(const Hop& h, uint32_t displaced, int64_t p) {
  h.lost[displaced] = 1;
  h.rank_at[displaced] = uint32_t(p) | kLinkBit;
}

// The slot word of padded position p, which holds a pick of neighbour id `col`: the id goes into
// the table (or, in a bucketed hop, into the word itself).  Returns false, and the word of an empty
// position, when the id is one the table cannot hold (the caller marks the row bad): the id is
// checked before it addresses anything.
template <typename IdT, typename TableT>
__device__ __forceinline__ bool place_pick(const Hop& h, const TableT& table, IdT col, int64_t p, bool look_first,
                                           bool bucketed, uint32_t* word) {
  *word = kInvalidSlot;
  if (!table.holds(col)) return false;
  if (bucketed) {
    *word = uint32_t(col) | kFirstBit;  // a first occurrence until the bucketed pass says otherwise; the table is left alone
    return true;
  }
  bool first;
  uint32_t met;
  uint32_t w = table.insert_min(col, uint32_t(p), &first, &met, look_first);
  if (h.index != 0) {
    if (first && met != kNoPosition) mark_lost(h, met, p);
    w = first ? (w | kFirstBit) : met;  // (the bit is provisional: void once the position is marked lost)
  }
  *word = w;
  return true;
}

// What becomes of padded position p: with a pick (edge `edge` of the graph) the picked id is placed
// and p's slot word recorded; without one the position is marked empty.
template <typename IdT, typename TableT>
__device__ __forceinline__ bool emit_pick(const Hop& h, const TableT& table, const TierView<IdT>& indices, int64_t p,
                                          bool have, int64_t edge, bool look_first, bool bucketed) {
  uint32_t word = kInvalidSlot;
  bool ok = true;
  if (have) ok = place_pick<IdT>(h, table, indices.at(edge), p, look_first, bucketed, &word);
  h.slot[p] = word;
  return ok;
}

// Ids that repeat a lot (hub sources) are cheaper to insert with a look at the entry first;
// the previous hop tells: if more than a fifth of its picks were not new ids, look first.
// (hop 0 has no history: look first only when it is big enough for contention to matter)
__device__ __forceinline__ bool look_before_insert(const Hop& h, int64_t s) {
  const int64_t picked = *h.prev_nnz;
  const int64_t fresh = s - *h.prev_n_seeds;  // ids the previous hop added to the frontier
  const bool first_hop = h.index == 0;
  const bool big = s * h.k >= (int64_t(1) << 17);
  const bool repeats = fresh * 5 < picked * 4;
  return bool((int(first_hop) & int(big)) | (int(!first_hop) & int(repeats)));
}

// One virtual block of the fill launch: 256 / G seed rows.
template <typename IdT, typename PtrT, typename TableT, int G, bool EARLY>
__device__ __forceinline__ void fill_rows(const Hop& h, int64_t vb, const TableT& table,
                                          const TierView<PtrT>& indptr, const TierView<IdT>& indices,
                                          bool replace, uint64_t rng_seed) {
  const int64_t gid = vb * kBlock + threadIdx.x;
  const int64_t i = gid / G;
  const int l = int(gid % G);
  // a launch sized far beyond the hop: blocks past its end wait for nothing but the length
  if (!EARLY && vb != 0 && vb * (kBlock / G) >= seeds_of(h)) return;
  // the wave's table for the search for repeated draws (below) is emptied here, where every lane
  // of the wave is still present
  __shared__ unsigned long long fold_lds[kBlock / kWave][kFoldSlots];
  if (replace) {
    unsigned long long* offers = fold_lds[threadIdx.x / kWave];
#pragma unroll
    for (int q = 0; q < kFoldSlots / kWave; ++q) offers[q * kWave + (threadIdx.x & (kWave - 1))] = ~0ull;
  }
  // the hop's length, what the previous hop found, and this group's seed id, requested together
  // (the seed list has room for s_max ids whatever the length turns out to be)
  const IdT seed = i < h.s_max ? static_cast<const IdT*>(h.seeds)[i] : IdT(0);
  const int64_t s = seeds_of(h);
  const bool look_first = look_before_insert(h, s);
  const bool bucketed = bucketed_now(h, s);
  if (h.n_seeds_out && vb == 0 && threadIdx.x == 0) *h.n_seeds_out = s;
  if (i >= s) return;  // whole groups leave together
  const int group_lane0 = (threadIdx.x & (kWave - 1)) - l;
  const int64_t row = int64_t(seed);
  // this lane's random block hangs on the ids only: computed while the offsets are on their way
  const PhiloxWords words = philox_draw_words(rng_seed, h.rng_stream, row, uint32_t(l));
  // nothing is addressed by an id or an offset before it has been checked
  const bool seed_ok = row_in_range(indptr, row) && table.holds(seed);
  int64_t b = 0, deg64 = 0;
  if (seed_ok) {
    b = int64_t(indptr.at(row));
    deg64 = int64_t(indptr.at(row + 1)) - b;
  }
  const bool bad = deg64 < 0 || deg64 > 0xffffffffLL || b < 0 || b + deg64 > indices.n;
  const uint32_t deg = bad ? 0u : uint32_t(deg64);
  const int k = h.k;
  if (l == 0 && h.index == 0) {  // the caller's seeds open the mapping list; compact_tile decides their first bits
    bool first;
    uint32_t displaced;
    h.slot[h.pos_base + i] =
        seed_ok ? table.insert_min(seed, uint32_t(h.pos_base + i), &first, &displaced) : kInvalidSlot;
  }
  uint32_t pos;
  const bool have = pick_position<G>(deg, k, replace, l, group_lane0, words, &pos);
  const bool live = l < k && have;
  const int64_t p = h.pos_base + seed_part(h, s) + i * k + l;
  // Draws with replacement repeat positions: on a row shorter than k most slots do.  Only the
  // lowest slot of each position reads the edge array and goes to the table; a repeat can never be
  // its id's smallest position, so it takes its leader's slot word, or position where that may be the
  // first, and touches nothing.  Repeats are found through a small table of the wave's own in LDS: every
  // slot of the row offers (position, lane) to the entry its position hashes to, the smallest
  // offer stays, and a slot that then reads its own position with a lower lane of its row has found
  // its leader.  Two positions that meet in one entry cost a missed repeat, never a wrong one.
  // Long rows (whose draws rarely repeat) skip the search.
  int leader = l;
  if (replace) {
    unsigned long long* offers = fold_lds[threadIdx.x / kWave];
    const int lane = threadIdx.x & (kWave - 1);
    const bool search = live && deg <= uint32_t(kFoldMaxRowPerPick * k);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint32_t entry = ((pos + uint32_t(group_lane0) * 0x9E3779B1u) * 0x85EBCA6Bu) >> (32 - kFoldSlotBits);
    if (search) atomicMin(&offers[entry], (static_cast<unsigned long long>(pos) << 8) | uint32_t(lane));
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (search) {
      const unsigned long long best = offers[entry];
      const int best_lane = int(best & 255u);
      if (uint32_t(best >> 8) == pos && best_lane < lane && best_lane >= group_lane0) leader = best_lane - group_lane0;
    }
  }
  uint32_t word = kInvalidSlot;
  bool pick_ok = true;
  if (live && leader == l) pick_ok = place_pick<IdT>(h, table, indices.at(b + pos), p, look_first, bucketed, &word);
  if (replace) {
    const uint32_t leader_word = __shfl(word, leader, G);
    const int leader_ok = __shfl(int(pick_ok), leader, G);
    if (live && leader != l) {
      word = leader_word == kInvalidSlot ? kInvalidSlot
           : h.index != 0 && (leader_word & kFirstBit) ? uint32_t(p - l + leader) : (leader_word & ~kFirstBit);
      pick_ok = leader_ok != 0;
    }
  }
  if (l < k) h.slot[p] = word;
  constexpr uint64_t group_mask = G == 64 ? ~uint64_t(0) : ((uint64_t(1) << (G & 63)) - 1);
  const bool picks_ok = ((__ballot(!pick_ok) >> group_lane0) & group_mask) == 0;
  if (l == 0)
    h.row_cnt[i] = !seed_ok ? kBadSeed : bad ? kBadRow : !picks_ok ? kBadPick
                 : (replace ? (deg == 0 ? 0u : uint32_t(k)) : (deg < uint32_t(k) ? deg : uint32_t(k)));
}

// Virtual blocks [0, fill_blocks): seed rows of this hop; then relabel_count blocks writing the
// previous hop's edge list (off the critical path); then, in hop 0's launch, blocks clearing the
// lost marks of the later hops.
template <typename IdT, typename PtrT, typename TableT, int G, bool STRIDE>
__global__ __launch_bounds__(kBlock) void hop_fill_kernel(Hop h, Hop prev, int64_t fill_blocks,
                                                          int64_t relabel_count, uint4* clear_begin,
                                                          int64_t clear_n16, TableT table, TierView<PtrT> indptr,
                                                          TierView<IdT> indices, bool replace, uint64_t rng_seed) {
  const int64_t clear_blocks = (clear_n16 + kBlock - 1) / kBlock;
  const int64_t total = fill_blocks + relabel_count + clear_blocks;
  DGS_FOR_VIRTUAL_BLOCKS(vb, total) {
    if (vb < fill_blocks) {
      fill_rows<IdT, PtrT, TableT, G, !STRIDE>(h, vb, table, indptr, indices, replace, rng_seed);
    } else if (!STRIDE && vb < fill_blocks + relabel_count) {  // (a striding launch is given no such blocks)
      relabel_tile<IdT, TableT, !STRIDE>(prev, table, vb - fill_blocks, threadIdx.x);
    } else {
      const int64_t i = (vb - fill_blocks - relabel_count) * kBlock + threadIdx.x;
      if (i < clear_n16) clear_begin[i] = make_uint4(0u, 0u, 0u, 0u);
    }
  }
}

// ---- weighted picks (choose.h) ----
//
// In a large hop a block takes up to choose_rows(k) rows: a thread looks each of them up, the block chooses their picks,
// and then every pick is placed by a thread of its own.  Rows above kLongRow positions are raced, or drawn
// from, by a whole block each.  They are queued before the launch, by the compact launch of the hop before
// (announce_long_rows) or, in hop 0, by the launch that clears (announce_long_seeds), so that they are
// worked on from its first moment, beside the others.
// A small hop (kSharedMaxRows) is a launch of larger blocks instead, with a wave for each row and as few rows to a
// block as still give every CU one: nothing waits at a barrier but the long rows, which the block takes one after
// the other at the end.  In hop 0 that reaches further (kSharedMaxSeeds): it saves the launch that queues.
// us a call of one hop, small / queued form: 4000 rows of 50 / 200 / 1000, 64 picks 64 / 71, 75 / 99, 84 / 114;
// 8192 rows of 10 / 50 / 1000 52 / 56, 58 / 62, 75 / 114; 12 000 of 200 77 / 99; 12 288 of 30 64 / 63 (draws 71 /
// 62, but 8192 of 50 61 / 59 and of 1000 67 / 117); 65 536 of 20 150 / 90.  1024 seeds, fanouts [5,10]: 101 / 107.
// The launch alone, 256 rows of 60 / 512 / 1000 / 2048 / 4000 / 17 000 positions, 5 picks: by a wave and, beyond
// 2048, a block 6.9 / 9.6 / 12.1 / 14.8 / 18.0 / 21.2 us.  With the phases of fill_rows_weighted here too, and a
// block's turn from 512 on, 9.3 / 13.1 / 16.8 / 18.8 / 21.3 / 25.0; with sorts of 64-bit keys (a wave up to 512)
// 7.7 / 12.6 / 13.5 / 14.7 / 15.9 / 29.8, and with 15 picks 16.4 / 15.9 / 18.6 / 23.0 / 37.8 where it is now 10.9 /
// 12.2 / 14.8 / 19.3 / 23.3: 1500 to 5000 positions and few picks are the one place that has lost (1 to 2 us).
// kLongRow 512 / 1024 / 2048: 287 / 278 / 276 us for a batch of 1024 seeds, fanouts [5,10,15].
constexpr uint32_t kLongRow = 2048;
static_assert(kLongRow <= kDrawRow && kLongRow <= kWaveDrawRow, "draw_rows and draw_by_wave take every row that is not long");
constexpr int64_t kMinQueueBlocks = 256, kMaxQueueBlocks = 512;  // (see queue_blocks)
constexpr int64_t kSharedMaxRows = 4096, kSharedMaxSeeds = 12288;  // of a later hop, of hop 0
constexpr int64_t kSharedBlocks = 256;  // one per CU
constexpr int kSharedRows = kLongBlock / kWave;  // a wave for each
constexpr int kSeedSegment = 256;       // seeds of one list of long rows in hop 0

// A seed row as one thread looks it up.
template <typename IdT>
struct WeightedRow {
  int64_t b;      // its first edge
  uint32_t deg;   // 0: nothing to pick
  IdT seed;
  bool seed_ok, bad;
  __device__ __forceinline__ bool chosen(int k, bool replace) const { return deg > 0 && (replace || deg > uint32_t(k)); }
};
template <typename IdT, typename PtrT, typename TableT>
__device__ __forceinline__ WeightedRow<IdT> look_up_row(bool is_row, IdT seed, const TableT& table, const TierView<PtrT>& indptr,
                                                        const TierView<IdT>& indices) {
  WeightedRow<IdT> r{0, 0u, IdT(0), true, false};
  if (is_row) {
    r.seed = seed;
    // nothing is addressed by an id or an offset before it has been checked
    r.seed_ok = row_in_range(indptr, int64_t(r.seed)) && table.holds(r.seed);
    int64_t deg64 = 0;
    if (r.seed_ok) {
      r.b = int64_t(indptr.at(int64_t(r.seed)));
      deg64 = int64_t(indptr.at(int64_t(r.seed) + 1)) - r.b;
    }
    r.bad = deg64 < 0 || deg64 > 0xffffffffLL || r.b < 0 || r.b + deg64 > indices.n;
    r.deg = r.bad ? 0u : uint32_t(deg64);
  }
  return r;
}

template <int NT, bool REPLACE>
struct ChooseLds {
  std::conditional_t<REPLACE, DrawRowsLds<NT>, RaceRowsLds<NT>> rows;
  uint32_t picks[kChooseRows];     // picks that the row has here; those of a long row come from somebody else
  uint32_t bad_pick[kChooseRows];
};
constexpr uint32_t kElsewhere = 0xffffffffu;

// The picks of the hop's rows [first, first + rows) but the long ones, by a whole block.
template <typename IdT, typename PtrT, typename TableT, bool REPLACE, int NT>
__device__ __forceinline__ void fill_rows_weighted(const Hop& h, int64_t s, int64_t first, int rows,
                                                   ChooseLds<NT, REPLACE>& lds, const TableT& table,
                                                   const TierView<PtrT>& indptr, const TierView<IdT>& indices,
                                                   const TierView<float>& probs, uint64_t rng_seed) {
  const int k = h.k;
  const bool look_first = look_before_insert(h, s);
  const bool bucketed = bucketed_now(h, s);
  if (int64_t(rows) > s - first) rows = int(s - first);
  const int t = threadIdx.x;
  WeightedRow<IdT> own;
  clear_entries(lds.rows, rows, k);
  if (t < kWave) {
    own = look_up_row<IdT, PtrT>(t < rows, t < rows ? static_cast<const IdT*>(h.seeds)[first + t] : IdT(0), table, indptr, indices);
    const bool chosen = k > 0 && own.chosen(k, REPLACE);
    const bool is_long = chosen && own.deg > kLongRow;
    set_row(lds.rows, own.b, int64_t(own.seed), chosen && !is_long ? own.deg : 0u);
    if (t < kChooseRows) {
      lds.picks[t] = is_long ? kElsewhere : chosen ? uint32_t(k) : REPLACE || k == 0 ? 0u : own.deg;
      lds.bad_pick[t] = 0;
    }
    if (t < rows && h.index == 0) {  // the caller's seeds open the mapping list
      bool first_seen;
      uint32_t displaced;
      h.slot[h.pos_base + first + t] =
          own.seed_ok ? table.insert_min(own.seed, uint32_t(h.pos_base + first + t), &first_seen, &displaced) : kInvalidSlot;
    }
  }
  __syncthreads();
  const int64_t p0 = h.pos_base + seed_part(h, s) + first * k;
  if (k == 0) {  // nothing to choose (a zero fanout)
  } else if constexpr (REPLACE) {
    draw_rows<NT>(lds.rows, rows, k, probs, rng_seed, h.rng_stream, [&](int r, int j, uint32_t pos) {
      if (!emit_pick<IdT>(h, table, indices, p0 + int64_t(r) * k + j, true, lds.rows.begin[r] + pos, look_first, bucketed))
        lds.bad_pick[r] = 1;
    });
  } else {
    race_rows<NT>(lds.rows, rows, k, probs, rng_seed, h.rng_stream);
  }
  // two picks a thread at a time, so that their ids are on their way together
  constexpr int kAhead = 2;
  int r = k > 0 ? t / k : rows, l = k > 0 ? t % k : 0;
  while (r < rows) {
    int at_row[kAhead], at_slot[kAhead];
    bool here[kAhead], have[kAhead];
    IdT id[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      at_row[u] = r;
      at_slot[u] = l;
      here[u] = have[u] = false;
      id[u] = IdT(0);
      if (r < rows) {
        const uint32_t n = lds.picks[r];
        here[u] = n != kElsewhere && !(REPLACE && n != 0);
        have[u] = here[u] && uint32_t(l) < n;
        uint32_t pos = uint32_t(l);  // copied rows keep their positions in order
        if constexpr (!REPLACE)
          if (have[u] && lds.rows.deg[r] != 0) pos = lds.rows.entry_pos[r * (k + 1) + l];
        if (have[u]) id[u] = indices.at(lds.rows.begin[r] + pos);
      }
      r += NT / k;
      l += NT % k;
      if (l >= k) {
        l -= k;
        ++r;
      }
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      if (!here[u]) continue;
      const int64_t p = p0 + int64_t(at_row[u]) * k + at_slot[u];
      uint32_t word = kInvalidSlot;
      if (have[u] && !place_pick<IdT>(h, table, id[u], p, look_first, bucketed, &word)) lds.bad_pick[at_row[u]] = 1;
      h.slot[p] = word;
    }
  }
  __syncthreads();
  if (t < rows && lds.picks[t] != kElsewhere)
    h.row_cnt[first + t] = !own.seed_ok ? kBadSeed : own.bad ? kBadRow : lds.bad_pick[t] != 0 ? kBadPick
                         : (REPLACE ? (own.deg == 0 ? 0u : uint32_t(k)) : (own.deg < uint32_t(k) ? own.deg : uint32_t(k)));
}

// The picks of one long row (a valid one: its edges are deg positions from b on), by a whole block.
template <int NT, bool REPLACE>
struct LongLds {
  std::conditional_t<REPLACE, DrawLongLds<NT>, RaceLongLds<NT>> row;
  int bad_pick;
};
template <typename IdT, typename TableT, bool REPLACE, int NT>
__device__ __forceinline__ void fill_long_row(const Hop& h, int64_t s, int64_t i, int64_t row, int64_t b, uint32_t deg,
                                              LongLds<NT, REPLACE>& lds, const TableT& table, const TierView<IdT>& indices,
                                              const TierView<float>& probs, uint64_t rng_seed) {
  const bool look_first = look_before_insert(h, s);
  const bool bucketed = bucketed_now(h, s);
  const int k = h.k;
  const int64_t p0 = h.pos_base + seed_part(h, s) + i * k;
  if (threadIdx.x == 0) lds.bad_pick = 0;
  __syncthreads();
  if constexpr (REPLACE) {
    draw_long<NT>(lds.row, probs, b, deg, k, rng_seed, h.rng_stream, row, [&](int j, uint32_t pick) {
      if (!emit_pick<IdT>(h, table, indices, p0 + j, true, b + pick, look_first, bucketed)) lds.bad_pick = 1;
    });
  } else {
    const uint32_t pos = race_long<NT>(lds.row, probs, b, deg, k, rng_seed, h.rng_stream, row);
    const int l = threadIdx.x;  // wave 0 holds the winners
    if (l < k && !emit_pick<IdT>(h, table, indices, p0 + l, pos < deg, b + pos, look_first, bucketed)) lds.bad_pick = 1;
  }
  __syncthreads();
  if (threadIdx.x == 0) h.row_cnt[i] = lds.bad_pick != 0 ? kBadPick : uint32_t(k);
  __syncthreads();
}

// Hop 0's clearing, and the lists of its long rows: segment by segment, so that nothing has to be cleared
// before them.
template <typename IdT, typename PtrT>
__global__ __launch_bounds__(kSeedSegment) void announce_long_seeds_kernel(Hop h, int64_t segments, uint4* clear_begin,
                                                                           int64_t clear_n16, TierView<PtrT> indptr,
                                                                           int64_t n_edges) {
  if (int64_t(blockIdx.x) >= segments) {
    const int64_t i = (int64_t(blockIdx.x) - segments) * kSeedSegment + threadIdx.x;
    if (i < clear_n16) clear_begin[i] = make_uint4(0u, 0u, 0u, 0u);
    return;
  }
  __shared__ int found;
  if (threadIdx.x == 0) found = 0;
  __syncthreads();
  const int64_t i = int64_t(blockIdx.x) * kSeedSegment + threadIdx.x;
  if (i < h.n_seeds_host) {
    const int64_t row = int64_t(static_cast<const IdT*>(h.seeds)[i]);
    if (row_in_range(indptr, row)) {  // (bad rows are found by the fill)
      const int64_t b = int64_t(indptr.at(row)), deg = int64_t(indptr.at(row + 1)) - b;
      if (deg > int64_t(kLongRow) && deg <= 0xffffffffLL && b >= 0 && b + deg <= n_edges)
        h.long_seeds[int64_t(blockIdx.x) * kSeedSegment + atomicAdd(&found, 1)] = uint8_t(threadIdx.x);
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) h.long_seed_count[blockIdx.x] = found;
}

// Virtual blocks: the queued long rows, the others, the previous hop's edge list.
template <typename IdT, typename PtrT, typename TableT, bool REPLACE>
__global__ __launch_bounds__(kBlock, REPLACE ? 3 : 4) void hop_fill_weighted_kernel(Hop h, Hop prev, int64_t queue_blocks,
                                                                   int64_t fill_blocks, int32_t rows_per_block,
                                                                   int64_t relabel_count,
                                                                   TableT table, TierView<PtrT> indptr,
                                                                   TierView<IdT> indices, TierView<float> probs,
                                                                   uint64_t rng_seed) {
  __shared__ union {
    ChooseLds<kBlock, REPLACE> choose;
    LongLds<kBlock, REPLACE> long_row;
  } lds;
  const int64_t total = queue_blocks + fill_blocks + relabel_count;
  for (int64_t vb = blockIdx.x; vb < total; vb += gridDim.x) {
    if (vb >= queue_blocks + fill_blocks) {
      relabel_tile<IdT, TableT, false>(prev, table, vb - queue_blocks - fill_blocks, threadIdx.x);  // always a striding launch
      continue;
    }
    const int64_t s = seeds_of(h);
    if (vb < queue_blocks) {
      const auto take = [&](int64_t i) {
        const int64_t row = int64_t(static_cast<const IdT*>(h.seeds)[i]);
        if (!table.holds(IdT(row)) || h.k == 0) return;
        const int64_t b = int64_t(indptr.at(row));
        const uint32_t deg = uint32_t(int64_t(indptr.at(row + 1)) - b);  // queued rows have a valid degree
        fill_long_row<IdT, TableT, REPLACE, kBlock>(h, s, i, row, b, deg, lds.long_row, table, indices, probs, rng_seed);
      };
      if (h.index == 0) {  // several blocks share a segment's list where there are fewer segments than blocks
        const int64_t segments = (s + kSeedSegment - 1) / kSeedSegment;
        const int64_t at_once = segments < queue_blocks ? segments : queue_blocks;
        const int64_t sharers = queue_blocks / at_once, sharer = vb / at_once;
        if (sharer < sharers)
          for (int64_t g = vb % at_once; g < segments; g += at_once)
            for (int64_t j = sharer; j < h.long_seed_count[g]; j += sharers)
              take(g * kSeedSegment + h.long_seeds[g * kSeedSegment + j]);
      } else {
        const int64_t n_long = *h.long_count;
        for (int64_t t = vb; t < n_long; t += queue_blocks) take(h.long_rows[t]);
      }
    } else {
      const int64_t at = vb - queue_blocks;
      if (h.n_seeds_out && at == 0 && threadIdx.x == 0) *h.n_seeds_out = s;
      const int64_t first = at * rows_per_block;
      if (first >= s) continue;  // whole blocks leave together
      fill_rows_weighted<IdT, PtrT, TableT, REPLACE, kBlock>(h, s, first, rows_per_block, lds.choose, table, indptr, indices, probs,
                                                             rng_seed);
    }
    __syncthreads();  // lds is rewritten by the block's next rows
  }
}

// The picks of one row, by one wave (all of its lanes have looked the row up): a lane has a pick, and in hop 0 the
// lane behind them, or the first one afterwards, the seed, which opens the mapping list.
struct WaveRaceLds {
  __align__(16) WaveList list;
  uint32_t entry_key[kMaxWeightedPicks + 1], entry_pos[kMaxWeightedPicks + 1];
};
template <bool REPLACE> using WaveLds = std::conditional_t<REPLACE, WaveDrawLds, WaveRaceLds>;
template <typename IdT, typename TableT, bool REPLACE>
__device__ __forceinline__ void fill_row_weighted(const Hop& h, int64_t s, int64_t i, const WeightedRow<IdT>& own, WaveLds<REPLACE>& lds,
                                                  const TableT& table, const TierView<IdT>& indices, const TierView<float>& probs,
                                                  uint64_t rng_seed) {
  const bool look_first = look_before_insert(h, s);
  const bool bucketed = bucketed_now(h, s);
  const int k = h.k, l = threadIdx.x & (kWave - 1);
  const bool chosen = k > 0 && own.chosen(k, REPLACE);
  const uint32_t n = chosen ? uint32_t(k) : REPLACE || k == 0 ? 0u : own.deg;
  const int64_t b = wave_uniform(own.b), row = wave_uniform(int64_t(own.seed));
  const uint32_t deg = wave_uniform(own.deg);
  uint32_t pos = uint32_t(l);  // copied rows keep their positions in order
  if (chosen) {
    if constexpr (REPLACE) {
      pos = draw_by_wave(lds, probs, b, deg, k, rng_seed, h.rng_stream, row);
    } else {
      race_by_wave<true>(lds.list, lds.entry_key, lds.entry_pos, true, k, probs, b, deg, rng_seed, h.rng_stream, row);
      if (l < k) pos = lds.entry_pos[l];
    }
  }
  const int64_t p0 = h.pos_base + seed_part(h, s) + i * k;
  bool ok = true;
  const auto place = [&](bool is_seed) {
    uint32_t word = kInvalidSlot;
    const int64_t p = is_seed ? h.pos_base + i : p0 + l;
    if (is_seed ? own.seed_ok : uint32_t(l) < n)  // (a lane may place a pick and then the seed: neither hides the other's fault)
      ok &= place_pick<IdT>(h, table, is_seed ? own.seed : indices.at(b + pos), p, look_first, bucketed, &word);
    h.slot[p] = word;
  };
  const bool seed_too = h.index == 0;
  if (l < k + int(seed_too)) place(l == k);
  if (seed_too && k == kWave && l == 0) place(true);
  const uint64_t bad = __ballot(!ok);
  if (l == 0)
    h.row_cnt[i] = !own.seed_ok ? kBadSeed : own.bad ? kBadRow : bad != 0 ? kBadPick
                 : (REPLACE ? (deg == 0 ? 0u : uint32_t(k)) : (deg < uint32_t(k) ? deg : uint32_t(k)));
}

// A small hop: blocks [0, fill_blocks) have rows_per_block (at most kSharedRows) seed rows each; the blocks
// of the previous hop's edge list and of the clearing, of kBlock threads elsewhere, are taken four at a time.
template <typename IdT, typename PtrT, typename TableT, bool REPLACE>
__global__ __launch_bounds__(kLongBlock) void hop_fill_weighted_shared_kernel(Hop h, Hop prev, int64_t fill_blocks,
                                                                              int32_t rows_per_block,
                                                                              int64_t relabel_count, uint4* clear_begin,
                                                                              int64_t clear_n16, TableT table,
                                                                              TierView<PtrT> indptr,
                                                                              TierView<IdT> indices,
                                                                              TierView<float> probs, uint64_t rng_seed) {
  if (int64_t(blockIdx.x) >= fill_blocks) {
    const int64_t vb = (int64_t(blockIdx.x) - fill_blocks) * (kLongBlock / kBlock) + threadIdx.x / kBlock;
    const int tid = threadIdx.x & (kBlock - 1);
    if (vb < relabel_count) {
      relabel_tile<IdT, TableT, false>(prev, table, vb, tid);
    } else {
      const int64_t i = (vb - relabel_count) * kBlock + tid;
      if (i < clear_n16) clear_begin[i] = make_uint4(0u, 0u, 0u, 0u);
    }
    return;
  }
  struct Listed { int64_t row, begin; uint32_t deg; int at; };
  __shared__ union {
    WaveLds<REPLACE> wave[kSharedRows];
    LongLds<kLongBlock, REPLACE> long_row;
  } lds;
  __shared__ Listed listed[kSharedRows];
  __shared__ int n_listed;
  const int64_t first = int64_t(blockIdx.x) * rows_per_block;
  const int wave = int(wave_uniform(uint32_t(threadIdx.x / kWave)));
  const int64_t i = first + wave;
  // (asked for together with the hop's length: the seed list has room for s_max ids)
  const IdT seed = wave < rows_per_block && i < h.s_max ? static_cast<const IdT*>(h.seeds)[i] : IdT(0);
  const int64_t s = seeds_of(h);
  if (h.n_seeds_out && blockIdx.x == 0 && threadIdx.x == 0) *h.n_seeds_out = s;
  if (first >= s) return;  // whole blocks leave together
  if (threadIdx.x == 0) n_listed = 0;
  __syncthreads();
  const bool has_row = wave < rows_per_block && i < s;
  const WeightedRow<IdT> own = look_up_row<IdT, PtrT>(has_row, seed, table, indptr, indices);
  if (has_row && h.k > 0 && own.deg > kLongRow) {
    if ((threadIdx.x & (kWave - 1)) == 0) {
      listed[atomicAdd(&n_listed, 1)] = Listed{int64_t(own.seed), own.b, own.deg, wave};
      if (h.index == 0) {  // (while the other waves are at their rows)
        uint32_t word;
        place_pick<IdT>(h, table, own.seed, h.pos_base + i, false, false, &word);
        h.slot[h.pos_base + i] = word;
      }
    }
  } else if (has_row) {
    fill_row_weighted<IdT, TableT, REPLACE>(h, s, i, own, lds.wave[wave], table, indices, probs, rng_seed);
  }
  __syncthreads();
  const int n = n_listed;
  for (int t = 0; t < n; ++t) {
    const Listed r = listed[t];
    fill_long_row<IdT, TableT, REPLACE, kLongBlock>(h, s, first + int64_t(wave_uniform(uint32_t(r.at))), wave_uniform(r.row),
                                                    wave_uniform(r.begin), wave_uniform(r.deg), lds.long_row, table, indices,
                                                    probs, rng_seed);
  }
}

// ---- the bucketed pass (buckets.h) ----------------------------------------------------------

template <typename IdT, bool HASHED>
__global__ __launch_bounds__(kBucketBlock) void bucket_sort_kernel(Hop h, Buckets b) {
  __shared__ SortLds<HASHED, BucketShape> lds;
  if (blockIdx.x == 0 && threadIdx.x == 0) *b.overflow = 0;  // (the per-bucket launch comes behind this one)
  const int64_t s = wave_uniform(seeds_of(h));
  if (!bucketed_now(h, s)) return;  // the hop outgrew the pass: it runs on the table
  const uint32_t front = uint32_t(front_units(s)), units = front + uint32_t(s * h.k);
  const int log_buckets = log_buckets_of(b, units);
  uint32_t* slot = h.slot + h.pos_base;
  for (uint32_t tile = blockIdx.x; tile * kBucketTile < units; tile += gridDim.x) {
    uint32_t id[BucketShape::kItems];
#pragma unroll
    for (int j = 0; j < BucketShape::kItems; ++j) {
      const uint32_t u = tile * kBucketTile + uint32_t(j * kBucketBlock) + threadIdx.x;
      id[j] = u >= front && u < units ? nth(slot, u - front) : kNoId;  // (id | kFirstBit, or kInvalidSlot)
    }
    if (tile * kBucketTile < front) {
#pragma unroll
      for (int j = 0; j < BucketShape::kItems; ++j) {
        const uint32_t u = tile * kBucketTile + uint32_t(j * kBucketBlock) + threadIdx.x;
        if (u < uint32_t(s)) id[j] = uint32_t(nth(static_cast<const IdT*>(h.frontier), u));
      }
    }
#pragma unroll
    for (int j = 0; j < BucketShape::kItems; ++j)  // (a position's word: a draw that repeats one of its own row's, no unit)
      if (id[j] != kNoId) id[j] = tile * kBucketTile + uint32_t(j * kBucketBlock) + threadIdx.x < front ? id[j]
                                : (id[j] & kFirstBit) != 0 ? id[j] & ~kFirstBit : kNoId;
    sort_tile<HASHED, BucketShape>(b, log_buckets, tile, id, lds, [&](int j, uint32_t before) {  // (a pick: frontier ids are different ones)
      const uint32_t u = tile * kBucketTile + uint32_t(j * kBucketBlock) + threadIdx.x, met = tile * kBucketTile + before;
      if (u >= front) nth(slot, u - front) = met < front ? met | kRankBit : uint32_t(h.pos_base) + (met - front);
    });
    __syncthreads();  // lds is rewritten by the block's next tile
  }
}
static_assert(kInvalidSlot == kNoId, "a position without a pick is an entry without an id");

__global__ __launch_bounds__(kBucketBlock, 8) void bucket_first_kernel(Hop h, Buckets b) {
  __shared__ __align__(16) uint32_t best[kBucketRange];
  __shared__ uint32_t counts[kMaxBucketTiles];
  const int64_t s = wave_uniform(seeds_of(h));
  if (!bucketed_now(h, s)) return;
  const uint32_t front = uint32_t(front_units(s)), tiles = (front + uint32_t(s * h.k) + kBucketTile - 1) / kBucketTile;
  clear_counts(counts, tiles);
  for (int i = blockIdx.x; i < 1 << b.log_buckets; i += gridDim.x)
    first_of_bucket_direct(b, bucket_in_turn(i, b.log_buckets), tiles, front, best, counts);
  add_counts(b, counts, tiles);
}

__global__ __launch_bounds__(kBucketBlock) void bucket_first_hashed_kernel(Hop h, Buckets b) {
  __shared__ HashedLds lds;
  const int64_t s = wave_uniform(seeds_of(h));
  if (!bucketed_now(h, s)) return;
  const uint32_t front = uint32_t(front_units(s)), units = front + uint32_t(s * h.k), tiles = (units + kBucketTile - 1) / kBucketTile;
  const int log_buckets = log_buckets_of(b, units);
  clear_counts(lds.counts, tiles);
  for (int i = blockIdx.x; i < 1 << log_buckets; i += gridDim.x)
    if (!first_of_bucket_hashed(b, log_buckets, bucket_in_turn(i, log_buckets), tiles, front, lds) && threadIdx.x == 0) *b.overflow = 1;
  add_counts(b, lds.counts, tiles);
}

// Whether the position `rel` of the hop, of slot word `word`, is the first one of its id (`rel` is below
// the hop's length); the answer is the same before and after compact_tile has brought the word's bit
// up to date.
template <typename TableT>
__device__ __forceinline__ bool is_first(const Hop& h, const TableT& table, int64_t rel, uint32_t word, bool lost) {
  if (word == kInvalidSlot) return false;
  return h.index == 0 ? table.value(word & ~kFirstBit) == uint32_t(h.pos_base + rel) : (word & kFirstBit) != 0 && !lost;
}

// ITEMS consecutive words of an array as one load or store.
template <int ITEMS> struct Items;
template <> struct Items<1> {
  typedef uint32_t words __attribute__((ext_vector_type(1)));
  static __device__ __forceinline__ uint32_t load_marks(const uint8_t* p) { return *p; }
};
template <> struct Items<4> {
  typedef uint32_t words __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ uint32_t load_marks(const uint8_t* p) { return *reinterpret_cast<const uint32_t*>(p); }
};

// The first occurrences of one tile: counted, ranked, appended to the frontier.  A thread takes ITEMS
// consecutive positions of every group: their slot words, their lost marks and their ranks move as
// one load or store each, whether the positions count or not (the arrays reach a tile beyond the last
// position).  Bound: the chain of waits (length and words, the tiles before, the stores), 6 us at the
// floor; 13 bytes per position and 12 per first occurrence otherwise (2.1 M positions, 980 k of them
// first: 13 us).
template <typename IdT, typename TableT, int NT, int ITEMS, int GROUPS, bool EARLY>
__device__ __forceinline__ void compact_tile(const Hop& h, int64_t tile, const TableT& table, int64_t* begin, int64_t* end) {
  *begin = *end = 0;  // the ranks that the tile adds
  using words = typename Items<ITEMS>::words;
  constexpr int kWaves = NT / kWave;
  constexpr int kGroup = NT * ITEMS;
  constexpr int64_t kTile = int64_t(kGroup) * GROUPS;
  __shared__ LookbackLds<NT> look;
  __shared__ int wave_count[GROUPS * kWaves];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  // the hop's length and this thread's slot words (EARLY: requested together)
  const int64_t s = seeds_of(h);
  const int64_t len = seed_part(h, s) + s * h.k;
  if (!EARLY && tile != 0 && tile * kTile >= len) return;
  const int64_t base = tile * kTile + threadIdx.x * ITEMS;
  words word[GROUPS];
  uint32_t lost[GROUPS];
#pragma unroll
  for (int g = 0; g < GROUPS; ++g) {
    const int64_t p = h.pos_base + base + g * kGroup;  // a multiple of ITEMS
    word[g] = *reinterpret_cast<const words*>(h.slot + p);
    lost[g] = h.index != 0 ? Items<ITEMS>::load_marks(h.lost + p) : 0u;
  }
  if (tile != 0 && tile * kTile >= len) return;  // whole blocks leave together
  uint32_t first[GROUPS];   // bit j: position j of the group's is its id's first
  int lane_before[GROUPS];  // first positions in the lanes below
#pragma unroll
  for (int g = 0; g < GROUPS; ++g) {
    first[g] = 0;
    const int64_t rel = base + g * kGroup;
    if (h.index == 0) {  // is_first's question to the table for all positions at once (slot 0 stands in where there is none)
      uint32_t least[ITEMS];
#pragma unroll
      for (int j = 0; j < ITEMS; ++j) {
        if (rel + j >= len) word[g][j] = kInvalidSlot;
        least[j] = table.value(word[g][j] != kInvalidSlot ? word[g][j] & ~kFirstBit : 0u);
      }
#pragma unroll
      for (int j = 0; j < ITEMS; ++j)
        if (word[g][j] != kInvalidSlot && least[j] == uint32_t(h.pos_base + rel + j)) first[g] |= 1u << j;
    } else {
#pragma unroll
      for (int j = 0; j < ITEMS; ++j)
        if (rel + j < len && is_first(h, table, rel + j, word[g][j], ((lost[g] >> (8 * j)) & 0xffu) != 0)) first[g] |= 1u << j;
    }
    const int c = __builtin_popcount(first[g]);  // its bits are summed over the lanes by ballots
    lane_before[g] = 0;
    int sum = 0;
#pragma unroll
    for (int bit = 0; (1 << bit) <= ITEMS; ++bit) {
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
  const tile_state before = tile_exclusive_prefix<NT, false>(h.pos_state, tile, tile_word(total), h.look_polls, look, [&](int64_t t) {
    int n = 0;
    for (int j = 0; j < GROUPS * ITEMS; ++j) {  // (a tile before this one is full)
      const int64_t rel = t * kTile + int64_t(j) * NT + threadIdx.x;
      n += is_first(h, table, rel, h.slot[h.pos_base + rel], h.index != 0 && h.lost[h.pos_base + rel] != 0);
    }
    __syncthreads();
    return tile_word(block_sum<NT, int>(n, wave_count));
  });
  const int64_t rank0 = first_rank(h, s) + tile_sum_of(before);
  *begin = rank0;
  *end = rank0 + total;
  if ((tile + 1) * kTile >= len && threadIdx.x == 0) {  // the last tile: the frontier's size is known
    *h.n_unique = rank0 + total;
    if (h.host_sizes) {
      if (h.index == 0) mirror_to_host(h.host_sizes, s);
      mirror_to_host(h.host_sizes + h.index + 1, rank0 + total);
    }
  }
#pragma unroll
  for (int g = 0; g < GROUPS; ++g) {
    const int64_t p = h.pos_base + base + g * kGroup;
    uint32_t rank = uint32_t(rank0) + uint32_t(lane_before[g]);
    words ranks;
    bool changed = false;
    uint32_t links = 0;  // bit j: position j has lost its bit, and a link is where its rank would be
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      ranks[j] = rank;
      const uint32_t bare = word[g][j] & ~kFirstBit;
      if ((first[g] >> j) & 1) {
        static_cast<IdT*>(h.frontier)[rank] = table.key(bare);
        ++rank;
        changed |= h.index == 0;
        if (h.index == 0) word[g][j] = bare | kFirstBit;  // the bit as relabel_tile reads it
      } else if (((lost[g] >> (8 * j)) & 0xffu) != 0) {
        changed = true;
        links |= 1u << j;
        word[g][j] = uint32_t(p) + uint32_t(j);  // its own position, where the link to a smaller one is
      }
    }
    if (links != 0) {
      const words there = *reinterpret_cast<const words*>(h.rank_at + p);
#pragma unroll
      for (int j = 0; j < ITEMS; ++j)
        if ((links >> j) & 1) ranks[j] = there[j];
    }
    *reinterpret_cast<words*>(h.rank_at + p) = ranks;  // (beside the links only the ones at first positions are ever read)
    if (changed) *reinterpret_cast<words*>(h.slot + p) = word[g];
  }
}

// The same for a tile of the bucketed pass: what a position's id is in the order of its first occurrences is known,
// in the order of the buckets.
template <typename IdT, bool HASHED>
__device__ __forceinline__ void compact_sorted_tile(const Hop& h, const Buckets& b, int64_t s, uint32_t tile) {
  constexpr int ITEMS = 4, GROUPS = BucketShape::kItems / ITEMS, kWaves = kBucketBlock / kWave;
  constexpr uint32_t kGroup = kBucketBlock * ITEMS;
  using words = typename Items<ITEMS>::words;
  __shared__ __align__(16) uint32_t least_of[kBucketTile];
  __shared__ uint32_t wave_before[kWaves];  // first occurrences in tiles before this one
  __shared__ int wave_count[GROUPS * kWaves];
  const uint32_t front = uint32_t(front_units(s)), units = front + uint32_t(s * h.k);
  const int log_buckets = log_buckets_of(b, units);
  const uint32_t at = threadIdx.x * ITEMS, first_unit = tile * kBucketTile;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  uint32_t* slot = h.slot + h.pos_base;
  words word[GROUPS];  // (positions and units are multiples of 4 together)
#pragma unroll
  for (int g = 0; g < GROUPS; ++g) {
    const uint32_t u = first_unit + g * kGroup + at;
    word[g] = words(kInvalidSlot);
    if (u >= front && u < units) word[g] = nth(reinterpret_cast<const words*>(slot), (u - front) / ITEMS);
  }
  uint32_t before = firsts_before<kBucketBlock>(b, tile);
  unsort_tile<HASHED, BucketShape>(b, log_buckets, tile, least_of);
#pragma unroll
  for (int d = kWave / 2; d > 0; d >>= 1) before += __shfl_xor(before, d, kWave);
  if (lane == 0) wave_before[wave] = before;
  __syncthreads();
  uint32_t first[GROUPS];
  int lane_before[GROUPS];
#pragma unroll
  for (int g = 0; g < GROUPS; ++g) {
    first[g] = 0;
    const uint32_t u = first_unit + g * kGroup + at;
    const words least = *reinterpret_cast<const words*>(least_of + g * kGroup + at);
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      if (u + j >= units) word[g][j] = kInvalidSlot;
      if (word[g][j] != kInvalidSlot && (word[g][j] & kFirstBit) != 0 && least[j] == u + j) first[g] |= 1u << j;
    }
    const int c = __builtin_popcount(first[g]);  // its bits are summed over the lanes by ballots
    lane_before[g] = 0;
    int sum = 0;
#pragma unroll
    for (int bit = 0; (1 << bit) <= ITEMS; ++bit) {
      const uint64_t mask = __ballot((c >> bit) & 1);
      lane_before[g] += __builtin_popcountll(mask & ((uint64_t(1) << lane) - 1)) << bit;
      sum += __builtin_popcountll(mask) << bit;
    }
    if (lane == 0) wave_count[g * kWaves + wave] = sum;
  }
  __syncthreads();
  // the groups' and waves' counts, in the order of the positions: one a lane, summed over the lanes
  static_assert(GROUPS * kWaves <= kWave, "a count per lane");
  const int own = lane < GROUPS * kWaves ? wave_count[lane] : 0;
  int upto = own;
#pragma unroll
  for (int d = 1; d < GROUPS * kWaves; d <<= 1) {
    const int lower = __shfl_up(upto, d, kWave);
    if (lane >= d) upto += lower;
  }
  uint32_t rank0 = wave_before[lane & (kWaves - 1)];
#pragma unroll
  for (int d = kWaves / 2; d > 0; d >>= 1) rank0 += __shfl_xor(rank0, d, kWave);
  rank0 += uint32_t(first_rank(h, s));
  if (first_unit + kBucketTile >= units && threadIdx.x == GROUPS * kWaves - 1) {  // the last tile: the frontier's size is known
    *h.n_unique = int64_t(rank0) + upto;
    if (h.host_sizes) mirror_to_host(h.host_sizes + h.index + 1, int64_t(rank0) + upto);
  }
#pragma unroll
  for (int g = 0; g < GROUPS; ++g) {
    const uint32_t u = first_unit + g * kGroup + at;
    uint32_t rank = rank0 + uint32_t(lane_before[g] + __shfl(upto - own, g * kWaves + wave, kWave));
    if (u < front || u >= units) continue;
    const words least = *reinterpret_cast<const words*>(least_of + g * kGroup + at);
    words ranks;
    bool changed = false;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      ranks[j] = rank;
      if ((first[g] >> j) & 1) {
        nth(static_cast<IdT*>(h.frontier), rank) = IdT(word[g][j] & ~kFirstBit);
        ++rank;
      } else if (word[g][j] != kInvalidSlot && (word[g][j] & kFirstBit) != 0) {
        changed = true;
        const uint32_t met = least[j] < u + j ? least[j] : u + j;  // (one that is not before its own is none that the pass left)
        const uint32_t p = uint32_t(h.pos_base) + (met - front);
        word[g][j] = met < front ? met | kRankBit : p;
        ranks[j] = met < front ? met : p | kLinkBit;  // for the draws of the row that repeat this one
      } else if (word[g][j] != kInvalidSlot) {  // no unit: the same, where the sort has folded it
        ranks[j] = (word[g][j] & kRankBit) != 0 ? word[g][j] & (kRankBit - 1) : word[g][j] | kLinkBit;
      }
    }
    nth(reinterpret_cast<words*>(h.rank_at + h.pos_base), (u - front) / ITEMS) = ranks;
    if (changed) nth(reinterpret_cast<words*>(slot), (u - front) / ITEMS) = word[g];
  }
}

// The long ones among the frontier's rows of ranks [begin, end), which this block has just appended, go
// onto the next hop's queue.
template <typename IdT, int NT>
__device__ __forceinline__ void announce_long_rows(const Hop& h, int64_t begin, int64_t end) {
  const auto offset = [&](int64_t i) {
    const int64_t at = i < h.indptr.threshold ? i : i - h.indptr.threshold;
    const void* p = i < h.indptr.threshold ? h.indptr.dev : h.indptr.host;
    return h.indptr.elem_bytes == 8 ? static_cast<const int64_t*>(p)[at] : int64_t(static_cast<const int32_t*>(p)[at]);
  };
  __syncthreads();  // the ids are there
  for (int64_t rank = begin + threadIdx.x; rank < end; rank += NT) {
    const int64_t row = int64_t(static_cast<const IdT*>(h.frontier)[rank]);
    if (row < 0 || row >= h.indptr.total - 1) continue;
    const int64_t b = offset(row), deg = offset(row + 1) - b;
    if (deg <= int64_t(kLongRow) || deg > 0xffffffffLL || b < 0 || b + deg > h.n_edges) continue;  // (a bad row is found by the fill)
    h.long_rows[atomicAdd(reinterpret_cast<unsigned long long*>(h.long_count), 1ull)] = rank;
  }
}

// Virtual blocks: one per NT * kRowItems rows (scan of the rows' pick counts), then one per position tile.  A
// launch that fits the grid cap has a block for each in the worst case; a launch that loops (STRIDE)
// goes over the tiles the hop really has.
//
// What else the launch may do (ALSO): queue the long rows among those it appends; or write the previous hop's edge list, in blocks
// from LeftEdges::compact_blocks on, behind all that others wait for, where the fill had to leave it (launch_fill): a launch of
// its own is 5 us at the floor, and this one, of two blocks a CU that wait for one another, has the room.  111 M nodes,
// 4096 seeds, fanouts [5,10,15], a batch with its features: 217.5 -> 210.4 us, on two other cards 221.5 -> 217.3, 219.8 -> 218.1.
// Launches that do neither are kernels of their own, of 4 registers less: a weighted batch of 1024 seeds, [5,10,15], with its features
// 265.3 -> 262.7 us.
enum CompactAlso { kNothing, kLongRows, kEdgeList };
struct LeftEdges {
  Hop prev;
  int64_t relabel_count;    // virtual blocks of its list
  uint32_t compact_blocks;
};
struct NoEdges {};
template <CompactAlso ALSO> using EdgesToo = std::conditional_t<ALSO == kEdgeList, LeftEdges, NoEdges>;
template <typename IdT, typename TableT, int NT, int ITEMS, int GROUPS, bool STRIDE, CompactAlso ALSO>
__global__ __launch_bounds__(NT, 4) void hop_compact_kernel(Hop h, int64_t row_tiles, TableT table, EdgesToo<ALSO> also) {
  constexpr int64_t kTile = int64_t(NT) * ITEMS * GROUPS;
  int64_t begin = 0, end = 0;
  uint32_t blocks = gridDim.x;
  if constexpr (ALSO == kEdgeList) {
    blocks = also.compact_blocks;
    if (blockIdx.x >= blocks) {
      constexpr int kPer = NT / kEdgeBlock;
      for (int64_t vb = int64_t(blockIdx.x - blocks) * kPer + threadIdx.x / kEdgeBlock; vb < also.relabel_count;
           vb += int64_t(gridDim.x - blocks) * kPer)
        relabel_tile<IdT, TableT, false>(also.prev, table, vb, int(threadIdx.x % kEdgeBlock));
      return;
    }
  }
  if (h.bucketed != 0 && bucketed_now(h, seeds_of(h))) return;
  if (!STRIDE) {
    const int64_t vb = blockIdx.x;
    if (vb < row_tiles) offsets_tile<NT, true>(h, vb);
    else compact_tile<IdT, TableT, NT, ITEMS, GROUPS, true>(h, vb - row_tiles, table, &begin, &end);
    if (ALSO == kLongRows) announce_long_rows<IdT, NT>(h, begin, end);
    return;
  }
  const int64_t s = seeds_of(h);
  const int64_t rows = s > 0 ? (s + NT * kRowItems - 1) / (NT * kRowItems) : 1;  // (tile 0 of either kind writes the lengths)
  const int64_t len = seed_part(h, s) + s * h.k;
  const int64_t total = rows + (len > 0 ? (len + kTile - 1) / kTile : 1);
  for (int64_t vb = blockIdx.x; vb < total; vb += blocks) {
    begin = end = 0;
    if (vb < rows) offsets_tile<NT, false>(h, vb);
    else compact_tile<IdT, TableT, NT, ITEMS, GROUPS, false>(h, vb - rows, table, &begin, &end);
    if (ALSO == kLongRows) announce_long_rows<IdT, NT>(h, begin, end);
    __syncthreads();  // the tiles' LDS is rewritten by the block's next one
  }
}

// The same of a bucketed hop (nothing, where the hop has outgrown the pass): virtual blocks of kBucketBlock threads.
template <typename IdT, bool HASHED, bool STRIDE>
__global__ __launch_bounds__(kBucketBlock) void hop_compact_sorted_kernel(Hop h, Buckets b) {
  constexpr int64_t kRows = kBucketBlock * kRowItems;
  const int64_t s = wave_uniform(seeds_of(h));
  if (!bucketed_now(h, s)) return;
  const uint32_t rows = uint32_t(s > 0 ? (s + kRows - 1) / kRows : 1);  // (tile 0 of either kind writes the lengths)
  const uint32_t units = uint32_t(front_units(s) + s * h.k);
  const uint32_t total = rows + (units > 0 ? (units + kBucketTile - 1) / kBucketTile : 1);
  for (uint32_t vb = blockIdx.x; vb < total; vb += gridDim.x) {
    if (vb < rows) offsets_tile<kBucketBlock, false>(h, vb);
    else compact_sorted_tile<IdT, HASHED>(h, b, s, vb - rows);
    if (!STRIDE) return;
    __syncthreads();  // the tiles' LDS is rewritten by the block's next one
  }
}

template <typename IdT, typename TableT, bool STRIDE>
__global__ __launch_bounds__(kBlock) void hop_relabel_kernel(Hop h, int64_t blocks, TableT table) {
  DGS_FOR_VIRTUAL_BLOCKS(vb, blocks) relabel_tile<IdT, TableT, !STRIDE>(h, table, vb, threadIdx.x);
}

__global__ void zero_sizes_kernel(int64_t* __restrict__ sizes, int n) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) sizes[i] = 0;
}

__global__ __launch_bounds__(kBlock) void clear_kernel(uint4* __restrict__ p, int64_t n16) {
  for (int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x; i < n16; i += int64_t(gridDim.x) * kBlock)
    p[i] = make_uint4(~0u, ~0u, ~0u, ~0u);
}

// ---- host side -------------------------------------------------------------------------------

enum class TableKind { kDirect, kPacked, kSplit };

struct Plan {
  int n_hops = 0;
  TableKind kind = TableKind::kSplit;
  int64_t s_max[DGS_MAX_HOPS + 1];
  int64_t nnz_max[DGS_MAX_HOPS];
  uint32_t capacity = 0;     // hash table slots (one table for all hops)
  size_t table_bytes = 0;    // 0 for the direct table
  bool weighted = false;     // picks by edge weight: per-hop queues for long rows
  bool bucketed = false;     // the last hop may find its first occurrences by the bucketed pass (if it turns out to fit)
  bool bucket_hashed = false; // ... with ids told apart by an LDS hash table (graphs beyond kBucketedMaxNodes)
  bool bucket_space = false; // the workspace has room for that pass
  int64_t bucket_tiles = 0;   // its tiles: all of the hop's units in the worst case, or as many as there is room for
  int64_t bucket_pos_cap = 0; // padded positions of the hop that these hold
  int32_t log_buckets = 0;
  int32_t hash_slots = kHashSlots;
  uint32_t n_nodes = 0;
};

// Tiles of the bucketed pass: the frontier before the last hop at its worst case, and as many of the
// hop's padded positions as there is room for (a hop beyond that runs on the table).
inline void plan_bucket_tiles(Plan* p) {
  const int64_t front = front_units(p->s_max[p->n_hops - 1]), pos = p->nnz_max[p->n_hops - 1], tile = kBucketTile;
  p->bucket_tiles = std::min<int64_t>(kMaxBucketTiles, (front + pos + tile - 1) / tile);
  p->bucket_pos_cap = p->bucket_tiles * tile - front;
  p->bucket_space = p->n_hops >= 2;  // (also where the frontier leaves the positions none: a call's workspace never gets smaller as it grows)
}

dgs_status make_plan(int64_t n_seeds, const int64_t* fanouts, int32_t n_hops, int32_t id_bytes,
                     int64_t n_nodes, int64_t n_edges, bool have_node_table, Plan* p) {
  DGS_REQUIRE(n_hops >= 1 && n_hops <= DGS_MAX_HOPS, DGS_ERR_INVALID, "sample_blocks: %d hops (1..%d)", n_hops,
              DGS_MAX_HOPS);
  DGS_REQUIRE(fanouts != nullptr && n_seeds >= 0, DGS_ERR_INVALID, "sample_blocks: bad argument");
  DGS_REQUIRE(width_ok(id_bytes), DGS_ERR_INVALID, "sample_blocks: id width %d is not 4 or 8", id_bytes);
  p->n_hops = n_hops;
  p->s_max[0] = n_seeds;
  for (int h = 0; h < n_hops; ++h) {
    DGS_REQUIRE(fanouts[h] >= 0 && fanouts[h] <= kMaxPicks, DGS_ERR_UNSUPPORTED,
                "sample_blocks: fanout %lld outside 0..%d (use the per-hop operators)", (long long)fanouts[h],
                kMaxPicks);
    p->nnz_max[h] = p->s_max[h] * fanouts[h];
    p->s_max[h + 1] = p->s_max[h] + p->nnz_max[h];
    DGS_REQUIRE(p->s_max[h + 1] <= kMaxPositions, DGS_ERR_UNSUPPORTED,
                "sample_blocks: worst-case frontier of hop %d exceeds 2^30 ids", h);
  }
  // room for the bucketed pass (whether a hop takes it is decided below and, from its real size, on the device)
  plan_bucket_tiles(p);
  if (have_node_table) {
    DGS_REQUIRE(n_nodes >= 0 && n_nodes < 0x7fffffffLL, DGS_ERR_UNSUPPORTED,
                "sample_blocks: a node table needs fewer than 2^31 nodes (have %lld)", (long long)n_nodes);
    p->kind = TableKind::kDirect;
    // The bucketed pass: slot words are ids (the direct table's).  (Test hook: 1 never, 2 whatever the size, 3 whatever the
    // size and hashed whatever the graph, 4 like 3 with on-chip tables of 256 slots, so that small inputs fill them
    // and go over their buckets in parts.)
    const int64_t mode = debug_option(DGS_DEBUG_SAMPLER_BUCKETED);
    const int64_t picks = p->nnz_max[n_hops - 1];
    p->bucket_hashed = n_nodes > kBucketedMaxNodes || mode == 3 || mode == 4;
    const bool full = n_edges / 2 >= n_nodes * fanouts[n_hops - 1];  // (the rows' positions, as a rule)
    const bool large = !p->bucket_hashed && picks >= (full ? kBucketedMinPicksFull : kBucketedMinPicks) && n_nodes >= kBucketedMinNodes;
    p->bucketed = p->bucket_space && p->bucket_pos_cap > 0 && n_nodes >= 1 && fanouts[n_hops - 1] >= 1 && mode != 1 &&
                  (large || mode >= 2);
    p->hash_slots = mode == 4 ? 256 : kHashSlots;
    int log_b = kMinLogBuckets;
    if (p->bucket_hashed) {  // (as many as its units may need: log_buckets_of)
      while (log_b < kMaxLogBuckets && (int64_t(kHashSlots / 2) << log_b) < p->bucket_tiles * kBucketTile) ++log_b;
    } else {
      while ((int64_t(kBucketRange) << log_b) < n_nodes) ++log_b;
    }
    p->log_buckets = log_b;
    p->n_nodes = uint32_t(n_nodes);
  } else {
    // ids fit the packed slot when every node id is below 2^32 - 1
    p->kind = id_bytes == 4 || (n_nodes >= 0 && n_nodes < 0xffffffffLL) ? TableKind::kPacked : TableKind::kSplit;
    // test hook: exercise the split (id array + value array) table on small graphs
    if (id_bytes == 8 && debug_option(DGS_DEBUG_FORCE_SPLIT_TABLE) != 0) p->kind = TableKind::kSplit;
    p->capacity = table_capacity(p->s_max[n_hops]);
    p->table_bytes = size_t(p->capacity) * (p->kind == TableKind::kPacked ? 8 : size_t(id_bytes) + 4);
  }
  return DGS_OK;
}

inline int64_t row_tiles_of(int64_t rows, int64_t len_max) { return (rows + row_tile_size(len_max) - 1) / row_tile_size(len_max); }
inline int64_t pos_tiles_of(int64_t len_max) {
  return len_max > 0 ? (len_max + pos_tile_size(len_max) - 1) / pos_tile_size(len_max) : 1;
}

// Lays the workspace out; with base == nullptr only the size is computed.
size_t layout(const Plan& p, const int64_t* fanouts, void* base, Hop* hops, void** table,
              Buckets* buckets = nullptr) {
  Carver c(base);
  char* t = c.take<char>(p.table_bytes);
  if (table) *table = t;
  // sum over hops of (seed part + s_max * k), every hop's base rounded up to a multiple of 16, and a
  // tile beyond the last position (see compact_tile)
  const size_t positions = size_t(p.s_max[p.n_hops]) + 16 * size_t(p.n_hops) + kMaxPosTile;
  uint32_t* slot = c.take<uint32_t>(positions);
  uint32_t* rank_at = c.take<uint32_t>(positions);
  uint8_t* lost = c.take<uint8_t>(positions);
  // the tile states of all hops, right behind the lost marks: cleared together by hop 0's fill launch
  size_t tiles = 0;
  for (int h = 0; h < p.n_hops; ++h) {
    const int64_t len = (h == 0 ? p.s_max[0] : 0) + p.nnz_max[h];
    tiles += row_tiles_of(p.s_max[h], len) + pos_tiles_of(len);
  }
  tile_state* states = c.take<tile_state>(tiles + 2);
  int64_t* long_count = p.weighted ? c.take<int64_t>(2) : nullptr;  // (cleared with them)
  int64_t* long_rows = p.weighted ? c.take<int64_t>(size_t(p.s_max[p.n_hops - 1])) : nullptr;
  int64_t pos_base = 0;
  for (int h = 0; h < p.n_hops; ++h) {
    const size_t s = size_t(p.s_max[h]);
    const size_t len = (h == 0 ? s : 0) + size_t(p.nnz_max[h]);
    Hop v{};
    v.row_cnt = c.take<uint32_t>(s);
    v.row_off = c.take<uint32_t>(s);
    v.bucketed = p.bucketed && h == p.n_hops - 1;
    v.row_state = states;
    states += row_tiles_of(int64_t(s), int64_t(len));
    v.pos_state = states;
    states += pos_tiles_of(int64_t(len));
    v.slot = slot;
    v.rank_at = rank_at;
    v.lost = lost;
    v.long_rows = long_rows;
    v.long_count = long_count;
    if (p.weighted && h == 0) {
      v.long_seeds = c.take<uint8_t>(s + kSeedSegment);
      v.long_seed_count = c.take<int32_t>(s / kSeedSegment + 1);
    }
    v.s_max = p.s_max[h];
    v.pos_base = pos_base;
    v.len_max = int64_t(len);
    v.k = int32_t(fanouts[h]);
    v.index = h;
    v.bucket_pos_cap = p.bucket_pos_cap;
    if (hops) hops[h] = v;
    pos_base += (int64_t(len) + 15) / 16 * 16;
  }
  if (p.bucket_space) {
    Buckets b{};
    b.tiles_max = int32_t(p.bucket_tiles);
    b.items = c.take<uint2>(size_t(b.tiles_max) * kBucketTile);  // (the larger form's)
    b.least = c.take<uint32_t>(size_t(b.tiles_max) * kBucketTile);
    b.piece = c.take<uint16_t>(size_t(b.tiles_max) * (kMaxBuckets + 1));
    b.firsts = c.take<uint32_t>(kCounters * kMaxBucketTiles);
    b.overflow = c.take<int>(4);
    b.log_buckets = p.log_buckets;
    b.n_ids = p.n_nodes;
    b.hashed = p.bucket_hashed ? 1 : 0;
    b.hash_slots = p.hash_slots;
    b.log_tile = kLocalBits;
    if (buckets) *buckets = b;
    if (hops)
      for (int h = 0; h < p.n_hops; ++h) hops[h].bucket_overflow = b.overflow;
  }
  return c.used + 256;
}

// The packed edge list of one hop as a launch of its own.
template <typename IdT, typename TableT>
void launch_relabel(const Hop& hop, const TableT& table, hipStream_t st) {
  const int64_t blocks = edge_blocks(hop.s_max, hop.k);
  if (blocks <= 0) return;
  if (is_capped(blocks))
    hipLaunchKernelGGL((hop_relabel_kernel<IdT, TableT, true>), dim3(capped_grid(blocks)), dim3(kBlock), 0, st, hop,
                       blocks, table);
  else
    hipLaunchKernelGGL((hop_relabel_kernel<IdT, TableT, false>), dim3(capped_grid(blocks)), dim3(kBlock), 0, st, hop,
                       blocks, table);
}

// `left`: blocks of the previous hop's edge list that are to be written too; set to 0 where the launch takes them.
template <typename IdT, typename TableT, int NT, int ITEMS, int GROUPS, CompactAlso ALSO>
void launch_compact_as(const Hop& hop, const Hop& prev, int64_t* left, const TableT& table, hipStream_t st) {
  const int64_t row_tiles = row_tiles_of(hop.s_max, hop.len_max);
  const int64_t blocks = row_tiles + pos_tiles_of(hop.len_max), at_once = std::min(grid_cap(), kLookbackGrid);
  const uint32_t grid = uint32_t(std::min(blocks, at_once));
  uint32_t more = 0;
  EdgesToo<ALSO> also{};
  if constexpr (ALSO == kEdgeList) {
    also = LeftEdges{prev, *left, grid};
    more = uint32_t(std::min((*left + NT / kEdgeBlock - 1) / (NT / kEdgeBlock), kLoopGrid));
    *left = 0;
  }
  if (blocks > at_once)
    hipLaunchKernelGGL((hop_compact_kernel<IdT, TableT, NT, ITEMS, GROUPS, true, ALSO>), dim3(grid + more), dim3(NT), 0, st, hop,
                       row_tiles, table, also);
  else
    hipLaunchKernelGGL((hop_compact_kernel<IdT, TableT, NT, ITEMS, GROUPS, false, ALSO>), dim3(grid + more), dim3(NT), 0, st, hop,
                       row_tiles, table, also);
}
template <typename IdT, typename TableT, int NT, int ITEMS, int GROUPS>
void launch_compact(const Hop& hop, const Hop& prev, int64_t* left, bool announce, const TableT& table, hipStream_t st) {
  if (announce) return launch_compact_as<IdT, TableT, NT, ITEMS, GROUPS, kLongRows>(hop, prev, left, table, st);
  if constexpr (ITEMS > 1) {  // (fills that leave the list are not in front of the others)
    if (*left > 0) return launch_compact_as<IdT, TableT, NT, ITEMS, GROUPS, kEdgeList>(hop, prev, left, table, st);
  }
  launch_compact_as<IdT, TableT, NT, ITEMS, GROUPS, kNothing>(hop, prev, left, table, st);
}

// The bucketed pass and the compact launch behind it.
template <typename IdT, bool HASHED>
void launch_bucketed(const Hop& hop, const Buckets& b, hipStream_t st) {
  const uint32_t at_most = uint32_t(std::min(grid_cap(), kLookbackGrid));
  hipLaunchKernelGGL((bucket_sort_kernel<IdT, HASHED>), dim3(std::min(at_most, uint32_t(b.tiles_max))), dim3(kBucketBlock), 0, st, hop, b);
  const uint32_t buckets = std::min(at_most, 1u << b.log_buckets);
  if constexpr (HASHED) hipLaunchKernelGGL(bucket_first_hashed_kernel, dim3(buckets), dim3(kBucketBlock), 0, st, hop, b);
  else hipLaunchKernelGGL(bucket_first_kernel, dim3(buckets), dim3(kBucketBlock), 0, st, hop, b);
  const int64_t blocks = (hop.s_max + kBucketBlock * kRowItems - 1) / (kBucketBlock * kRowItems) + b.tiles_max;
  if (is_capped(blocks))
    hipLaunchKernelGGL((hop_compact_sorted_kernel<IdT, HASHED, true>), dim3(capped_grid(blocks)), dim3(kBucketBlock), 0, st, hop, b);
  else
    hipLaunchKernelGGL((hop_compact_sorted_kernel<IdT, HASHED, false>), dim3(uint32_t(blocks)), dim3(kBucketBlock), 0, st, hop, b);
}

// Returns the blocks of the previous hop's edge list that are left to be written behind this launch.
template <typename IdT, typename PtrT, typename TableT, int G>
int64_t launch_fill(const Hop& cur, const Hop& prev, int64_t relabel_count, uint4* clear_begin, int64_t clear_n16,
                    const TableT& table, const dgs_view& indptr, const dgs_view& indices, bool replace,
                    uint64_t rng_seed, hipStream_t st) {
  const int64_t fill_blocks = (cur.s_max * G + kBlock - 1) / kBlock;
  const int64_t clear_blocks = (clear_n16 + kBlock - 1) / kBlock;
  const int64_t total = fill_blocks + relabel_count + clear_blocks;
  if (is_capped(total)) {
    // A launch that loops over its virtual blocks keeps the previous hop's edge list out of the
    // loop: with it the kernel needs 85-90 vector registers and five waves fit a SIMD instead of
    // seven (measured on a 136 k-row hop: 46 us against 39).  That list goes with the compact launch or is one of its own,
    // behind this one (the previous hop's table entries do not change any more: positions only grow).
    hipLaunchKernelGGL((hop_fill_kernel<IdT, PtrT, TableT, G, true>), dim3(capped_grid(total - relabel_count)), dim3(kBlock), 0, st,
                       cur, prev, fill_blocks, int64_t(0), clear_begin, clear_n16, table,
                       TierView<PtrT>(indptr), TierView<IdT>(indices), replace, rng_seed);
    return relabel_count;
  }
  hipLaunchKernelGGL((hop_fill_kernel<IdT, PtrT, TableT, G, false>), dim3(capped_grid(total)), dim3(kBlock), 0, st,
                     cur, prev, fill_blocks, relabel_count, clear_begin, clear_n16, table,
                     TierView<PtrT>(indptr), TierView<IdT>(indices), replace, rng_seed);
  return 0;
}

// Blocks of a weighted launch that take queued long rows, in front of `others`.  256 keep a block on every CU, which
// a frontier of hubs leaves waiting for its chains: 512 where they and the others fit the GPU at once, four
// blocks to a CU (three where the picks are drawn), or where there are several rounds of the others anyway.  In between the others would be dealt
// out unevenly behind them (2048 seeds, fanouts [10,10], rows of 300: 129 us with 256, 137 with 512).
// us a call, 256 / 512: 16 384 rows of 3000 750 / 441 (10 picks), 455 / 279 (draws); of 17 000 1572 / 926, 1360 /
// 791; 300 of 20 000 among them 134 / 107, 129 / 104; 1024 seeds, fanouts [10,10], rows of 3000 548 / 358, 352 / 239.
// Draws by 12 289 seeds of 1000 positions, no long row among them: 133 with 256 or 383, 141 with 512.
// Batches whose long rows are a few hundred: level.  1024 or 2048: 290 for the first, and 2 to 5 us more for those.
inline int64_t queue_blocks(int64_t others, bool replace) {
  if (others >= 1024) return kMaxQueueBlocks;
  const int64_t slots = replace ? 768 : 1024;
  return std::min(kMaxQueueBlocks, std::max(kMinQueueBlocks, slots - others));
}

// Whether a weighted hop is a launch of kLongBlock-thread blocks (see above).
inline bool weighted_shared(const Hop& h) { return h.s_max <= (h.index == 0 ? kSharedMaxSeeds : kSharedMaxRows); }

template <typename IdT, typename PtrT, typename TableT, bool REPLACE>
void launch_fill_weighted(const Hop& cur, const Hop& prev, int64_t relabel_count, uint4* clear_begin, int64_t clear_n16,
                          const TableT& table, const dgs_view& indptr, const dgs_view& indices, const dgs_view& probs,
                          uint64_t rng_seed, hipStream_t st) {
  const int64_t clear_blocks = (clear_n16 + kBlock - 1) / kBlock;
  if (weighted_shared(cur)) {
    const int64_t rows = std::min<int64_t>(kSharedRows, std::max<int64_t>(1, (cur.s_max + kSharedBlocks - 1) / kSharedBlocks));
    const int64_t fill_blocks = (cur.s_max + rows - 1) / rows;
    const int64_t others = (relabel_count + clear_blocks + kLongBlock / kBlock - 1) / (kLongBlock / kBlock);
    hipLaunchKernelGGL((hop_fill_weighted_shared_kernel<IdT, PtrT, TableT, REPLACE>), dim3(uint32_t(fill_blocks + others)),
                       dim3(kLongBlock), 0, st, cur, prev, fill_blocks, int32_t(rows), relabel_count, clear_begin, clear_n16, table,
                       TierView<PtrT>(indptr), TierView<IdT>(indices), TierView<float>(probs), rng_seed);
    return;
  }
  if (cur.index == 0) {
    const int64_t segments = (cur.s_max + kSeedSegment - 1) / kSeedSegment;
    hipLaunchKernelGGL((announce_long_seeds_kernel<IdT, PtrT>), dim3(uint32_t(segments + clear_blocks)), dim3(kSeedSegment), 0, st,
                       cur, segments, clear_begin, clear_n16, TierView<PtrT>(indptr), indices.total);
  }
  const int64_t rows = choose_rows(cur.k);
  const int64_t fill_blocks = (cur.s_max + rows - 1) / rows;
  const int64_t queued = queue_blocks(fill_blocks + relabel_count, REPLACE);
  const int64_t total = queued + fill_blocks + relabel_count;
  hipLaunchKernelGGL((hop_fill_weighted_kernel<IdT, PtrT, TableT, REPLACE>), dim3(capped_grid(total)), dim3(kBlock), 0, st, cur,
                     prev, queued, fill_blocks, int32_t(rows), relabel_count, table, TierView<PtrT>(indptr), TierView<IdT>(indices),
                     TierView<float>(probs), rng_seed);
}

template <typename IdT, typename PtrT, typename TableT>
dgs_status run_blocks(const Plan& p, Hop* hops, const Buckets& buckets, const TableT& table, const dgs_view& indptr,
                      const dgs_view& indices, const dgs_view* probs, bool replace, uint64_t rng_seed,
                      void** sizes_ticket, EdgeJob* left, hipStream_t st) {
  for (int h = 0; h < p.n_hops; ++h) {
    const Hop& cur = hops[h];
    const Hop prev = h > 0 ? hops[h - 1] : Hop{};
    const int64_t surplus = h > 0 ? edge_blocks(prev.s_max, prev.k) : 0;
    // the launch of hop 0 also clears the lost marks of all later hops and the tile states of all
    // hops, which lie behind them
    uint4* clear_begin = nullptr;
    int64_t clear_n16 = 0;
    if (h == 0) {
      const Hop& last = hops[p.n_hops - 1];
      clear_begin = reinterpret_cast<uint4*>(cur.lost + (p.n_hops > 1 ? hops[1].pos_base : p.s_max[1] / 16 * 16));
      const char* end = reinterpret_cast<const char*>(last.pos_state + pos_tiles_of(last.len_max));  // (two spare words follow)
      if (p.weighted) end = reinterpret_cast<const char*>(cur.long_count + 2);  // (which comes next)
      clear_n16 = (end - reinterpret_cast<const char*>(clear_begin) + 15) / 16;
    }
    int64_t left_over = 0;
    if (p.weighted) {
      if (replace) launch_fill_weighted<IdT, PtrT, TableT, true>(cur, prev, surplus, clear_begin, clear_n16, table, indptr, indices, *probs, rng_seed, st);
      else launch_fill_weighted<IdT, PtrT, TableT, false>(cur, prev, surplus, clear_begin, clear_n16, table, indptr, indices, *probs, rng_seed, st);
    } else if (cur.k <= 8) left_over = launch_fill<IdT, PtrT, TableT, 8>(cur, prev, surplus, clear_begin, clear_n16, table, indptr, indices, replace, rng_seed, st);
    else if (cur.k <= 16) left_over = launch_fill<IdT, PtrT, TableT, 16>(cur, prev, surplus, clear_begin, clear_n16, table, indptr, indices, replace, rng_seed, st);
    else if (cur.k <= 32) left_over = launch_fill<IdT, PtrT, TableT, 32>(cur, prev, surplus, clear_begin, clear_n16, table, indptr, indices, replace, rng_seed, st);
    else left_over = launch_fill<IdT, PtrT, TableT, 64>(cur, prev, surplus, clear_begin, clear_n16, table, indptr, indices, replace, rng_seed, st);
    DGS_LAUNCH_CHECK();

    if constexpr (std::is_same_v<TableT, DirectTable<IdT>>) {
      if (cur.bucketed) {  // (the last hop)
        if (buckets.hashed) launch_bucketed<IdT, true>(cur, buckets, st);
        else launch_bucketed<IdT, false>(cur, buckets, st);
        DGS_LAUNCH_CHECK();
        if (cur.len_max <= cur.bucket_pos_cap) {  // (it cannot outgrow the pass)
          if (left_over > 0) launch_relabel<IdT>(prev, table, st);
          DGS_LAUNCH_CHECK();
          break;
        }
      }
    }
    // (a queue holds the whole frontier: from hop 0 on, where a later hop reads it; hops only get larger)
    const bool announce = p.weighted && h + 1 < p.n_hops && !weighted_shared(hops[p.n_hops - 1]);
    switch (pos_tile_kind(cur.len_max)) {
      case kShortTile: launch_compact<IdT, TableT, 256, 1, 1>(cur, prev, &left_over, announce, table, st); break;
      case kMiddleTile: launch_compact<IdT, TableT, 256, 4, 4>(cur, prev, &left_over, announce, table, st); break;
      case kLongTile: launch_compact<IdT, TableT, 512, 4, 4>(cur, prev, &left_over, announce, table, st); break;
    }
    if (left_over > 0) launch_relabel<IdT>(prev, table, st);
    DGS_LAUNCH_CHECK();
  }
  // every length is final here: mark the point the caller may wait for
  if (sizes_ticket) {
    const dgs_status ts = dgs_ticket_record(st, sizes_ticket);
    if (ts != DGS_OK) return ts;
  }
  const Hop& last = hops[p.n_hops - 1];
  if (left != nullptr && p.n_hops > 1) {
    *left = edge_job(last);
    left->blocks = edge_blocks(last.s_max, last.k);
    left->id_bytes = int32_t(sizeof(IdT));
    return DGS_OK;
  }
  launch_relabel<IdT>(last, table, st);
  DGS_LAUNCH_CHECK();
  return DGS_OK;
}

// Whether the call is one launch of one block (one_block.h): the more launches that saves, the more
// positions one CU may work through.  us per batch with its features, one block / the launches: one hop,
// 770 positions 44.3 / 48.8, 1023 44.9 / 49.6, 2024 49.4 / 50.2, 3960 60.1 / 50.8; two hops, 1056 50.1 / 56.4,
// 1980 54.1 / 56.2, 2640 56.3 / 56.4, 4092 65.9 / 59.1; three hops, 1728 56.4 / 87.1, 3024 62.6 / 89.1, 3888
// 67.3 / 89.1 (what saves them more than a launch floor is that the host sends one launch).
inline bool one_block_fits(const Plan& p) {
  const int64_t limit = std::min<int64_t>(kOnePositions, int64_t(1024) * p.n_hops);
  return !p.weighted && p.kind != TableKind::kSplit && p.s_max[p.n_hops] <= limit &&
         debug_option(DGS_DEBUG_SAMPLER_BUCKETED) == 0 && debug_option(DGS_DEBUG_SAMPLER_GRID_CAP) == 0 &&
         debug_option(DGS_DEBUG_LOOKBACK_POLLS) == 0;  // (test hooks of the launches it replaces)
}

template <typename IdT, typename PtrT>
dgs_status run_one_block(const Plan& p, const Hop* hops, int64_t* sizes, const dgs_view& indptr, const dgs_view& indices,
                         bool replace, uint64_t rng_seed, void** sizes_ticket, hipStream_t st) {
  OneBlockBatch q{};
  q.seeds = hops[0].seeds;
  q.n_seeds = p.s_max[0];
  q.frontier = hops[0].frontier;
  q.sizes = sizes;
  q.host_sizes = hops[0].host_sizes;
  q.id_limit = p.kind == TableKind::kDirect ? uint64_t(indptr.total - 1) : 0xffffffffull;  // what the table would hold
  q.rng_seed = rng_seed;
  q.first_stream = hops[0].rng_stream;
  q.n_hops = p.n_hops;
  q.replace = replace;
  for (int h = 0; h < p.n_hops; ++h) {
    q.k[h] = hops[h].k;
    q.src_local[h] = hops[h].src_local;
    q.dst_local[h] = hops[h].dst_local;
  }
  hipLaunchKernelGGL((one_block_kernel<IdT, PtrT>), dim3(1), dim3(kOneBlock), 0, st, q, TierView<PtrT>(indptr), TierView<IdT>(indices));
  DGS_LAUNCH_CHECK();
  return sizes_ticket ? dgs_ticket_record(st, sizes_ticket) : DGS_OK;
}

template <typename IdT, typename PtrT>
dgs_status run_blocks_table(const Plan& p, Hop* hops, const Buckets& buckets, void* hash_table, void* node_table,
                            uint32_t epoch, const dgs_view& indptr, const dgs_view& indices, const dgs_view* probs,
                            bool replace, uint64_t rng_seed, void** sizes_ticket, EdgeJob* left, hipStream_t st) {
  if (one_block_fits(p))
    return run_one_block<IdT, PtrT>(p, hops, hops[0].n_seeds_out, indptr, indices, replace, rng_seed, sizes_ticket, st);
  if (p.kind == TableKind::kDirect)
    return run_blocks<IdT, PtrT, DirectTable<IdT>>(p, hops, buckets, DirectTable<IdT>(node_table, epoch, uint32_t(indptr.total - 1)),
                                                   indptr, indices, probs, replace, rng_seed, sizes_ticket, left, st);
  const int64_t n16 = int64_t(p.table_bytes / 16);
  hipLaunchKernelGGL(clear_kernel, dim3(capped_grid((n16 + kBlock - 1) / kBlock)), dim3(kBlock), 0, st,
                     static_cast<uint4*>(hash_table), n16);
  DGS_LAUNCH_CHECK();
  if (p.kind == TableKind::kPacked)
    return run_blocks<IdT, PtrT, Table<IdT, true>>(p, hops, buckets, Table<IdT, true>(hash_table, p.capacity), indptr,
                                                   indices, probs, replace, rng_seed, sizes_ticket, left, st);
  return run_blocks<IdT, PtrT, Table<IdT, false>>(p, hops, buckets, Table<IdT, false>(hash_table, p.capacity), indptr,
                                                  indices, probs, replace, rng_seed, sizes_ticket, left, st);
}

}  // namespace
}  // namespace dgs

DGS_API dgs_status dgs_sample_blocks_plan(int64_t n_seeds, const int64_t* fanouts, int32_t n_hops,
                                          int64_t* seeds_max, int64_t* edges_max) {
  dgs::Plan p;
  dgs_status s = dgs::make_plan(n_seeds, fanouts, n_hops, 8, -1, -1, false, &p);
  if (s != DGS_OK) return s;
  DGS_REQUIRE(seeds_max && edges_max, DGS_ERR_INVALID, "sample_blocks_plan: null output");
  for (int h = 0; h <= n_hops; ++h) seeds_max[h] = p.s_max[h];
  for (int h = 0; h < n_hops; ++h) edges_max[h] = p.nnz_max[h];
  return DGS_OK;
}

DGS_API size_t dgs_sample_blocks_workspace_bytes(int64_t n_seeds, const int64_t* fanouts, int32_t n_hops,
                                                 int32_t id_bytes) {
  dgs::Plan p;
  // sized for the split hash table, the largest of the layouts
  if (dgs::make_plan(n_seeds, fanouts, n_hops, id_bytes, -1, -1, false, &p) != DGS_OK) return 0;
  p.kind = dgs::TableKind::kSplit;
  p.table_bytes = size_t(p.capacity) * (size_t(id_bytes) + 4);
  return dgs::layout(p, fanouts, nullptr, nullptr, nullptr);
}

DGS_API size_t dgs_node_table_bytes(int64_t n_nodes) {
  return n_nodes > 0 && n_nodes < 0x7fffffffLL ? size_t(n_nodes) * 8 : 0;
}

DGS_API size_t dgs_sample_blocks_weighted_workspace_bytes(int64_t n_seeds, const int64_t* fanouts, int32_t n_hops,
                                                          int32_t id_bytes) {
  dgs::Plan p;
  // sized for the split hash table, the largest of the layouts (used when there is no node table)
  if (dgs::make_plan(n_seeds, fanouts, n_hops, id_bytes, -1, -1, false, &p) != DGS_OK) return 0;
  p.kind = dgs::TableKind::kSplit;
  p.table_bytes = size_t(p.capacity) * (size_t(id_bytes) + 4);
  p.weighted = true;
  return dgs::layout(p, fanouts, nullptr, nullptr, nullptr);
}

namespace {
dgs_status sample_blocks_entry(const void* seeds, int32_t id_bytes, int64_t n_seeds, dgs_view indptr,
                               dgs_view indices, const dgs_view* probs, const int64_t* fanouts, int32_t n_hops,
                               int32_t replace, uint64_t rng_seed, uint32_t first_stream, void* node_table,
                               uint32_t node_table_epoch, void* frontier, const dgs_block_out* outs,
                               int64_t* sizes_dev, int64_t* sizes_host, void** sizes_ticket, dgs::EdgeJob* left,
                               void* workspace, size_t workspace_bytes, void* stream) {
  using namespace dgs;
  Plan p;
  // node count = indptr entries - 1
  dgs_status s = make_plan(n_seeds, fanouts, n_hops, id_bytes, indptr.total - 1, indices.total, node_table != nullptr, &p);
  if (s != DGS_OK) return s;
  if (probs != nullptr) {
    DGS_REQUIRE(probs->elem_bytes == 4 && probs->total == indices.total, DGS_ERR_INVALID,
                "sample_blocks_weighted: %lld weights of %d bytes for %lld edges (float32, one per edge)",
                (long long)probs->total, probs->elem_bytes, (long long)indices.total);
    p.weighted = true;
    // weighted picks: the fill is bound by the races, not by its atomics, and the bucketed pass
    // changes the step by a per cent either way (measured with three and four batches in flight)
    if (debug_option(DGS_DEBUG_SAMPLER_BUCKETED) < 2) p.bucketed = false;
  }
  const size_t need = probs != nullptr ? dgs_sample_blocks_weighted_workspace_bytes(n_seeds, fanouts, n_hops, id_bytes)
                                       : dgs_sample_blocks_workspace_bytes(n_seeds, fanouts, n_hops, id_bytes);
  DGS_REQUIRE(width_ok(indptr.elem_bytes), DGS_ERR_INVALID, "sample_blocks: indptr width %d", indptr.elem_bytes);
  DGS_REQUIRE(indices.elem_bytes == id_bytes, DGS_ERR_INVALID,
              "sample_blocks: indices width %d differs from the seed width %d", indices.elem_bytes, id_bytes);
  DGS_REQUIRE(outs != nullptr && sizes_dev != nullptr, DGS_ERR_INVALID, "sample_blocks: null output");
  DGS_REQUIRE(node_table == nullptr || (node_table_epoch >= 1 && node_table_epoch < 0xfffffff0u), DGS_ERR_INVALID,
              "sample_blocks: node table epoch %u outside 1..2^32-17 (refill the table with 0xFF and restart at 1)",
              node_table_epoch);
  DGS_REQUIRE(sizes_ticket == nullptr || sizes_host != nullptr, DGS_ERR_INVALID,
              "sample_blocks: a sizes_ticket needs sizes_host");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (n_seeds == 0) {  // nothing to launch: every size is zero
    // a fill kernel, not a memset node: the call may be recorded into a graph
    hipLaunchKernelGGL(zero_sizes_kernel, dim3(1), dim3(64), 0, st, sizes_dev, 3 * n_hops + 1);
    DGS_LAUNCH_CHECK();
    if (sizes_host)
      for (int i = 0; i < 3 * n_hops + 1; ++i) sizes_host[i] = 0;
    return sizes_ticket ? dgs_ticket_record(st, sizes_ticket) : DGS_OK;
  }
  DGS_REQUIRE(seeds != nullptr && frontier != nullptr, DGS_ERR_INVALID, "sample_blocks: null seeds or frontier");
  DGS_REQUIRE(workspace != nullptr && workspace_bytes >= need, DGS_ERR_WORKSPACE,
              "sample_blocks: workspace of %zu B, need %zu", workspace_bytes, need);
  DGS_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 255) == 0, DGS_ERR_WORKSPACE,
              "sample_blocks: workspace must be 256-byte aligned");
  Hop hops[DGS_MAX_HOPS];
  void* hash_table = nullptr;
  Buckets buckets{};
  layout(p, fanouts, workspace, hops, &hash_table, &buckets);
  for (int h = 0; h < n_hops; ++h) {
    Hop& t = hops[h];
    DGS_REQUIRE(p.nnz_max[h] == 0 || (outs[h].src_local && outs[h].dst_local), DGS_ERR_INVALID,
                "sample_blocks: null edge buffers for hop %d", h);
    t.seeds = h == 0 ? seeds : frontier;
    t.n_seeds = sizes_dev + h;
    t.n_seeds_host = h == 0 ? n_seeds : -1;
    t.n_seeds_out = h == 0 ? sizes_dev : nullptr;
    t.prev_nnz = sizes_dev + n_hops + (h == 0 ? 1 : h);  // edges of hop h - 1 (hop 0: any readable word)
    t.prev_n_seeds = sizes_dev + (h == 0 ? 0 : h - 1);
    t.n_unique = sizes_dev + h + 1;
    t.nnz = sizes_dev + n_hops + 1 + h;
    t.flags = sizes_dev + 2 * n_hops + 1 + h;
    t.host_sizes = sizes_host;
    t.n_hops = n_hops;
    t.look_polls = lookback_polls();
    t.frontier = frontier;
    t.src_local = outs[h].src_local;
    t.dst_local = outs[h].dst_local;
    t.rng_stream = first_stream + uint32_t(h);
    t.indptr = indptr;
    t.n_edges = indices.total;
  }
  const bool rep = replace != 0;
  if (id_bytes == 8)
    return indptr.elem_bytes == 8
               ? run_blocks_table<int64_t, int64_t>(p, hops, buckets, hash_table, node_table, node_table_epoch, indptr, indices, probs, rep, rng_seed, sizes_ticket, left, st)
               : run_blocks_table<int64_t, int32_t>(p, hops, buckets, hash_table, node_table, node_table_epoch, indptr, indices, probs, rep, rng_seed, sizes_ticket, left, st);
  return indptr.elem_bytes == 8
             ? run_blocks_table<int32_t, int64_t>(p, hops, buckets, hash_table, node_table, node_table_epoch, indptr, indices, probs, rep, rng_seed, sizes_ticket, left, st)
             : run_blocks_table<int32_t, int32_t>(p, hops, buckets, hash_table, node_table, node_table_epoch, indptr, indices, probs, rep, rng_seed, sizes_ticket, left, st);
}
}  // namespace

DGS_API dgs_status dgs_sample_blocks(const void* seeds, int32_t id_bytes, int64_t n_seeds, dgs_view indptr,
                                     dgs_view indices, const int64_t* fanouts, int32_t n_hops, int32_t replace,
                                     uint64_t rng_seed, uint32_t first_stream, void* node_table,
                                     uint32_t node_table_epoch, void* frontier, const dgs_block_out* outs,
                                     int64_t* sizes_dev, int64_t* sizes_host, void** sizes_ticket,
                                     void* workspace, size_t workspace_bytes, void* stream) {
  return sample_blocks_entry(seeds, id_bytes, n_seeds, indptr, indices, nullptr, fanouts, n_hops, replace, rng_seed,
                             first_stream, node_table, node_table_epoch, frontier, outs, sizes_dev, sizes_host,
                             sizes_ticket, nullptr, workspace, workspace_bytes, stream);
}

DGS_API dgs_status dgs_sample_blocks_weighted(const void* seeds, int32_t id_bytes, int64_t n_seeds, dgs_view indptr,
                                              dgs_view indices, dgs_view probs, const int64_t* fanouts,
                                              int32_t n_hops, int32_t replace, uint64_t rng_seed,
                                              uint32_t first_stream, void* node_table, uint32_t node_table_epoch,
                                              void* frontier, const dgs_block_out* outs, int64_t* sizes_dev,
                                              int64_t* sizes_host, void** sizes_ticket, void* workspace,
                                              size_t workspace_bytes, void* stream) {
  return sample_blocks_entry(seeds, id_bytes, n_seeds, indptr, indices, &probs, fanouts, n_hops, replace, rng_seed,
                             first_stream, node_table, node_table_epoch, frontier, outs, sizes_dev, sizes_host,
                             sizes_ticket, nullptr, workspace, workspace_bytes, stream);
}

static_assert(sizeof(dgs::EdgeJob) <= sizeof(dgs_edge_job), "a job fits the caller's words");
DGS_API dgs_status dgs_sample_blocks_leave_edges(const void* seeds, int32_t id_bytes, int64_t n_seeds, dgs_view indptr,
                                                 dgs_view indices, const dgs_view* probs, const int64_t* fanouts,
                                                 int32_t n_hops, int32_t replace, uint64_t rng_seed, uint32_t first_stream,
                                                 void* node_table, uint32_t node_table_epoch, void* frontier,
                                                 const dgs_block_out* outs, int64_t* sizes_dev, int64_t* sizes_host,
                                                 dgs_edge_job* left, void* workspace, size_t workspace_bytes, void* stream) {
  DGS_REQUIRE(left != nullptr, DGS_ERR_INVALID, "sample_blocks_leave_edges: null job");
  dgs::EdgeJob job{};
  const dgs_status s = sample_blocks_entry(seeds, id_bytes, n_seeds, indptr, indices, probs, fanouts, n_hops, replace, rng_seed,
                                           first_stream, node_table, node_table_epoch, frontier, outs, sizes_dev, sizes_host,
                                           nullptr, &job, workspace, workspace_bytes, stream);
  *left = dgs_edge_job{};
  memcpy(left, &job, sizeof(job));
  return s;
}
