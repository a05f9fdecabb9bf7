// All hops of a small batch in one launch of one block, with the ids' table, the frontier and the ranks
// in LDS.
//
// A batch of a few seeds is a chain of launches that each take their 5 us floor whatever they do, and a
// host that sends them one after the other: 16 seeds over fanouts [5,10] are five sampler launches, and
// take 56.4 us with the host's part and the features where one block needs 50.1; three hops of 5 from 8
// seeds 87.1 and 56.4.
// Here a hop is four steps between barriers of one block: picks (G lanes per seed row) and their
// insertion, first occurrences and ranks (a scan over positions), the rows' edge offsets (a scan over
// rows), the edge list.  Results are those of the launches in pipeline.hip: same picks, same order of
// positions, same flags.  Bound: latency, about 2 us a hop for the offsets and neighbour ids of every
// 1024 / G rows, and one CU's LDS atomics.
#ifndef DGS_CSRC_ONE_BLOCK_H_
#define DGS_CSRC_ONE_BLOCK_H_

#include "common.h"
#include "picks.h"
#include "table.h"

namespace dgs {

constexpr int kOneBlock = 1024;
constexpr int kOneItems = 4;
constexpr int kOnePositions = kOneBlock * kOneItems;  // the caller's seeds and all hops' padded picks, at most
constexpr int kOneSlots = 2 * kOnePositions;          // entries of the LDS table: at most half full

struct OneBlockBatch {
  const void* seeds;
  int64_t n_seeds;
  void* frontier;
  int64_t* sizes;       // n_hops + 1 frontier sizes, then n_hops edge counts, then n_hops flag words
  int64_t* host_sizes;  // optional pinned mirror of them
  uint64_t id_limit;    // picked ids must be below it (at most 2^32 - 1)
  uint64_t rng_seed;
  uint32_t first_stream;
  int32_t n_hops;
  int32_t replace;
  int32_t k[DGS_MAX_HOPS];
  void* src_local[DGS_MAX_HOPS];
  void* dst_local[DGS_MAX_HOPS];
};

struct OneBlockLds {
  unsigned long long table[kOneSlots];  // id << 32 | smallest position; all ones: empty
  uint32_t front[kOnePositions];        // ids by rank
  uint32_t row[kOnePositions];          // per row of the hop: picks, then first edge << 8 | picks
  uint16_t slot[kOnePositions];         // per position: its id's table entry
  uint16_t rank_at[kOnePositions];      // per first position: its id's rank
  int scan[kOneBlock / kWave];
  int flags;
};
constexpr uint16_t kOneNoSlot = 0xffffu;
static_assert(kOneSlots <= kOneNoSlot && DGS_MAX_HOPS <= 16, "table entries and hops fit their words");

__device__ __forceinline__ uint16_t one_block_insert(OneBlockLds& lds, uint32_t id, uint32_t position) {
  const unsigned long long packed = (static_cast<unsigned long long>(id) << 32) | position;
  uint32_t at = hash_id(id) & uint32_t(kOneSlots - 1);
  for (;;) {  // ends: fewer ids than entries
    const unsigned long long cur = atomicCAS(&lds.table[at], ~0ull, packed);
    if (cur == ~0ull) break;
    if (uint32_t(cur >> 32) == id) {
      if (cur > packed) atomicMin(&lds.table[at], packed);
      break;
    }
    at = (at + 1) & uint32_t(kOneSlots - 1);
  }
  return uint16_t(at);
}

// Picks of hop h's s rows, G lanes per row; positions pos0 + row * k + slot, hop 0's rows themselves at
// the position of their number.  Nothing is addressed by an id or an offset before it has been checked.
template <typename IdT, typename PtrT, int G>
__device__ __forceinline__ void one_block_picks(OneBlockLds& lds, const OneBlockBatch& q, int h, int s, int pos0,
                                                const TierView<PtrT>& indptr, const TierView<IdT>& indices) {
  const int k = q.k[h];
  const bool replace = q.replace != 0;
  const int l = threadIdx.x & (G - 1);
  const int group_lane0 = (threadIdx.x & (kWave - 1)) - l;
  const uint32_t stream = q.first_stream + uint32_t(h);
  for (int i0 = 0; i0 < s; i0 += kOneBlock / G) {
    const int i = i0 + int(threadIdx.x) / G;
    const bool live = i < s;
    int64_t row = -1;
    if (live) row = h == 0 ? int64_t(static_cast<const IdT*>(q.seeds)[i]) : int64_t(lds.front[i]);
    const bool seed_ok = row_in_range(indptr, row) && uint64_t(row) < q.id_limit;
    int64_t b = 0, deg64 = 0;
    if (seed_ok) {
      b = int64_t(indptr.at(row));
      deg64 = int64_t(indptr.at(row + 1)) - b;
    }
    const PhiloxWords words = philox_draw_words(q.rng_seed, stream, row, uint32_t(l));
    const bool bad = deg64 < 0 || deg64 > 0xffffffffLL || b < 0 || b + deg64 > indices.n;
    const uint32_t deg = bad ? 0u : uint32_t(deg64);
    if (live && l == 0 && h == 0) lds.slot[i] = seed_ok ? one_block_insert(lds, uint32_t(row), uint32_t(i)) : kOneNoSlot;
    uint32_t pos = 0;
    const bool have = pick_position<G>(deg, k, replace, l, group_lane0, words, &pos) && live && l < k;
    bool pick_ok = true;
    uint16_t slot = kOneNoSlot;
    const int p = pos0 + i * k + l;
    if (have) {
      const IdT id = indices.at(b + pos);
      pick_ok = uint64_t(int64_t(id)) < q.id_limit;
      if (pick_ok) slot = one_block_insert(lds, uint32_t(id), uint32_t(p));
    }
    if (live && l < k) lds.slot[p] = slot;
    constexpr uint64_t group_mask = G == 64 ? ~uint64_t(0) : ((uint64_t(1) << (G & 63)) - 1);
    const bool picks_ok = ((__ballot(!pick_ok) >> group_lane0) & group_mask) == 0;
    if (live && l == 0) {
      const int flag = !seed_ok ? 2 : bad ? 1 : !picks_ok ? 4 : 0;  // (the hop's flag word, as in pipeline.hip)
      if (flag) atomicOr(&lds.flags, flag);
      lds.row[i] = flag ? 0u : uint32_t(pick_count(int64_t(deg), k, replace));
    }
  }
}

template <typename IdT, typename PtrT>
__global__ __launch_bounds__(kOneBlock) void one_block_kernel(OneBlockBatch q, TierView<PtrT> indptr, TierView<IdT> indices) {
  __shared__ OneBlockLds lds;
  const auto publish = [&](int word, int64_t v) {
    q.sizes[word] = v;
    if (q.host_sizes) mirror_to_host(q.host_sizes + word, v);
  };
  for (int e = threadIdx.x; e < kOneSlots; e += kOneBlock) lds.table[e] = ~0ull;
  if (threadIdx.x == 0) publish(0, q.n_seeds);
  int s = int(q.n_seeds);  // rows of the hop
  int found = 0;           // ids of the frontier so far
  int begin = 0;           // the hop's first position
  for (int h = 0; h < q.n_hops; ++h) {
    const int k = q.k[h];
    const int pos0 = begin + (h == 0 ? s : 0);
    const int end = pos0 + s * k;
    if (threadIdx.x == 0) lds.flags = 0;
    __syncthreads();
    if (k <= 8) one_block_picks<IdT, PtrT, 8>(lds, q, h, s, pos0, indptr, indices);
    else if (k <= 16) one_block_picks<IdT, PtrT, 16>(lds, q, h, s, pos0, indptr, indices);
    else if (k <= 32) one_block_picks<IdT, PtrT, 32>(lds, q, h, s, pos0, indptr, indices);
    else one_block_picks<IdT, PtrT, 64>(lds, q, h, s, pos0, indptr, indices);
    __syncthreads();
    // a position is its id's first if the table kept it: ranks in the order of positions
    uint32_t id[kOneItems];
    bool first[kOneItems];
    int c = 0;
#pragma unroll
    for (int j = 0; j < kOneItems; ++j) {
      const int p = begin + int(threadIdx.x) * kOneItems + j;
      const uint16_t slot = p < end ? lds.slot[p] : kOneNoSlot;
      const unsigned long long held = slot != kOneNoSlot ? lds.table[slot] : ~0ull;
      id[j] = uint32_t(held >> 32);
      first[j] = uint32_t(held) == uint32_t(p);
      c += first[j];
    }
    int fresh;
    int rank = found + block_exclusive_scan<kOneBlock, int>(c, &fresh, lds.scan);
#pragma unroll
    for (int j = 0; j < kOneItems; ++j) {
      if (!first[j]) continue;
      lds.rank_at[begin + int(threadIdx.x) * kOneItems + j] = uint16_t(rank);
      lds.front[rank] = id[j];
      static_cast<IdT*>(q.frontier)[rank] = IdT(id[j]);
      ++rank;
    }
    // the rows' first edges
    uint32_t n[kOneItems];
    int edges = 0;
#pragma unroll
    for (int j = 0; j < kOneItems; ++j) {
      const int i = int(threadIdx.x) * kOneItems + j;
      n[j] = i < s ? lds.row[i] : 0u;
      edges += int(n[j]);
    }
    int nnz;
    int off = block_exclusive_scan<kOneBlock, int>(edges, &nnz, lds.scan);
#pragma unroll
    for (int j = 0; j < kOneItems; ++j) {
      const int i = int(threadIdx.x) * kOneItems + j;
      if (i < s) lds.row[i] = uint32_t(off) << 8 | n[j];
      off += int(n[j]);
    }
    if (threadIdx.x == 0) {
      publish(h + 1, found + fresh);
      publish(q.n_hops + 1 + h, nnz);
      publish(2 * q.n_hops + 1 + h, lds.flags);
    }
    __syncthreads();
    IdT* src = static_cast<IdT*>(q.src_local[h]);
    IdT* dst = static_cast<IdT*>(q.dst_local[h]);
    for (int t = threadIdx.x; t < s * k; t += kOneBlock) {
      const int i = t / k, l = t - i * k;
      const uint32_t row = lds.row[i];
      if (l >= int(row & 255u)) continue;  // (every pick of a row that has edges is in the table)
      const int o = int(row >> 8) + l;
      src[o] = IdT(lds.rank_at[uint32_t(lds.table[lds.slot[pos0 + t]])]);
      dst[o] = h == 0 ? IdT(lds.rank_at[uint32_t(lds.table[lds.slot[i]])]) : IdT(i);
    }
    __syncthreads();  // the rows' words are rewritten by the next hop
    found += fresh;
    s = found;
    begin = end;
  }
}

}  // namespace dgs
#endif
