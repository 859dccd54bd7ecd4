/*
 * gridburst.hpp -- rounds of small frontiers run back to back in one launch
 * of resident workgroups (the grid bursts of BFS and SSSP).
 *
 * A long-diameter graph has thousands of rounds of a few thousand arcs, and a
 * round as launches costs their boundaries (25-40 us) for microseconds of
 * memory work.  In a burst a round costs its dependent memory round trips and
 * one exchange between the workgroups.  What bounds it is a wave's
 * instruction and latency chain, not bandwidth, so:
 *  - a workgroup appends what it discovers to its own list segment, counted in
 *    LDS; a wave takes kGroup entries and gives each arc a lane;
 *  - an entry of a list of at most kInline arcs carries the arcs themselves,
 *    loaded while the vertex's claim is in flight;
 *  - the exchange is the barrier: one word per workgroup, which every
 *    workgroup polls;
 *  - where the device holds four times as many, four times as many
 *    workgroups are launched and every fourth works: workgroups are dealt to
 *    the eight dies round robin, so those sit on two dies and hand the lists,
 *    claims and words to one another through two L2s (any other placement
 *    only costs time).
 * Everything the workgroups exchange is written and read with agent-scope
 * atomics, so no L2 is written back or invalidated.
 */
#pragma once

#include <algorithm>
#include <initializer_list>

#include "traverse.hpp"

namespace sg::gb {

using namespace sg::trav;

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
constexpr int kBig = 64;     /* lists this long are cut into pieces, a wave per piece */
constexpr int kPiece = 256;  /* arcs of a piece: four per lane */
constexpr int kInline = 4;   /* lists up to this long are carried by their entry */
constexpr int kGroup = 64 / kInline; /* entries a wave takes at a time, a lane per arc */
constexpr int kMaxWgs = 1024;
constexpr int kStride = 4;
/* BFS, 3001 x 2999 grid: 16 workgroups 26.0 ms (on one die), 32 23.9 on one
 * die and 22.7 on two, 64 30.2 and 23.0 */
constexpr int kDefaultWgs = 32;

/* pieces of the next round's long list (three rotating copies: the copy a
 * round adds into was cleared two rounds earlier) */
struct alignas(128) Sums {
  unsigned long long npieces;
  unsigned long long pad[15];
};

/* a workgroup's figures of one round: entries of its segment, discoveries
 * (the entries, and the vertices cut into pieces), pieces, arcs and largest
 * degree of the discoveries */
struct Local {
  uint32_t cnt, disc, mx, npieces;
  unsigned long long deg;
};

/* a wave's share of them: the same in every lane */
struct Acc {
  uint32_t disc, mx, npieces;
  unsigned long long deg;
};

/* The word of a workgroup and round: the round's epoch (8 bits), whether the
 * figures are in the wide slot (1), entries of the segment, which are then
 * the discoveries (15), their arcs (24), their largest degree (16). */
constexpr int kCntBits = 15, kDegBits = 24, kMxBits = 16;
struct alignas(32) Wide { /* a round with long lists, or figures beyond the word's fields */
  unsigned long long disc, deg, mx, cnt; /* cnt: segment entries | pieces << 32 */
};
constexpr unsigned int kPiecesClamp = 1u << 20; /* above every capacity: the burst then ends */

struct Exchange {
  Sums* sums;                /* [3] */
  unsigned long long* slots; /* [2][kMaxWgs] */
  Wide* wide;                /* [2][kMaxWgs] */
  uint32_t* stop;            /* a wait ran out */
  uint64_t wait_ticks;
};

struct Totals {
  unsigned long long disc, deg, mx, npieces;
  uint32_t most; /* entries of the longest segment */
};

/* Entry p of workgroup w's segment: the segments are interleaved by groups of
 * kGroup entries, so that a round's entries lie in a few pages whatever the
 * segments' capacity. */
__device__ __forceinline__ int64_t entry_at(uint32_t w, uint32_t p, uint32_t wgs) {
  return (int64_t)((p / kGroup) * wgs + w) * kGroup + p % kGroup;
}

/* Add a wave's figures to its workgroup's (LDS). */
__device__ __forceinline__ void add_local(Local* l, const Acc& acc) {
  if (acc.disc && lane_id() == 0) {
    atomicAdd(&l->disc, acc.disc);
    atomicAdd(&l->deg, acc.deg);
    atomicMax(&l->mx, acc.mx);
    if (acc.npieces) atomicAdd(&l->npieces, acc.npieces);
  }
}

/* First wave of the workgroup, once the stores of all its waves have
 * completed: publish the workgroup's word, wait for every workgroup's, and
 * sum them; s_n gets the entries of each segment and the local figures start
 * again from zero.  The words hand every workgroup the round's totals in the
 * round trip of the barrier (0.5-1.0 us for 16-32 workgroups of one die; an
 * arrival counter, a generation word and then the totals took 2.0-2.7).  Two
 * rotating copies: a workgroup writes a copy again only after every workgroup
 * has read its previous contents.  The wait is bounded: past wait_ticks of
 * the constant-rate clock `stop` is raised and every workgroup leaves.
 * False: the wait ran out, here or elsewhere.  `extra` takes part in the
 * maximum with the degrees (callers that have no use for those). */
__device__ __forceinline__ bool exchange(const Exchange& x, Local* local, int round, uint32_t rank, uint32_t wgs,
                                         uint32_t* s_n, Totals& tot, unsigned long long extra = 0) {
  const int lane = lane_id();
  unsigned long long* slots = x.slots + (int64_t)(round & 1) * kMaxWgs;
  Wide* wide = x.wide + (int64_t)(round & 1) * kMaxWgs;
  const uint32_t epoch = (uint32_t)(round + 1) & 0xFFu;
  const Local l = *local;
  const unsigned long long mx = extra > l.mx ? extra : (unsigned long long)l.mx;
  const bool w = l.npieces || l.cnt >= (1u << kCntBits) || l.deg >= (1ull << kDegBits) || mx >= (1ull << kMxBits);
  if (w) { /* the wide slot completes before the word says so */
    if (lane == 0) {
      const uint32_t np = l.npieces > kPiecesClamp ? kPiecesClamp : l.npieces;
      put_coherent(&wide[rank].disc, (unsigned long long)l.disc);
      put_coherent(&wide[rank].deg, l.deg);
      put_coherent(&wide[rank].mx, mx);
      put_coherent(&wide[rank].cnt, (unsigned long long)l.cnt | (unsigned long long)np << 32);
    }
    wait_stores_complete();
  }
  if (lane == 0) {
    unsigned long long v = (unsigned long long)epoch << 56;
    v |= w ? 1ull << 55
           : (unsigned long long)l.cnt << (kDegBits + kMxBits) | l.deg << kMxBits | mx;
    put_coherent(&slots[rank], v);
    *local = Local{0, 0, 0, 0, 0};
  }
  tot = Totals{0, 0, 0, 0, 0};
  const uint64_t t0 = wall_clock64();
  for (uint32_t b = 0; b < wgs; b += 64) {
    const bool in = b + lane < wgs;
    unsigned long long v = 0;
    for (uint32_t poll = 1;; ++poll) {
      if (in) v = atomic_load(&slots[b + lane]);
      if (!ballot(in && (uint32_t)(v >> 56) != epoch)) break;
      if (poll % 64) continue; /* the bound on the wait, now and then */
      uint32_t leave = 0;
      if (lane == 0) {
        if ((uint64_t)(wall_clock64() - t0) > x.wait_ticks) atomic_or(x.stop, 1u);
        leave = atomic_load(x.stop);
      }
      if (ballot(leave != 0)) return false;
    }
    const bool far = (v >> 55) & 1ull;
    uint32_t c = (uint32_t)(v >> (kDegBits + kMxBits)) & ((1u << kCntBits) - 1);
    if (!ballot(far)) { /* 64 sums of 15 and of 24 bits stay below 2^32 */
      const uint32_t sum = wave_sum_u32(c), top = wave_max_u32((uint32_t)v & ((1u << kMxBits) - 1));
      tot.disc += sum;
      tot.deg += wave_sum_u32((uint32_t)(v >> kMxBits) & ((1u << kDegBits) - 1));
      tot.mx = top > tot.mx ? top : tot.mx;
    } else {
      unsigned long long d = c, g = (v >> kMxBits) & ((1ull << kDegBits) - 1), m = v & ((1ull << kMxBits) - 1);
      unsigned long long np = 0;
      if (far) {
        const Wide* q = wide + b + lane;
        d = atomic_load(&q->disc);
        g = atomic_load(&q->deg);
        m = atomic_load(&q->mx);
        np = atomic_load(&q->cnt);
        c = (uint32_t)np;
        np >>= 32;
      }
      m = wave_max_u64(m);
      tot.disc += wave_sum_u64(d);
      tot.deg += wave_sum_u64(g);
      tot.npieces += wave_sum_u64(np);
      tot.mx = m > tot.mx ? m : tot.mx;
    }
    if (in) s_n[b + lane] = c;
    const uint32_t most = wave_max_u32(c);
    tot.most = most > tot.most ? most : tot.most;
  }
  return true;
}

/* The group of entries that step k of a wave takes: group k of segment w goes
 * to workgroup (w + k) % wgs (a power of two), so that a long segment is
 * spread over all of them and nobody has to search for its share. */
__device__ __forceinline__ uint32_t segment_of(uint32_t k, uint32_t rank, uint32_t wgs) {
  return (rank - k) & (wgs - 1);
}

/* before each burst: the flag, the piece counters and the words' epochs */
static __global__ void reset_kernel(Exchange x, int32_t wgs) {
  if (threadIdx.x == 0) *x.stop = 0u;
  if (threadIdx.x < 3) x.sums[threadIdx.x].npieces = 0ull;
  for (int i = threadIdx.x; i < 2 * wgs; i += blockDim.x) x.slots[(i & 1) * kMaxWgs + (i >> 1)] = 0ull;
}

/* --------------------------------------------------------- host side --- */
/* List capacities of a burst whose rounds have at most `arcs` arcs.  While the
 * discoveries' arcs stay within that, their pieces number at most arcs / 256
 * + arcs / 64; a segment holds a workgroup's even share of one discovery per
 * arc, and some.  A round that needs more of either ends the burst. */
inline int64_t seg_cap(int64_t arcs, int wgs) { return (arcs / wgs + 1024) / kGroup * kGroup; }
inline int64_t cap_pieces(int64_t arcs) { return arcs / 32 + 64; }

/* Workgroups of a burst (a power of two; all resident at once, `occ` per
 * compute unit) and the stride between them in the launch. */
struct Plan {
  int wgs, stride;
};
inline Plan plan(sg_device_t dev, int occ, int wanted) {
  const int fit = dev->cus * std::max(1, occ);
  int w = std::min(std::min(wanted > 0 ? wanted : kDefaultWgs, fit), kMaxWgs);
  while (w & (w - 1)) w &= w - 1;
  return Plan{w, w * kStride <= fit ? kStride : 1};
}

/* One allocation for all of a workspace's burst buffers (an allocation costs
 * a first pass on a graph tens of microseconds): its parts, 256 bytes apart. */
struct Part {
  void** p;
  size_t bytes;
};
inline int alloc_parts(sg_device_t dev, void** base, std::initializer_list<Part> parts) {
  auto room = [](size_t b) { return (b + 255) / 256 * 256; };
  size_t total = 0;
  for (const Part& q : parts) total += room(q.bytes);
  SG_TRY(alloc_device(dev, base, total));
  char* at = static_cast<char*>(*base);
  for (const Part& q : parts) {
    *q.p = at;
    at += room(q.bytes);
  }
  return SG_OK;
}
constexpr size_t kSumsBytes = 3 * sizeof(Sums), kSlotsBytes = 2 * kMaxWgs * sizeof(unsigned long long),
                 kWideBytes = 2 * kMaxWgs * sizeof(Wide), kStopBytes = 128;

} // namespace sg::gb
