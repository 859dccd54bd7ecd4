/*
 * sssp.hip -- single-source shortest paths for gfx950 (SSSP::run,
 * algorithms/sssp.hpp:152-210).
 *
 * Label-correcting relaxation, as the reference: a round relaxes all arcs of
 * its frontier with an atomic minimum on the tentative distance
 * (sssp.hpp:180-189, sync/atomics.hpp:76-81) and vertices whose distance
 * dropped become dirty again (the filter of sssp.hpp:192-196 only
 * deduplicates them, which a bitmap does by construction).  The reference
 * relaxes every dirty vertex each round (frontier Bellman-Ford); here a round
 * takes only the dirty vertices with distance below a threshold T (the near
 * set) and defers the rest, raising T to (smallest deferred distance) + delta
 * when the near set runs dry -- the bucket order of delta-stepping, which
 * relaxes far fewer arcs on weighted graphs.  delta = infinity is the
 * reference's schedule: every dirty vertex each round, exactly so in launched
 * rounds and one workgroup's bursts; a grid burst's round holds a vertex once
 * for every time that the round before lowered it.  Within a bucket, light iterations relax only the
 * arcs lighter than delta and one heavy iteration the others; the adjacency is
 * read from a light-first copy (per vertex the light arcs, then the heavy
 * ones) so each phase reads only its own arcs.  Each round reads its frontier
 * through the degree-class queues (thread / wave / workgroup bins), relaxes
 * with a plain-load pre-check before the atomic, and marks improved vertices
 * dirty with a test-then-OR.  Shortest distances are unique, so the result does not
 * depend on delta or on the relaxation order.
 *
 * Distances have the weights' 4-byte type: uint32 weights use integer min,
 * float weights (non-negative) compare through their bit patterns.  The
 * unreached value is n+1 in that type (sssp.hpp:43), and so is the value that
 * distances start from: a vertex whose distance is n+1 or more stays
 * unreached, as in the reference.
 */
#include <algorithm>
#include <cmath>
#include <limits>
#include <cstring>

#include "gridburst.hpp"
#include "traverse.hpp"

using namespace sg::trav;
namespace gb = sg::gb;

namespace {

template<typename W>
struct DistOps;
template<>
struct DistOps<uint32_t> {
  static constexpr bool is_float = false;
  __host__ __device__ static uint32_t bits(uint32_t x) { return x; }
  __host__ __device__ static uint32_t value(uint32_t b) { return b; }
};
template<>
struct DistOps<float> {
  static constexpr bool is_float = true;
  __host__ __device__ static uint32_t bits(float x) { return __builtin_bit_cast(uint32_t, x); }
  __host__ __device__ static float value(uint32_t b) { return __builtin_bit_cast(float, b); }
};

template<typename OffT, typename W>
struct SsspArgs {
  const int32_t* cols;
  const W* w;
  uint32_t* dist; /* distance bits */
  uint64_t* next_bm;
  int64_t w0;
  QEntry* qin[3];
  const QueueHdr* qin_hdr;
  /* heavy rounds that pull (light-first adjacency of an undirected graph) */
  const OffT* off;
  const int32_t* light;      /* light arcs per vertex */
  const uint64_t* settled;   /* every vertex settled by a finished bucket (including the current one) */
  const uint64_t* frontier;  /* the current bucket's settled set */
  int64_t n;
};

/* Device-resident control block of the round loop (written only by
 * the last workgroup of sssp_select_kernel; kernel boundaries order the
 * accesses). */
struct SsspCtl {
  uint32_t T_bits;    /* threshold: near = distance below T */
  int32_t done;       /* no dirty vertex left: later iterations are no-ops */
  int32_t relax;      /* the current iteration relaxes (its near set is not empty) */
  int32_t rounds;     /* iterations that relaxed so far */
  int32_t heavy;      /* the current iteration relaxes the heavy arcs of the bucket's settled set */
  int32_t heavy_next; /* the next iteration is the heavy one */
  int32_t r_pending;  /* vertices were relaxed in this bucket since its heavy iteration */
  int32_t pull;       /* the current (heavy) iteration pulls into the vertices not yet settled */
  int32_t burst;      /* the current (Bellman-Ford) round is small: the write pass's last workgroup runs it
                         and the following small rounds */
  int32_t pad1;
  unsigned long long relaxed;    /* arcs relaxed so far */
  unsigned long long heavy_done; /* heavy arcs of every settled set so far */
};

struct alignas(64) RoundLog {
  int32_t iter, done, relax, rounds;
  int32_t fail; /* a wait of a grid burst ran out */
  int64_t near_v, near_e;
  unsigned long long relaxed;
};

constexpr int kRing = 8;

/* Light iterations relax the arcs lighter than delta, the heavy iteration of
 * a bucket the others (delta-stepping's light / heavy split: a heavy arc
 * from a settled bucket cannot land inside it, so it is relaxed once).  The
 * adjacency is the light-first copy, and the queue entries already cover only
 * the phase's part of each list, so every visited arc is relaxed. */
constexpr int kPullHead = 32; /* heavy arcs a lane scans alone before the wave helps */

/* Heavy round by pull (undirected graphs; in-arcs are the out-arcs and the
 * weights are symmetric): a heavy arc (u, v) can only lower dist[v] if v is
 * not settled yet (dist[u] >= T - delta and w >= delta give at least T), so
 * each vertex not yet settled takes the minimum of dist[u] + w over its heavy
 * arcs from the bucket's settled set and becomes dirty if that is below its
 * distance.  Every such vertex belongs to one lane, so its distance is
 * written without an atomic, and the settled distances it reads are final.
 * A wave loads 64 words of the settled bitmap and compacts their clear bits;
 * lists longer than kPullHead are finished by the whole wave.  Returns the
 * arcs from the settled set that were relaxed. */
template<typename OffT, typename W>
__device__ __forceinline__ unsigned long long heavy_pull(const SsspArgs<OffT, W>& a) {
  unsigned long long cnt = 0;
  const int lane = lane_id();
  const int64_t gwave = ((int64_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
  const int64_t nwaves = ((int64_t)gridDim.x * kBlock) >> 6;
  const int tail_bits = (int)(a.n & 63);
  for (int64_t base = gwave * 64; base < a.w0; base += nwaves * 64) {
    const int64_t myw = base + lane;
    uint64_t myun = myw < a.w0 ? ~a.settled[myw] : 0ull;
    if (myw == a.w0 - 1 && tail_bits) myun &= (1ull << tail_bits) - 1ull;
    const uint32_t c = (uint32_t)__popcll(myun);
    const uint32_t incl = wave_inclusive_scan(c);
    const uint32_t total = wave_lane(incl, 63);
    for (uint32_t t0 = 0; t0 < total; t0 += 64) {
      const uint32_t t = t0 + lane;
      const int owner = scan_owner(incl, t);
      const uint32_t before = __shfl(incl - c, owner, 64);
      const uint64_t un = shfl_u64(myun, owner);
      const bool active = t < total;
      int64_t v = 0, j = 0, e = 0;
      uint32_t dv = 0, best = 0xFFFFFFFFu;
      if (active) {
        v = (base + owner) * 64 + select_bit(un, t - before);
        j = (int64_t)a.off[v] + a.light[v];
        e = (int64_t)a.off[v + 1];
        dv = a.dist[v];
        best = dv;
        const int64_t he = e - j > kPullHead ? j + kPullHead : e;
        for (; j < he; j += 4) { /* four ids, then four bitmap probes, then the hits' distances */
          uint32_t u[4];
          bool h[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) u[k] = j + k < he ? (uint32_t)a.cols[j + k] : 0u;
#pragma unroll
          for (int k = 0; k < 4; ++k) h[k] = j + k < he && test_bit(a.frontier, u[k]);
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (h[k]) {
              ++cnt;
              const uint32_t nb = DistOps<W>::bits(DistOps<W>::value(a.dist[u[k]]) + a.w[j + k]);
              best = nb < best ? nb : best;
            }
        }
        if (j > he) j = he;
      }
      uint64_t pending = ballot(active && j < e);
      while (pending) {
        const int k2 = __ffsll((unsigned long long)pending) - 1;
        pending &= pending - 1;
        const int64_t jb = (int64_t)wave_lane((uint64_t)j, k2), je = (int64_t)wave_lane((uint64_t)e, k2);
        uint32_t m = 0xFFFFFFFFu;
        for (int64_t jj = jb + lane; jj < je; jj += 64) {
          const uint32_t u = (uint32_t)a.cols[jj];
          if (test_bit(a.frontier, u)) {
            ++cnt;
            const uint32_t nb = DistOps<W>::bits(DistOps<W>::value(a.dist[u]) + a.w[jj]);
            m = nb < m ? nb : m;
          }
        }
        m = ~(uint32_t)wave_max_u64(~(unsigned long long)m); /* wave minimum */
        if (lane == k2) best = m < best ? m : best;
      }
      if (active && best < dv) {
        a.dist[v] = best;
        atomic_or(&a.next_bm[v >> 6], 1ull << (v & 63));
      }
    }
  }
  return cnt;
}

template<typename OffT, typename W>
__global__ void __launch_bounds__(kBlock) relax_kernel(SsspArgs<OffT, W> a, const SsspCtl* ctl,
                                                       unsigned long long* relax_slots) {
  if (ctl->done || !ctl->relax) return;
  unsigned long long cnt = 0;
  if (ctl->pull) {
    cnt = heavy_pull(a);
  } else {
    for_each_queued_arc<OffT>(a.qin, a.qin_hdr, a.cols, [&](uint32_t u, uint32_t v, int64_t e) {
      const W wt = a.w[e];
      ++cnt;
      /* a stale dist[u] is an upper bound: u is dirty again if it improved */
      const W du = DistOps<W>::value(a.dist[u]);
      const W nd = du + wt;
      const uint32_t nb = DistOps<W>::bits(nd);
      if (nb < a.dist[v]) {
        const uint32_t old = atomic_min(&a.dist[v], nb);
        if (nb < old) {
          const uint64_t bit = 1ull << (v & 63);
          if (!(a.next_bm[v >> 6] & bit)) atomic_or(&a.next_bm[v >> 6], bit);
        }
      }
    });
  }
  /* arcs relaxed in this phase: one atomic per workgroup into 64 slots */
  __shared__ unsigned long long red[kBlock / 64];
  cnt = wave_sum_u64(cnt);
  if (lane_id() == 0) red[threadIdx.x >> 6] = cnt;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t = 0;
    for (int w = 0; w < kBlock / 64; ++w) t += red[w];
    if (t) atomic_add(&relax_slots[(blockIdx.x % kSlots) * 16], t);
  }
}

/* The light-first adjacency: a wave per vertex writes the arcs lighter than
 * dlt from the front of the vertex's range (in order) and the others from the
 * back, and records the light count. */
template<typename OffT, typename W>
__global__ void __launch_bounds__(kBlock) split_build_kernel(const OffT* off, const int32_t* cols, const W* w,
                                                             int64_t n, W dlt, int32_t* scols, W* sw,
                                                             int32_t* light, unsigned long long* heavy_total) {
  const int lane = lane_id();
  const int64_t gwave = ((int64_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
  const int64_t nwaves = ((int64_t)gridDim.x * kBlock) >> 6;
  unsigned long long heavy = 0; /* lane 0: heavy arcs of the wave's vertices */
  for (int64_t v = gwave; v < n; v += nwaves) {
    const int64_t b = (int64_t)off[v], e = (int64_t)off[v + 1];
    int64_t front = b, back = e;
    for (int64_t j0 = b; j0 < e; j0 += 64) {
      const int64_t j = j0 + lane;
      const bool ok = j < e;
      int32_t c = 0;
      W x = 0;
      if (ok) {
        c = cols[j];
        x = w[j];
      }
      const bool lt = ok && x < dlt, hv = ok && !(x < dlt);
      const uint64_t ml = ballot(lt), mh = ballot(hv);
      if (lt) {
        const int64_t p = front + lanes_below(ml);
        scols[p] = c;
        sw[p] = x;
      }
      if (hv) {
        const int64_t p = back - 1 - lanes_below(mh);
        scols[p] = c;
        sw[p] = x;
      }
      front += __popcll(ml);
      back -= __popcll(mh);
    }
    if (lane == 0) {
      light[v] = (int32_t)(front - b);
      heavy += (unsigned long long)(e - front);
    }
  }
  if (lane == 0 && heavy) atomic_add(heavy_total, heavy);
}

/* per-block counters of the split, one 128-byte line per slot */
struct alignas(128) SplitSlot {
  unsigned long long far_count;
  unsigned int far_min; /* distance bits; 4-byte distances order like their bits */
  unsigned int pad0;
  unsigned long long pad[14];
};

/* near = dirty vertices with distance < T (moved out of the dirty bitmap into
 * the round's frontier bitmap); count and smallest distance of the rest.  One
 * word per thread (word i), its dirty bits walked by the lane itself: on the
 * dense bands of a grid this beats spreading them over the wave.  The heavy
 * iteration's frontier is the bucket's settled set instead.  All threads of
 * the workgroup call. */
template<typename W>
__device__ __forceinline__ void split_word(int64_t i, int64_t w0, bool heavy_next, bool bellman, uint32_t T_bits,
                                           uint64_t* dirty, uint64_t* near_bm, uint64_t* settled,
                                           uint64_t* settled_all, const uint32_t* dist, SplitSlot* slots) {
  if (heavy_next) {
    if (i < w0) {
      const uint64_t r = settled[i];
      near_bm[i] = r;
      if (r) {
        settled[i] = 0;
        settled_all[i] |= r;
      }
    }
    return;
  }
  if (bellman) { /* the reference's schedule: T is the largest weight, so every dirty vertex is near */
    if (i < w0) {
      const uint64_t f = dirty[i];
      near_bm[i] = f;
      if (f) {
        dirty[i] = 0;
        settled[i] |= f;
      }
    }
    return;
  }
  const W T = DistOps<W>::value(T_bits);
  unsigned long long far = 0;
  unsigned int fmin = 0xFFFFFFFFu;
  if (i < w0) {
    const uint64_t f = dirty[i];
    uint64_t nb = 0;
    for (uint64_t rest = f; rest; rest &= rest - 1) {
      const int b = __ffsll((unsigned long long)rest) - 1;
      const uint32_t db = dist[i * 64 + b];
      if (DistOps<W>::value(db) < T) nb |= 1ull << b;
      else fmin = db < fmin ? db : fmin;
    }
    near_bm[i] = nb;
    if (nb) {
      dirty[i] = f & ~nb;
      settled[i] |= nb;
    }
    far = (unsigned long long)__popcll(f & ~nb);
  }
  far = wave_sum_u64(far);
  unsigned long long m = wave_max_u64(~(unsigned long long)fmin); /* min via max of complement */
  fmin = ~(unsigned int)m;
  if (lane_id() == 0 && (far || fmin != 0xFFFFFFFFu)) {
    SplitSlot* sl = slots + (blockIdx.x % kSlots);
    if (far) atomic_add(&sl->far_count, far);
    atomic_min(&sl->far_min, fmin);
  }
}

__global__ void split_slots_reset_kernel(SplitSlot* slots, const SsspCtl* ctl) {
  if (ctl->done) return;
  const int i = threadIdx.x;
  if (i < kSlots) {
    slots[i].far_count = 0;
    slots[i].far_min = 0xFFFFFFFFu;
  }
}

/* ------------------------------------------------------------ bursts --- */
/* Rounds of the reference's schedule (every dirty vertex relaxed each round)
 * on a graph of long diameter have small frontiers, and each costs a
 * selection, a write and a relax launch.  When a round has at most
 * burst_arcs arcs, the last workgroup of the write pass relaxes it and the
 * following rounds back to back, one workgroup barrier per round, for as
 * long as they stay small.  The frontier moves between two lists of (first
 * arc, vertex, degree) entries; a round lays the list's arcs end to end (an
 * exclusive scan of the lengths in LDS) and each thread takes every
 * kBlock-th arc, finding its entry by binary search.  A relaxation that
 * lowers dist[v] sets v's dirty bit; the lane that set it appends v to the
 * next list.  Before a round the bits of its list are cleared (the split's
 * job in the launched rounds), so a vertex lowered again during its own
 * round is relaxed again in the next.  The burst stops when a round lowers
 * nothing or the next list is too large: its vertices keep their dirty bits
 * and the next iteration's selection takes them from the bitmap. */
/* what the bursts tell of their rounds: vertices and arcs of round r at
 * [2 r] and [2 r + 1], zeros where a round was a launch (the iteration's
 * record has it).  A round's vertices are its list's entries: a grid burst
 * lists a vertex again when it is lowered again in the same round. */
__device__ __forceinline__ void record_round(unsigned long long* rounds, int64_t r, unsigned long long vertices,
                                             unsigned long long arcs) {
  if (!rounds || r >= SG_MAX_LEVELS_RECORDED) return;
  rounds[2 * r] = vertices;
  rounds[2 * r + 1] = arcs;
}
constexpr int kSsspBurstDefault = 4096;
/* With far lists the grid bursts take the rounds from the start but for those
 * of a few arcs, which one workgroup takes faster, to the end on a path
 * (20,000 vertices: 53.6 ms, in a grid burst 67), and hands over as the queues
 * of the round that is larger. */
constexpr int64_t kTinyArcs = 8;
constexpr int kSsspBurstMax = 8192; /* entries (and arcs) of a burst round; LDS for its scan */

template<typename OffT, typename W>
struct SsspBurst {
  const OffT* off;
  const int32_t* cols;
  const W* w;
  uint32_t* dist;
  uint64_t* dirty;
  QEntry* q[3]; /* the round's queues (written by this launch) */
  const QueueHdr* hdr;
  QEntry* list[2]; /* kSsspBurstMax entries each */
  int64_t burst_arcs;
  int hand_over; /* a round beyond burst_arcs goes to the queues (out_hdr counts them) and not to the bitmap */
  QueueHdr* out_hdr;
  Tuning tune;
  unsigned long long* relax_slots;
  unsigned long long* rounds; /* record_round's */
  uint32_t* arrive; /* kArriveWords zeroed words */
};

template<typename OffT, typename W>
__device__ __forceinline__ void sssp_burst(const SsspBurst<OffT, W>& b, SsspCtl* ctl) {
  __shared__ uint32_t s_pref[kSsspBurstMax + 1];
  __shared__ uint32_t s_wtot[kBlock / 64];
  __shared__ uint32_t s_next, s_next_arcs;
  __shared__ uint32_t s_class[3];
  __shared__ unsigned long long s_deg, s_maxdeg;
  const QueueHdr h = *b.hdr;
  const uint32_t n0 = h.count[0], n1 = h.count[1];
  uint32_t cnt = h.count[0] + h.count[1] + h.count[2];
  const int lane = lane_id(), wv = threadIdx.x >> 6;
  /* the first round's entries, the three class queues, gathered into the
   * list that the second round writes */
  for (uint32_t i = threadIdx.x; i < cnt; i += kBlock)
    b.list[1][i] = i < n0 ? b.q[0][i] : (i < n0 + n1 ? b.q[1][i - n0] : b.q[2][i - n0 - n1]);
  __syncthreads();
  unsigned long long arcs = 0;
  int32_t rounds = 0;
  const int32_t first_round = ctl->rounds - 1; /* counted by the selection */
  for (int it = 0;; ++it) {
    const QEntry* in = b.list[(it + 1) & 1];
    QEntry* out = b.list[it & 1];
    auto entry = [&](uint32_t i) -> QEntry { return in[i]; };
    /* exclusive scan of the lengths: thread t owns a run of kPer entries */
    constexpr int kPer = kSsspBurstMax / kBlock;
    const uint32_t first = threadIdx.x * kPer;
    uint32_t run = 0;
    for (int k = 0; k < kPer; ++k)
      if (first + k < cnt) run += (uint32_t)entry(first + k).len;
    const uint32_t incl = wave_inclusive_scan(run);
    if (lane == 63) s_wtot[wv] = incl;
    if (threadIdx.x == 0) s_next = s_next_arcs = 0;
    __syncthreads();
    uint32_t base = 0, total = 0;
    for (int w = 0; w < kBlock / 64; ++w) {
      base += w < wv ? s_wtot[w] : 0u;
      total += s_wtot[w];
    }
    uint32_t pos = base + incl - run;
    for (int k = 0; k < kPer; ++k)
      if (first + k < cnt) {
        s_pref[first + k] = pos;
        pos += (uint32_t)entry(first + k).len;
      }
    if (threadIdx.x == 0) {
      s_pref[cnt] = total;
      record_round(b.rounds, first_round + rounds, rounds == 0 ? h.nvert : (unsigned long long)cnt, total);
    }
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < total; t += kBlock) {
      uint32_t lo = 0, hi = cnt; /* s_pref[lo] <= t < s_pref[hi] */
      while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (s_pref[mid] <= t) lo = mid;
        else hi = mid;
      }
      const QEntry e = entry(lo);
      const int64_t j = e.start + (int64_t)(t - s_pref[lo]);
      const uint32_t u = (uint32_t)e.v, v = (uint32_t)b.cols[j];
      /* distances lowered earlier in the burst were lowered by atomics at L2:
       * read them with agent-scope loads, past any older copy in L1 */
      const uint32_t du = __hip_atomic_load(&b.dist[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const uint32_t nb = DistOps<W>::bits(DistOps<W>::value(du) + b.w[j]);
      if (nb < __hip_atomic_load(&b.dist[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) &&
          nb < atomic_min(&b.dist[v], nb)) {
        const uint64_t bit = 1ull << (v & 63);
        if (!(atomic_or(&b.dirty[v >> 6], bit) & bit)) {
          const int64_t s0 = (int64_t)b.off[v], d = (int64_t)(b.off[v + 1] - b.off[v]);
          if (d > 0) { /* a vertex without arcs stays dirty for the selection */
            const uint32_t p = atomicAdd(&s_next, 1u);
            if (p < (uint32_t)kSsspBurstMax) {
              QEntry q;
              q.start = s0;
              q.v = (int32_t)v;
              q.len = (int32_t)d;
              out[p] = q;
            }
            atomicAdd(&s_next_arcs, (uint32_t)(d < (int64_t)kSsspBurstMax ? d : kSsspBurstMax));
          }
        }
      }
    }
    __syncthreads();
    arcs += total;
    ++rounds;
    const uint32_t nc = s_next, na = s_next_arcs;
    /* hand back (the next list keeps its dirty bits) or stop */
    if (nc == 0 || nc > (uint32_t)kSsspBurstMax || (int64_t)na > b.burst_arcs) break;
    for (uint32_t i = threadIdx.x; i < nc; i += kBlock) {
      const uint32_t v = (uint32_t)out[i].v;
      atomic_and(&b.dirty[v >> 6], ~(1ull << (v & 63)));
    }
    __syncthreads();
    cnt = nc;
  }
  const uint32_t nc = s_next;
  if (b.hand_over && nc != 0 && nc <= (uint32_t)kSsspBurstMax) { /* uniform: the same in every thread */
    const QEntry* out = b.list[(rounds - 1) & 1];
    if (threadIdx.x < 3) s_class[threadIdx.x] = 0;
    if (threadIdx.x == 0) s_deg = s_maxdeg = 0;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < nc; i += kBlock) {
      const QEntry e = out[i];
      atomic_and(&b.dirty[(uint32_t)e.v >> 6], ~(1ull << (e.v & 63)));
      const int cls = e.len < b.tune.t_medium ? 0 : e.len < b.tune.t_large ? 1 : 2;
      const uint32_t pieces = cls < 2 ? 1u : (uint32_t)((e.len + b.tune.chunk - 1) / b.tune.chunk);
      const uint32_t at = atomicAdd(&s_class[cls], pieces);
      if (cls < 2) b.q[cls][at] = e;
      for (uint32_t c = 0; cls == 2 && c < pieces; ++c)
        b.q[2][at + c] = QEntry{e.start + (int64_t)c * b.tune.chunk, e.v,
                                min(b.tune.chunk, e.len - (int32_t)c * b.tune.chunk)};
      atomicAdd(&s_deg, (unsigned long long)e.len);
      atomicMax(&s_maxdeg, (unsigned long long)e.len);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      QueueHdr o{};
      for (int k = 0; k < 3; ++k) o.count[k] = s_class[k];
      o.nvert = nc;
      o.deg = s_deg;
      o.maxdeg = s_maxdeg;
      *b.out_hdr = o;
      record_round(b.rounds, first_round + rounds, nc, s_deg);
      ctl->rounds += rounds;
      ctl->relaxed += arcs + s_deg - (unsigned long long)h.deg;
      ctl->burst = 0;
      atomic_add(&b.relax_slots[0], arcs);
    }
    return;
  }
  if (threadIdx.x == 0) {
    /* the selection counted the first round; the relax launch has nothing left */
    ctl->rounds += rounds - 1;
    ctl->relaxed += arcs - (unsigned long long)h.deg;
    ctl->relax = 0;
    ctl->burst = 0;
    atomic_add(&b.relax_slots[0], arcs);
  }
}

template<typename OffT, typename W>
__global__ void __launch_bounds__(kBlock) near_write_kernel(CompactArgs<OffT> a, SsspBurst<OffT, W> b, SsspCtl* ctl) {
  if (ctl->done || !ctl->relax || ctl->pull) return;
  const bool burst = ctl->burst != 0;
  const bool wrote = compact_write_body<OffT>(a, ctl->heavy ? 1 : 0);
  /* a burst round has at most burst_arcs arcs, so few waves write entries and publish them */
  if (!burst || !last_to_arrive<false>(b.arrive, wrote)) return;
  sssp_burst(b, ctl);
}

/* ------------------------------------------------------ small graphs --- */
/* A graph of at most kSmallVerts vertices and kSmallArcs arcs: every round in
 * one launch of one workgroup, with the distances, the lists and the dirty
 * bits in LDS (150 of the CU's 160 KB) and one workgroup barrier per round;
 * only offsets, ids and weights are read from memory.  Launched rounds and
 * grid bursts are bound by launches, exchanges and agent-scope atomics here,
 * this by the rounds' chains of loads and LDS operations (3 us a round on a
 * grid).  Per call, before and after: RMAT of 1,186 arcs 231 -> 38 us, 12,002
 * arcs 333 -> 96, 45,187 (directed, float) 435 -> 163, 85,128 arcs 717 -> 250;
 * grids of 20 x 20 (weights 1 to 7, so that every vertex is reached below
 * n + 1) 320 -> 104, 60 x 70 1,214 -> 350.  The vertices are bounded by
 * LDS; the arcs by the grid bursts' own limit, from which the automatic
 * schedule keeps the order of the launched rounds (here a distance lowered in
 * a round is seen at once, which saves a tenth of the relaxations). */
constexpr int kSmallVerts = 16384;
constexpr int64_t kSmallArcs = 1 << 17;
constexpr int kSmallThreads = 1024, kSmallWaves = kSmallThreads / 64;
constexpr int kSmallHub = 256;                              /* a longer list is cut into pieces of so many arcs */
constexpr int kSmallHubs = (int)(kSmallArcs / kSmallHub);   /* more lists than that are not longer */

struct SmallLog { /* pinned coherent host memory */
  int32_t rounds, fail;
  int64_t reached_v, reached_e;
  unsigned long long relaxed;
  int64_t round_v[SG_MAX_LEVELS_RECORDED], round_e[SG_MAX_LEVELS_RECORDED];
};

template<typename OffT, typename W>
struct SmallArgs {
  const OffT* off;
  const int32_t* cols;
  const W* w;
  uint32_t* dist;
  int32_t n, src;
  uint32_t unreached;
  int32_t max_rounds;
  SmallLog* log;
};

struct SmallShared {
  uint32_t dist[kSmallVerts];
  uint16_t list[2][kSmallVerts];      /* the round's entries and the next one's */
  uint16_t hub[2][kSmallHubs];        /* those of more than kSmallHub arcs */
  uint32_t dirty[2][kSmallVerts / 32]; /* in the next list, by the parity of the round that put it there */
  uint64_t is_hub[kSmallVerts / 64];
  uint8_t mark[kSmallWaves][256];     /* first arc of an entry among a wave's 256: its lane + 1 */
  uint2 ent[kSmallWaves][64];         /* an entry's first arc less the arcs before it; its distance */
  uint32_t cnt[3];                    /* entries (low half) and hubs (high) put by the rounds, in turn */
  unsigned long long arcs[3];
};

/* Relax the (up to) four arcs of each lane, from distances du over weights wt
 * to the vertices y. */
template<typename W>
__device__ __forceinline__ void small_relax4(SmallShared& sh, const uint32_t (&y)[4], const W (&wt)[4],
                                             const uint32_t (&du)[4], const bool (&ok)[4], int r) {
  const int nx = (r + 1) & 1;
  uint64_t ml[4], mh[4];
  uint32_t cl = 0, ch = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    bool fresh = false;
    if (ok[k]) {
      const uint32_t nb = DistOps<W>::bits(DistOps<W>::value(du[k]) + wt[k]);
      if (nb < sh.dist[y[k]] && nb < atomicMin(&sh.dist[y[k]], nb)) {
        const uint32_t bit = 1u << (y[k] & 31);
        fresh = !(atomicOr(&sh.dirty[r & 1][y[k] >> 5], bit) & bit);
      }
    }
    const bool hub = fresh && (sh.is_hub[y[k] >> 6] >> (y[k] & 63) & 1);
    ml[k] = __ballot(fresh && !hub);
    mh[k] = __ballot(hub);
    cl += (uint32_t)__popcll(ml[k]);
    ch += (uint32_t)__popcll(mh[k]);
  }
  if (cl + ch == 0) return;
  uint32_t at = 0;
  if (lane_id() == 0) at = atomicAdd(&sh.cnt[r % 3], cl | ch << 16);
  at = wave_lane(at, 0);
  uint32_t pl = at & 0xffffu, ph = at >> 16;
  const uint64_t me = 1ull << lane_id();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (ml[k] & me) sh.list[nx][pl + lanes_below(ml[k])] = (uint16_t)y[k];
    if (mh[k] & me) sh.hub[nx][ph + lanes_below(mh[k])] = (uint16_t)y[k];
    pl += (uint32_t)__popcll(ml[k]);
    ph += (uint32_t)__popcll(mh[k]);
  }
}

template<typename OffT, typename W>
__global__ void __launch_bounds__(kSmallThreads) sssp_small_kernel(SmallArgs<OffT, W> a) {
  __shared__ SmallShared sh;
  const int lane = lane_id(), wv = threadIdx.x >> 6;
  for (int i = threadIdx.x; i < (a.n + 63) / 64 * 64; i += kSmallThreads) {
    sh.dist[i] = i == a.src ? 0u : a.unreached;
    int64_t s = 0, e = 0;
    if (i < a.n) list_bounds(a.off, (uint32_t)i, s, e);
    const uint64_t hubs = __ballot(e - s > kSmallHub);
    if (lane == 0) sh.is_hub[i >> 6] = hubs;
    if (lane < 4) sh.dirty[lane & 1][(i >> 6) * 2 + (lane >> 1)] = 0u;
  }
  if (threadIdx.x == 0) {
    int64_t s, e;
    list_bounds(a.off, (uint32_t)a.src, s, e);
    if (e - s > kSmallHub) sh.hub[0][0] = (uint16_t)a.src;
    else sh.list[0][0] = (uint16_t)a.src;
    sh.cnt[2] = e - s > kSmallHub ? 1u << 16 : 1u;
    sh.cnt[0] = 0u;
    sh.arcs[0] = 0ull;
  }
  unsigned long long relaxed = 0;
  int r = 0;
  for (;; ++r) {
    __syncthreads();
    const uint32_t both = sh.cnt[(r + 2) % 3], cnt = both & 0xffffu, hubs = both >> 16;
    if (threadIdx.x == 0) {
      /* the counters of the round after this one: last read a round ago */
      sh.cnt[(r + 1) % 3] = 0u;
      sh.arcs[(r + 1) % 3] = 0ull;
      if (r > 0) {
        const unsigned long long arcs = sh.arcs[(r + 2) % 3];
        relaxed += arcs;
        if (r <= SG_MAX_LEVELS_RECORDED) a.log->round_e[r - 1] = (int64_t)arcs;
      }
      if (both != 0 && r < SG_MAX_LEVELS_RECORDED) a.log->round_v[r] = (int64_t)cnt + hubs;
    }
    if (both == 0 || r >= a.max_rounds) break;
    const int cur = r & 1, was = cur ^ 1;
    unsigned long long arcs = 0;
    /* short lists: a wave lays a group of entries end to end and takes four
     * arcs per lane; the arcs' entries by marking where each one starts */
    uint32_t group = 64;
    while (group > 4 && cnt <= kSmallWaves * (group / 2)) group >>= 1;
    for (uint32_t base = (uint32_t)wv * group; base < cnt; base += kSmallWaves * group) {
      int64_t s = 0, e = 0;
      uint32_t u = 0, du = 0;
      if (lane < (int)group && base + lane < cnt) {
        u = sh.list[cur][base + lane];
        list_bounds(a.off, u, s, e);
        du = sh.dist[u];
        atomicAnd(&sh.dirty[was][u >> 5], ~(1u << (u & 31)));
      }
      const uint32_t len = (uint32_t)(e - s), incl = wave_inclusive_scan(len), excl = incl - len;
      const uint32_t total = wave_lane(incl, 63);
      sh.ent[wv][lane] = make_uint2((uint32_t)s - excl, du);
      arcs += total;
      uint32_t carry = 0;
      for (uint32_t t0 = 0; t0 < total; t0 += 256) {
        *reinterpret_cast<uint32_t*>(&sh.mark[wv][4 * lane]) = 0u;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (len != 0 && excl >= t0 && excl < t0 + 256) sh.mark[wv][excl - t0] = (uint8_t)(lane + 1);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const uint32_t four = *reinterpret_cast<const uint32_t*>(&sh.mark[wv][4 * lane]);
        uint32_t own[4];
        own[0] = four & 0xffu;
#pragma unroll
        for (int k = 1; k < 4; ++k) own[k] = max(own[k - 1], four >> (8 * k) & 0xffu);
        const uint32_t upto = wave_prefix(own[3], [](uint32_t x, uint32_t y) { return max(x, y); });
        uint32_t left = __shfl_up(upto, 1, 64);
        left = max(lane == 0 ? 0u : left, carry);
        carry = max(carry, wave_lane(upto, 63));
        uint32_t y[4], d[4];
        W wt[4];
        bool ok[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint32_t t = t0 + 4 * lane + k;
          ok[k] = t < total;
          const uint2 en = sh.ent[wv][max(own[k], left) - 1];
          const uint32_t j = ok[k] ? en.x + t : 0u;
          y[k] = (uint32_t)a.cols[j];
          wt[k] = a.w[j];
          d[k] = en.y;
        }
        small_relax4<W>(sh, y, wt, d, ok, r);
      }
    }
    /* long lists: their pieces go to the waves in turn */
    uint32_t pbase = 0;
    for (uint32_t i = 0; i < hubs; ++i) {
      const uint32_t u = sh.hub[cur][i];
      int64_t s, e;
      list_bounds(a.off, u, s, e);
      const uint32_t len = (uint32_t)(e - s), np = (len + kSmallHub - 1) / kSmallHub;
      const uint32_t du = sh.dist[u];
      if (threadIdx.x == 0) {
        atomicAnd(&sh.dirty[was][u >> 5], ~(1u << (u & 31)));
        arcs += len;
      }
      for (uint32_t pc = (wv - pbase) % kSmallWaves; pc < np; pc += kSmallWaves) {
        uint32_t y[4], d[4];
        W wt[4];
        bool ok[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint32_t o = pc * kSmallHub + 64 * k + lane;
          ok[k] = o < len;
          const uint32_t j = (uint32_t)s + (ok[k] ? o : 0u);
          y[k] = (uint32_t)a.cols[j];
          wt[k] = a.w[j];
          d[k] = du;
        }
        small_relax4<W>(sh, y, wt, d, ok, r);
      }
      pbase += np;
    }
    if (lane == 0 && arcs != 0) atomicAdd(&sh.arcs[r % 3], arcs);
  }
  uint64_t rv = 0, re = 0;
  for (int i = threadIdx.x; i < a.n; i += kSmallThreads) {
    const uint32_t d = sh.dist[i];
    a.dist[i] = d;
    int64_t s, e;
    list_bounds(a.off, (uint32_t)i, s, e);
    rv += d != a.unreached ? 1u : 0u;
    re += d != a.unreached ? (uint64_t)(e - s) : 0u;
  }
  rv = wave_sum_u64(rv);
  re = wave_sum_u64(re);
  __syncthreads(); /* the marks and entries are read no more */
  unsigned long long* red = reinterpret_cast<unsigned long long*>(sh.ent);
  if (lane == 0) {
    red[2 * wv] = rv;
    red[2 * wv + 1] = re;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    rv = re = 0;
    for (int w = 0; w < kSmallWaves; ++w) {
      rv += red[2 * w];
      re += red[2 * w + 1];
    }
    a.log->rounds = r;
    a.log->fail = sh.cnt[(r + 2) % 3] != 0u ? 1 : 0;
    a.log->reached_v = (int64_t)rv;
    a.log->reached_e = (int64_t)re;
    a.log->relaxed = relaxed;
  }
}

/* automatic delta = half the mean arc weight: of 0.125-1.0 times the mean,
 * the least geometric mean of time / the run's best (1.026) over the 30
 * training graphs the rule below sends to buckets (0.25: 1.18; 1.0: 1.19) */
constexpr double kAutoDeltaFactor = 0.5;

/* The automatic bucket width for a mean arc weight. */
template<typename W>
__host__ __device__ inline double auto_delta(double mean) {
  const double least = DistOps<W>::is_float ? 1e-30 : 1.0, d = kAutoDeltaFactor * mean;
  return d < least ? least : d;
}

/* Threshold after a dry iteration: the smallest deferred distance plus
 * delta, at least one representable step above it. */
template<typename W>
__device__ __forceinline__ uint32_t next_threshold(uint32_t fmin_bits, double delta, double w_max) {
  const W dmin = DistOps<W>::value(fmin_bits);
  const double t = (double)dmin + delta;
  W tn = (W)(t < w_max ? t : w_max);
  if (!(tn > dmin)) {
    /* non-negative finite floats order like their bit patterns: +1 is the next float up */
    if constexpr (DistOps<W>::is_float) tn = DistOps<W>::value(fmin_bits + 1u);
    else tn = dmin + 1u;
  }
  return DistOps<W>::bits(tn);
}

/* ------------------------------------------------------- grid bursts --- */
/* Rounds of the reference's schedule too large for one workgroup but too small
 * to fill the chip -- a 1201 x 1301 grid has thousands of about ten thousand
 * arcs, 42 us each as three launches -- run back to back in one launch of
 * resident workgroups (gridburst.hpp), one exchange per round.  It starts
 * from the queues the write pass of the same iteration wrote and stops when a
 * round lowers nothing or the next one has more than grid_arcs arcs (or needs
 * longer lists): what is left gets its dirty bits back and the next
 * iteration's selection takes it from the bitmap.
 *
 * Every relaxation that lowers dist[v] appends v with the distance it gave, so
 * nothing has to be deduplicated: a vertex lowered twice in a round is listed
 * twice, but the entry with the larger distance lowers nothing that the other
 * does not, so copies do not multiply.  An entry carries vertex and length,
 * distance, and for lists of at most gb::kInline arcs heads and weights,
 * loaded while the minimum is in flight: a round's chain is the entry, the
 * head's distance and list bounds, the minimum with the head's own list, and
 * the store of the next entry.
 *
 * Near and far (the automatic schedule only).  Relaxing every lowered vertex
 * at once, the reference's order, relaxes an arc dozens of times on a grid.
 * With a round at a few microseconds it pays to put off what lies beyond a
 * threshold T (the near-far piles of Davidson, Baxter, Garland and Owens,
 * IPDPS 2014): a vertex lowered to T or more goes to its workgroup's far list
 * instead, and when a round leaves nothing near, T moves to the smallest far
 * distance plus a step and a far pass takes what is below it, dropping what
 * has been lowered since.  The step follows the rounds' sizes: doubled when a
 * bucket's rounds had fewer than kNearFew arcs on average, which cost their
 * latency whatever they hold, halved above kNearMany, where they take several
 * turns of the waves (2,048 / 8,192: 14.8 ms on the grid below, 4,096 /
 * 16,384: 14.0, 8,192 / 32,768: 14.7, 16,384 / 49,152: 27.3 with half the
 * workgroups, where 4,096 / 16,384 took 16.6).
 *
 * 1201 x 1301 grid, u32 weights: 66.6 ms by launches and single-workgroup
 * bursts (364 M relaxations, 42 us a launched round), 14.1 so (24 M, 5.2 us a
 * round). */
constexpr int kSsspGridWgs = 64; /* 32: 15.1 ms, 128: 15.2 */
constexpr int64_t kSsspGridArcs = 1 << 17;
constexpr int64_t kNearFew = 4096, kNearMany = 16384;
/* far entries per workgroup: an even share of a quarter of the vertices; what
 * does not fit waits for the burst's end */
inline uint32_t far_capacity(int64_t n, int wgs) {
  return (uint32_t)std::min<int64_t>(std::max<int64_t>(n / (4 * wgs), 1024), 1 << 18);
}

template<typename OffT, typename W>
struct SsspGrid {
  const OffT* off;
  const int32_t* cols;
  const W* w;
  int64_t m, mean; /* arcs; of a vertex */
  uint32_t* dist;
  uint64_t* dirty;
  QEntry* q[3]; /* the round's queues */
  const QueueHdr* hdr;
  /* [parity]: `total` entries of two words (vertex | length << 32; first
   * arc), then `total` distances, kInline heads and kInline weights per entry */
  uint64_t* list[2];
  int64_t total;
  uint32_t seg_cap;
  QEntry* pieces[2];
  int64_t cap_pieces, grid_arcs;
  uint64_t* far[2]; /* [parity]: far_cap entries per workgroup, vertex | distance << 32 */
  uint32_t far_cap;
  const double* weight_sum; /* of all arcs, for the first step of T; null: no far list */
  double w_max;
  gb::Exchange x;
  unsigned long long* relax_slots;
  unsigned long long* rounds; /* record_round's */
  RoundLog* log;
  uint32_t stride; /* the burst's workgroups are those with blockIdx.x % stride == 0 */
};
constexpr int64_t kSsspGridWords(int64_t total) { return 2 * total + total / 2 + total / 2 * gb::kInline * 2; }

template<typename OffT, typename W>
struct SsspGridOut {
  uint64_t* list;
  uint32_t rank, wgs;
  QEntry* pieces;
  gb::Sums* sums;
  gb::Local* local;
  uint64_t* far; /* the workgroup's far list and its counter (LDS) */
  uint32_t* far_n;
  uint32_t T; /* bits of the threshold (no far list: above every distance) */
};

/* Append this lane's (v, d) to the workgroup's far list (all lanes call). */
template<typename OffT, typename W>
__device__ __forceinline__ void sssp_far_append(const SsspGrid<OffT, W>& a, const SsspGridOut<OffT, W>& o, bool is_far,
                                                uint32_t v, uint32_t d) {
  const uint64_t m = ballot(is_far);
  if (!m) return;
  uint32_t at = 0;
  if (lane_id() == 0) at = atomicAdd(o.far_n, (uint32_t)__popcll(m));
  at = __builtin_amdgcn_readfirstlane(at) + lanes_below(m);
  if (!is_far) return;
  if (at < a.far_cap) o.far[at] = (uint64_t)v | (uint64_t)d << 32;
  else atomic_or(&a.dirty[v >> 6], 1ull << (v & 63)); /* no room: left to the rounds after the burst */
}

/* Append this lane's vertices with their lists (ms[k]: the lanes of the k-th
 * whose lists are short; the caller holds the heads and weights of those of at
 * most kInline arcs). */
template<int K, typename OffT, typename W>
__device__ __forceinline__ void sssp_grid_append(const SsspGrid<OffT, W>& a, const SsspGridOut<OffT, W>& o,
                                                 const uint32_t (&y)[K], const uint32_t (&nb)[K], const bool (&low)[K],
                                                 const int64_t (&vs)[K], const int64_t (&ve)[K],
                                                 const uint32_t (&id)[K][gb::kInline],
                                                 const uint32_t (&wt)[K][gb::kInline], gb::Acc& acc);

/* Relax the (up to) K arcs of each lane: head y[k], distance nb[k] over it. */
template<int K, typename OffT, typename W>
__device__ __forceinline__ void sssp_grid_relax(const SsspGrid<OffT, W>& a, const uint32_t (&y)[K],
                                                const uint32_t (&nb)[K], const bool (&ok)[K],
                                                const SsspGridOut<OffT, W>& o, gb::Acc& acc) {
  uint32_t d[K];
  int64_t vs[K], ve[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    d[k] = 0;
    vs[k] = ve[k] = 0;
    if (ok[k]) {
      d[k] = atomic_load(&a.dist[y[k]]);
      list_bounds(a.off, y[k], vs[k], ve[k]);
    }
  }
  uint32_t id[K][gb::kInline], wt[K][gb::kInline];
  bool low[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    low[k] = ok[k] && nb[k] < d[k];
    if (low[k]) d[k] = atomic_min(&a.dist[y[k]], nb[k]);
    if (low[k] && nb[k] < o.T && ve[k] - vs[k] <= gb::kInline) {
      load_ids4(a.cols, vs[k], a.m, id[k]);
      load_ids4(reinterpret_cast<const int32_t*>(a.w), vs[k], a.m, wt[k]);
    }
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    low[k] = low[k] && nb[k] < d[k] && ve[k] > vs[k]; /* a vertex without arcs has nothing to relax */
    const bool is_far = low[k] && nb[k] >= o.T;
    sssp_far_append(a, o, is_far, y[k], nb[k]);
    low[k] = low[k] && !is_far;
  }
  sssp_grid_append<K>(a, o, y, nb, low, vs, ve, id, wt, acc);
}

template<int K, typename OffT, typename W>
__device__ __forceinline__ void sssp_grid_append(const SsspGrid<OffT, W>& a, const SsspGridOut<OffT, W>& o,
                                                 const uint32_t (&y)[K], const uint32_t (&nb)[K], const bool (&low)[K],
                                                 const int64_t (&vs)[K], const int64_t (&ve)[K],
                                                 const uint32_t (&id)[K][gb::kInline],
                                                 const uint32_t (&wt)[K][gb::kInline], gb::Acc& acc) {
  uint64_t ms[K];
  uint32_t cs = 0;
  bool pieces = false;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const bool big = ve[k] - vs[k] >= gb::kBig;
    ms[k] = ballot(low[k] && !big);
    cs += (uint32_t)__popcll(ms[k]);
    pieces = pieces || (low[k] && big);
  }
  const bool any_pieces = ballot(pieces) != 0;
  if (cs == 0 && !any_pieces) return;
  uint32_t at = 0;
  if (cs) {
    if (lane_id() == 0) at = atomicAdd(&o.local->cnt, cs);
    at = __builtin_amdgcn_readfirstlane(at);
    acc.disc += cs;
  }
  uint32_t* dists = reinterpret_cast<uint32_t*>(o.list + 2 * a.total);
  uint64_t* heads = o.list + 2 * a.total + a.total / 2;
  uint64_t* wts = heads + a.total / 2 * gb::kInline;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if (!ms[k]) continue;
    const uint32_t len = (uint32_t)(ve[k] - vs[k]);
    const bool mine = low[k] && len < (uint32_t)gb::kBig;
    acc.deg += wave_sum_u32(mine ? len : 0u);
    const uint32_t p = at + lanes_below(ms[k]);
    if (mine && p < a.seg_cap) {
      const int64_t i = gb::entry_at(o.rank, p, o.wgs);
      put_coherent(o.list + i, (uint64_t)y[k] | (uint64_t)len << 32);
      put_coherent(dists + i, nb[k]);
      if (len <= (uint32_t)gb::kInline) {
        put_coherent(heads + 2 * i, (uint64_t)id[k][0] | (uint64_t)id[k][1] << 32);
        put_coherent(heads + 2 * i + 1, (uint64_t)id[k][2] | (uint64_t)id[k][3] << 32);
        put_coherent(wts + 2 * i, (uint64_t)wt[k][0] | (uint64_t)wt[k][1] << 32);
        put_coherent(wts + 2 * i + 1, (uint64_t)wt[k][2] | (uint64_t)wt[k][3] << 32);
      } else {
        put_coherent(o.list + a.total + i, (uint64_t)vs[k]);
      }
    } else if (mine) { /* no room: the burst ends with this round */
      atomic_or(&a.dirty[y[k] >> 6], 1ull << (y[k] & 63));
    }
    at += (uint32_t)__popcll(ms[k]);
  }
  if (!any_pieces) return;
  uint32_t np = 0, npc[K];
  unsigned long long deg = 0;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int64_t len = ve[k] - vs[k];
    npc[k] = (low[k] && len >= gb::kBig) ? (uint32_t)((len + gb::kPiece - 1) / gb::kPiece) : 0u;
    np += npc[k];
    if (npc[k]) deg += (unsigned long long)len;
    acc.disc += (uint32_t)__popcll(ballot(npc[k] != 0));
  }
  const uint32_t ip = wave_inclusive_scan(np);
  const uint32_t tp = wave_lane(ip, 63);
  unsigned long long bp = 0;
  if (lane_id() == 63) bp = atomic_add(&o.sums->npieces, (unsigned long long)tp);
  bp = wave_lane((uint64_t)bp, 63) + (ip - np);
  acc.deg += wave_sum_u64(deg);
  acc.npieces = tp > gb::kPiecesClamp || acc.npieces + tp > gb::kPiecesClamp ? gb::kPiecesClamp : acc.npieces + tp;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int64_t len = ve[k] - vs[k];
    for (uint32_t c = 0; c < npc[k]; ++c, ++bp) {
      const int64_t from = (int64_t)c * gb::kPiece;
      const int64_t l = len - from < gb::kPiece ? len - from : gb::kPiece;
      if ((int64_t)bp < a.cap_pieces) store_entry_coherent(o.pieces + bp, QEntry{vs[k] + from, (int32_t)y[k], (int32_t)l});
      else atomic_or(&a.dirty[y[k] >> 6], 1ull << (y[k] & 63));
    }
  }
}

/* 64 lists of a wave laid end to end (merge path), four arcs per lane per
 * round; du: the distance of each lane's list */
template<typename OffT, typename W>
__device__ __forceinline__ void sssp_grid_merge(const SsspGrid<OffT, W>& a, int64_t start, uint32_t len, uint32_t du,
                                                const SsspGridOut<OffT, W>& o, gb::Acc& acc) {
  const int lane = lane_id();
  const uint32_t incl = wave_inclusive_scan(len);
  const uint32_t total = wave_lane(incl, 63);
  const uint32_t excl = incl - len;
  for (uint32_t t0 = 0; t0 < total; t0 += 4 * 64) {
    uint32_t y[4], nb[4];
    bool ok[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t t = t0 + 64 * k + lane;
      const int owner = scan_owner(incl, t);
      const uint32_t before = __shfl(excl, owner, 64);
      const int64_t j = shfl_i64(start, owner) + (t - before);
      const uint32_t d = __shfl(du, owner, 64);
      ok[k] = t < total;
      y[k] = ok[k] ? (uint32_t)a.cols[j] : 0u;
      nb[k] = ok[k] ? DistOps<W>::bits(DistOps<W>::value(d) + a.w[j]) : 0u;
    }
    sssp_grid_relax<4>(a, y, nb, ok, o, acc);
  }
}

/* pieces of long lists, a wave per entry */
template<typename OffT, typename W>
__device__ __forceinline__ void sssp_grid_pieces(const SsspGrid<OffT, W>& a, const QEntry* ents, int64_t cnt,
                                                 const SsspGridOut<OffT, W>& o, gb::Acc& acc, uint32_t gwave,
                                                 uint32_t nwaves, bool coherent) {
  const int lane = lane_id();
  for (int64_t i = gwave; i < cnt; i += nwaves) {
    const QEntry qe = coherent ? load_entry_coherent(ents + i) : ents[i];
    const W du = DistOps<W>::value(atomic_load(&a.dist[qe.v]));
    for (int64_t o0 = 0; o0 < qe.len; o0 += 4 * 64) {
      uint32_t y[4], nb[4];
      bool ok[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int64_t j = o0 + 64 * k + lane;
        ok[k] = j < qe.len;
        y[k] = ok[k] ? (uint32_t)a.cols[qe.start + j] : 0u;
        nb[k] = ok[k] ? DistOps<W>::bits(du + a.w[qe.start + j]) : 0u;
      }
      sssp_grid_relax<4>(a, y, nb, ok, o, acc);
    }
  }
}

template<typename OffT, typename W>
__global__ void __launch_bounds__(gb::kThreads) sssp_grid_kernel(SsspGrid<OffT, W> a, SsspCtl* ctl, int32_t iter) {
  __shared__ uint32_t s_n[gb::kMaxWgs], s_most;
  __shared__ gb::Local s_local;
  __shared__ int32_t s_next; /* 0: another round, 1: none, 2: a wait ran out, 3: a far pass */
  __shared__ int64_t s_pieces;
  __shared__ uint32_t s_far_n[2], s_far_top, s_T; /* far entries; complement of the smallest kept one's bits */
  if (blockIdx.x % a.stride) return;
  const QueueHdr h0 = *a.hdr;
  /* the same for every workgroup */
  if (ctl->done || !ctl->relax || ctl->pull || (int64_t)h0.deg > a.grid_arcs) return;
  /* a source of so many arcs that the next round, at the mean of arcs per
   * vertex, is far beyond the burst's: sorting it into the far lists and out
   * of them again is for nothing (a clique of 1,800: 445 us, without 390) */
  if (ctl->rounds == 1 && (int64_t)h0.deg * a.mean > 2 * a.grid_arcs) return;
  const uint32_t rank = blockIdx.x / a.stride, wgs = gridDim.x / a.stride;
  const int lane = lane_id(), wv = threadIdx.x >> 6;
  const uint32_t gwave = (uint32_t)wv * wgs + rank, nwaves = wgs * gb::kWaves; /* across the workgroups first */
  const bool lead = rank == 0 && threadIdx.x == 0;
  /* arcs and entries of the round; arcs of the rounds before it (first wave) */
  unsigned long long arcs = h0.deg, entries = h0.nvert, relaxed = 0;
  int32_t rounds = 0;
  const int32_t first_round = ctl->rounds - 1; /* counted by the selection */
  const bool piles = a.weight_sum != nullptr;
  const double first_step = piles ? 4.0 * auto_delta<W>(*a.weight_sum / (double)a.m) : 0.0;
  double step = first_step;                           /* first wave, like what follows */
  unsigned long long bucket_arcs = 0, bucket_rounds = 0;
  bool far_pass = piles; /* every thread's; the first sorts the queues into the far lists (T = 0) */
  int fp = 0;            /* the far list in use */
  if (threadIdx.x == 0) {
    s_local = gb::Local{0, 0, 0, 0, 0};
    s_far_n[0] = s_far_n[1] = s_far_top = 0;
    s_T = piles ? 0u : 0xFFFFFFFFu;
  }
  __syncthreads();
  for (int it = 0;; ++it) {
    const int cur = it & 1;
    if (lead) /* the copy of the round after next: its pieces were last counted two rounds ago */
      atomic_store(&a.x.sums[(it + 1) % 3].npieces, 0ull);
    gb::Acc acc{0, 0, 0, 0};
    const SsspGridOut<OffT, W> o{a.list[cur ^ 1], rank, wgs, a.pieces[cur ^ 1], a.x.sums + (it % 3), &s_local,
                                   a.far[far_pass ? fp ^ 1 : fp] + (int64_t)rank * a.far_cap,
                                   &s_far_n[far_pass ? fp ^ 1 : fp], s_T};
    uint32_t far_top = 0;
    if (it == 0 && piles) {
      for (int q = 0; q < 3; ++q)
        for (int64_t base = (int64_t)gwave * 64; base < h0.count[q]; base += (int64_t)nwaves * 64) {
          QEntry qe{0, 0, 0};
          uint32_t d = 0;
          bool is_far = base + lane < h0.count[q];
          if (is_far) {
            qe = a.q[q][base + lane];
            is_far = q < 2 || qe.start == (int64_t)a.off[qe.v]; /* a long list's first chunk stands for it */
            d = atomic_load(&a.dist[qe.v]);
          }
          sssp_far_append(a, o, is_far, (uint32_t)qe.v, d);
          if (is_far) far_top = ~d > far_top ? ~d : far_top;
        }
    } else if (far_pass) {
      const uint64_t* mine = a.far[fp] + (int64_t)rank * a.far_cap;
      const uint32_t cnt = s_far_n[fp] < a.far_cap ? s_far_n[fp] : a.far_cap;
      for (uint32_t base = (uint32_t)wv * 64; base < cnt; base += gb::kThreads) {
        uint32_t y[1] = {0}, nb[1] = {0}, id[1][gb::kInline], wt[1][gb::kInline];
        int64_t vs[1] = {0}, ve[1] = {0};
        bool low[1] = {base + lane < cnt};
        bool is_far = false;
        if (low[0]) {
          const uint64_t e = mine[base + lane];
          y[0] = (uint32_t)e;
          nb[0] = (uint32_t)(e >> 32);
          const uint32_t d = atomic_load(&a.dist[y[0]]);
          list_bounds(a.off, y[0], vs[0], ve[0]);
          is_far = d == nb[0] && nb[0] >= o.T; /* otherwise lowered since: it has another entry */
          low[0] = d == nb[0] && !is_far;
        }
        if (low[0] && ve[0] - vs[0] <= gb::kInline) {
          load_ids4(a.cols, vs[0], a.m, id[0]);
          load_ids4(reinterpret_cast<const int32_t*>(a.w), vs[0], a.m, wt[0]);
        }
        sssp_far_append(a, o, is_far, y[0], nb[0]);
        if (is_far) far_top = ~nb[0] > far_top ? ~nb[0] : far_top;
        sssp_grid_append<1>(a, o, y, nb, low, vs, ve, id, wt, acc);
      }
    } else if (it == 0) {
      for (int64_t base = (int64_t)gwave * 64; base < h0.count[0]; base += (int64_t)nwaves * 64) {
        QEntry qe{0, 0, 0};
        uint32_t du = 0;
        if (base + lane < h0.count[0]) {
          qe = a.q[0][base + lane];
          du = atomic_load(&a.dist[qe.v]);
        }
        sssp_grid_merge(a, qe.start, (uint32_t)qe.len, du, o, acc);
      }
      sssp_grid_pieces(a, a.q[1], h0.count[1], o, acc, gwave, nwaves, false);
      sssp_grid_pieces(a, a.q[2], h0.count[2], o, acc, gwave, nwaves, false);
    } else {
      const uint64_t* in = a.list[cur];
      const uint32_t* dists = reinterpret_cast<const uint32_t*>(in + 2 * a.total);
      const uint32_t* heads = reinterpret_cast<const uint32_t*>(in + 2 * a.total + a.total / 2);
      const uint32_t* wts = heads + a.total * gb::kInline;
      const uint32_t most = s_most;
      for (uint32_t k = wv; k * gb::kGroup < most; k += gb::kWaves) {
        const uint32_t w = gb::segment_of(k, rank, wgs);
        if (k * gb::kGroup >= s_n[w]) continue;
        const uint32_t i = k * gb::kGroup + (uint32_t)lane / gb::kInline;
        const int64_t e = gb::entry_at(w, i, wgs);
        const uint32_t sub = (uint32_t)lane % gb::kInline;
        const bool has = i < s_n[w];
        uint64_t e0 = 0;
        uint32_t du = 0, wt = 0, y[1] = {0};
        if (has) {
          e0 = atomic_load(in + e);
          du = atomic_load(dists + e);
          y[0] = atomic_load(heads + gb::kInline * e + sub);
          wt = atomic_load(wts + gb::kInline * e + sub);
        }
        const uint32_t len = (uint32_t)(e0 >> 32);
        if (ballot(len > (uint32_t)gb::kInline)) {
          int64_t start = 0; /* the entry's first lane lays its list */
          if (has && sub == 0)
            start = len > (uint32_t)gb::kInline ? (int64_t)atomic_load(in + a.total + e) : (int64_t)a.off[(uint32_t)e0];
          sssp_grid_merge(a, start, sub == 0 ? len : 0u, du, o, acc);
        } else {
          const bool ok[1] = {sub < len};
          const uint32_t nb[1] = {DistOps<W>::bits(DistOps<W>::value(du) + DistOps<W>::value(wt))};
          sssp_grid_relax<1>(a, y, nb, ok, o, acc);
        }
      }
      sssp_grid_pieces(a, a.pieces[cur], s_pieces, o, acc, gwave, nwaves, true);
    }
    gb::add_local(&s_local, acc);
    if (far_pass) {
      far_top = wave_max_u32(far_top);
      if (lane == 0 && far_top) atomicMax(&s_far_top, far_top);
    }
    wait_stores_complete(); /* the lists: no fences, they are written and read coherently */
    __syncthreads();
    if (wv == 0) {
      gb::Totals t{};
      int32_t next = 2;
      /* whether anything is far, and after a far pass the smallest of it */
      const uint32_t kept = s_far_n[far_pass ? fp ^ 1 : fp];
      const unsigned long long extra = !kept ? 0ull : far_pass ? 1ull << 32 | s_far_top : 1ull;
      if (gb::exchange(a.x, &s_local, it, rank, wgs, s_n, t, extra)) {
        if (!far_pass) {
          if (lead) record_round(a.rounds, first_round + rounds, entries, arcs);
          relaxed += arcs;
          bucket_arcs += arcs;
          ++bucket_rounds;
          ++rounds;
        }
        arcs = t.deg;
        entries = t.disc;
        const bool fits = (int64_t)t.deg <= a.grid_arcs && t.most <= a.seg_cap && (int64_t)t.npieces <= a.cap_pieces;
        next = t.disc > 0 ? (fits ? 0 : 1) : t.mx ? 3 : 1;
        if (next == 3) { /* the bucket is done: on by a step, or where that found nothing from the smallest left */
          if (bucket_rounds) {
            if (bucket_arcs < (unsigned long long)kNearFew * bucket_rounds) step *= 2.0;
            else if (bucket_arcs > (unsigned long long)kNearMany * bucket_rounds && step > first_step / 64) step *= 0.5;
          }
          bucket_arcs = bucket_rounds = 0;
          uint32_t from = far_pass ? ~(uint32_t)t.mx : s_T;
          /* the first bucket counts from the source, wherever the burst starts */
          if (it == 0 && (double)DistOps<W>::value(from) < step) from = 0;
          const uint32_t T = next_threshold<W>(from, step, a.w_max);
          if (lane == 0) s_T = T;
        }
      }
      if (lane == 0) {
        s_next = next;
        s_most = t.most;
        s_pieces = (int64_t)(t.npieces < (unsigned long long)a.cap_pieces ? t.npieces : (unsigned long long)a.cap_pieces);
        if (far_pass) {
          s_far_n[fp] = 0; /* read; the next far pass fills it */
          s_far_top = 0;
        }
      }
    }
    __syncthreads();
    if (far_pass) fp ^= 1;
    far_pass = s_next == 3;
    if (s_next == 0 || s_next == 3) continue;
    if (s_next == 1) { /* what the last round lowered goes back to the dirty bitmap */
      const uint64_t* left = a.list[cur ^ 1];
      const uint32_t mine = s_n[rank] < a.seg_cap ? s_n[rank] : a.seg_cap;
      for (uint32_t i = threadIdx.x; i < mine; i += gb::kThreads) {
        const uint32_t v = (uint32_t)atomic_load(left + gb::entry_at(rank, i, wgs));
        atomic_or(&a.dirty[v >> 6], 1ull << (v & 63));
      }
      const uint64_t* far = a.far[fp] + (int64_t)rank * a.far_cap;
      const uint32_t nf = piles ? (s_far_n[fp] < a.far_cap ? s_far_n[fp] : a.far_cap) : 0u;
      for (uint32_t i = threadIdx.x; i < nf; i += gb::kThreads) {
        const uint32_t v = (uint32_t)far[i];
        atomic_or(&a.dirty[v >> 6], 1ull << (v & 63));
      }
      for (int64_t i = (int64_t)rank * gb::kThreads + threadIdx.x; i < s_pieces; i += (int64_t)wgs * gb::kThreads) {
        const uint32_t v = (uint32_t)load_entry_coherent(a.pieces[cur ^ 1] + i).v;
        atomic_or(&a.dirty[v >> 6], 1ull << (v & 63));
      }
    }
    break;
  }
  if (s_next == 2) { /* a wait ran out: the next iteration's record says so */
    if (threadIdx.x == 0) {
      ctl->done = 1;
      RoundLog e{};
      e.iter = -1;
      e.done = 1;
      e.fail = 1;
      RoundLog* slot = &a.log[(iter + 1) % kRing];
      *slot = e;
      __threadfence_system();
      __hip_atomic_store(&slot->iter, iter + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __threadfence_system();
    }
    return;
  }
  if (!lead) return;
  /* the selection counted one round (none, where the first does not fit the
   * lists); the relax launch has nothing left */
  ctl->rounds += rounds - 1;
  ctl->relaxed += relaxed - h0.deg;
  ctl->relax = 0;
  atomic_add(&a.relax_slots[0], relaxed);
}

/* Where a selection launch keeps its scratch and writes its decision. */
struct SelectArgs {
  uint64_t *dirty, *near_bm, *settled, *settled_all;
  const uint32_t* dist;
  SplitSlot* slots;
  int64_t w0, nblocks; /* bitmap words; count-pass workgroups (sums to scan) */
  uint32_t* arrive;    /* kArriveWords zeroed words */
  RoundLog* log;
  const unsigned long long* heavy_total;
  double delta, w_max;
  int32_t pull_mode;
  int32_t bellman;    /* the reference's schedule (no buckets) */
  int64_t burst_arcs; /* rounds of the reference's schedule with at most this many arcs run as a burst (0: never) */
};

/* One iteration's selection, count and decision in one launch.  Each
 * workgroup splits the 256 words of the dirty bitmap that its four count
 * tiles cover (thread t splits the word that it then counts, so no other
 * workgroup's near bits are needed), counts the near set's queue entries,
 * and the last workgroup to finish scans the counts and decides: relax /
 * advance the threshold / stop, and the iteration's record into the pinned
 * ring.  A heavy iteration pulls (pull_mode 1), pushes (-1), or (0) pulls
 * when the heavy arcs of the vertices not yet settled -- all heavy arcs less
 * those of every settled set so far, in-arcs being out-arcs on an undirected
 * graph -- are fewer than those of the bucket's settled set.  The far
 * statistics are added into `slots` with atomics; the last workgroup reads
 * them through agent-coherent loads and clears them for the next
 * iteration. */
template<typename OffT, typename W>
__global__ void __launch_bounds__(kBlock) sssp_select_kernel(CompactArgs<OffT> ca, SelectArgs sa, SsspCtl* ctl,
                                                             int32_t iter) {
  __shared__ QueueHdr tot;
  if (ctl->done) return;
  const bool heavy_next = ctl->heavy_next != 0;
  split_word<W>((int64_t)blockIdx.x * kBlock + threadIdx.x, sa.w0, heavy_next, sa.bellman != 0, ctl->T_bits,
                sa.dirty, sa.near_bm, sa.settled, sa.settled_all, sa.dist, sa.slots);
  compact_count_body<OffT, kFromBitmap>(ca, heavy_next ? 1 : 0);
  if (!last_to_arrive<true>(sa.arrive, false)) return;
  compact_scan_body_t<kBlock, 8, true>(ca.blocks, sa.nblocks, ca.hdr, &tot);
  __syncthreads();
  if (threadIdx.x != 0) return;
  RoundLog e{};
  e.iter = iter;
  e.near_v = (int64_t)tot.nvert;
  e.near_e = (int64_t)tot.deg;
  ctl->pull = 0;
  ctl->burst = 0;
  if (heavy_next) { /* this iteration relaxes the heavy arcs of the settled set */
    ctl->heavy_next = 0;
    ctl->r_pending = 0;
    ctl->heavy = 1;
    ctl->relax = tot.nvert > 0 ? 1 : 0;
    const unsigned long long done_arcs = ctl->heavy_done + tot.deg;
    ctl->heavy_done = done_arcs;
    if (tot.nvert > 0) {
      const unsigned long long ht = *sa.heavy_total;
      const unsigned long long pull_arcs = ht > done_arcs ? ht - done_arcs : 0ull;
      const bool pull = sa.pull_mode > 0 || (sa.pull_mode == 0 && pull_arcs < tot.deg);
      ctl->pull = pull ? 1 : 0;
      ctl->rounds += 1;
      ctl->relaxed += pull ? pull_arcs : tot.deg;
    }
  } else if (tot.nvert > 0) {
    ctl->heavy = 0;
    ctl->relax = 1;
    ctl->r_pending = 1;
    ctl->rounds += 1;
    ctl->relaxed += tot.deg;
    ctl->burst = (sa.bellman && (int64_t)tot.deg <= sa.burst_arcs) ? 1 : 0;
  } else {
    ctl->heavy = 0;
    ctl->relax = 0;
    if (ctl->r_pending && sa.delta > 0.0) {
      ctl->heavy_next = 1; /* the bucket's light phase is over */
    } else {
      unsigned long long far = 0;
      uint32_t fmin = 0xFFFFFFFFu;
      for (int k = 0; k < kSlots; ++k) {
        far += __hip_atomic_load(&sa.slots[k].far_count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t mk = __hip_atomic_load(&sa.slots[k].far_min, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        fmin = mk < fmin ? mk : fmin;
      }
      if (far == 0) ctl->done = 1;
      else ctl->T_bits = next_threshold<W>(fmin, sa.delta, sa.w_max);
      ctl->r_pending = 0;
    }
  }
  for (int k = 0; k < kSlots; ++k) { /* the next iteration's split adds into cleared slots */
    sa.slots[k].far_count = 0;
    sa.slots[k].far_min = 0xFFFFFFFFu;
  }
  e.done = ctl->done;
  e.relax = ctl->relax;
  e.rounds = ctl->rounds;
  e.relaxed = ctl->relaxed;
  /* every field, then (after a system-scope fence) the iteration number the
   * host polls for */
  RoundLog* slot = &sa.log[iter % kRing];
  e.iter = -1;
  *slot = e;
  __threadfence_system();
  __hip_atomic_store(&slot->iter, iter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __threadfence_system();
}

template<typename OffT>
__global__ void sssp_init_kernel(const OffT* off, uint32_t* dist, uint32_t unreached, int64_t n, int32_t src,
                                 QEntry* q0, QEntry* q1, QEntry* q2, QueueHdr* hdr, Tuning t,
                                 unsigned long long* rounds) {
  const int64_t tid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = tid; i < n; i += stride) dist[i] = i == src ? 0u : unreached;
  for (int64_t i = tid; rounds && i < 2 * SG_MAX_LEVELS_RECORDED; i += stride) rounds[i] = 0ull;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    QEntry* const q[3] = {q0, q1, q2};
    enqueue_single(off, t, q, hdr, src);
  }
}

__global__ void set_bit_kernel(uint64_t* bm, int32_t v) { bm[v >> 6] |= 1ull << (v & 63); }

template<typename W>
__global__ void weight_sum_kernel(const W* w, int64_t m, double* out) {
  double acc = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x)
    acc += (double)w[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  if (lane_id() == 0) atomicAdd(out, acc);
}

template<typename OffT>
__global__ void reached_kernel(const OffT* off, const uint32_t* dist, uint32_t unreached, int64_t n,
                               unsigned long long* out) {
  uint64_t e = 0, c = 0;
  for (int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; v < n; v += (int64_t)gridDim.x * blockDim.x)
    if (dist[v] != unreached) {
      e += (uint64_t)(off[v + 1] - off[v]);
      ++c;
    }
  /* one atomic pair per workgroup (not per wave) */
  __shared__ unsigned long long red[2][4];
  e = wave_sum_u64(e);
  c = wave_sum_u64(c);
  if (lane_id() == 0) {
    red[0][threadIdx.x >> 6] = e;
    red[1][threadIdx.x >> 6] = c;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long te = 0, tc = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
      te += red[0][w];
      tc += red[1][w];
    }
    atomicAdd(&out[0], te);
    atomicAdd(&out[1], tc);
  }
}

struct SsspWorkspace {
  /* dirty vertices, near set of the round, bucket's settled set, every vertex settled so far */
  uint64_t* bm[4] = {nullptr, nullptr, nullptr, nullptr};
  unsigned long long* acc = nullptr;
  SplitSlot* slots = nullptr;
  SsspCtl* ctl = nullptr;
  unsigned long long* relax_slots = nullptr; /* kSlots x 16 (one cache line each) */
  unsigned long long* rounds = nullptr;      /* behind them: record_round's, SG_MAX_LEVELS_RECORDED pairs */
  uint32_t* arrive = nullptr; /* arrival counters of the selection and write launches (kArriveWords each), zero
                                 between launches */
  QEntry* burst_list[2] = {nullptr, nullptr}; /* kSsspBurstMax entries each */
  /* grid bursts, allocated on the first run of the reference's schedule */
  void* grid_base = nullptr; /* holds the following */
  gb::Exchange grid_x{};
  uint64_t* grid_list[2] = {nullptr, nullptr};
  QEntry* grid_pieces[2] = {nullptr, nullptr};
  uint64_t* grid_far[2] = {nullptr, nullptr};
  int grid_wgs = 0, grid_stride = 1;
  RoundLog* log = nullptr; /* kRing entries, pinned coherent host memory */
  SmallLog* small_log = nullptr; /* graphs of at most kSmallVerts vertices */
  hipEvent_t ev[kRing] = {};
  hipEvent_t ev_pre[kRing] = {}; /* before each iteration's relax launch (record_relax) */
  QueueSet qs;
  int64_t w0 = 0;
};

void sssp_ws_free(SsspWorkspace* w) {
  if (!w) return;
  (void)hipFree(w->bm[0]);
  (void)hipFree(w->bm[1]);
  (void)hipFree(w->bm[2]);
  (void)hipFree(w->bm[3]);
  (void)hipFree(w->acc);
  (void)hipFree(w->slots);
  (void)hipFree(w->ctl);
  (void)hipFree(w->relax_slots);
  (void)hipFree(w->arrive);
  (void)hipFree(w->burst_list[0]);
  (void)hipFree(w->burst_list[1]);
  (void)hipFree(w->grid_base);
  if (w->log) (void)hipHostFree(w->log);
  if (w->small_log) (void)hipHostFree(w->small_log);
  for (hipEvent_t e : w->ev)
    if (e) (void)hipEventDestroy(e);
  for (hipEvent_t e : w->ev_pre)
    if (e) (void)hipEventDestroy(e);
  w->qs.release();
  delete w;
}


int sssp_workspace_for(sg_graph_t g, SsspWorkspace** out) {
  auto* ws = static_cast<SsspWorkspace*>(g->sssp_ws);
  if (!ws) {
    sg_device_t dev = g->dev;
    const int64_t n = g->n;
    ws = new SsspWorkspace();
    ws->w0 = (n + 63) / 64;
    int st = SG_OK;
    if ((st = sg::alloc_device(dev, (void**)&ws->bm[0], 8 * (ws->w0 + 1))) ||
        (st = sg::alloc_device(dev, (void**)&ws->bm[1], 8 * (ws->w0 + 1))) ||
        (st = sg::alloc_device(dev, (void**)&ws->bm[2], 8 * (ws->w0 + 1))) ||
        (st = sg::alloc_device(dev, (void**)&ws->bm[3], 8 * (ws->w0 + 1))) ||
        (st = sg::alloc_device(dev, (void**)&ws->acc, 16)) ||
        (st = sg::alloc_device(dev, (void**)&ws->slots, sizeof(SplitSlot) * kSlots)) ||
        (st = sg::alloc_device(dev, (void**)&ws->ctl, sizeof(SsspCtl))) ||
        (st = sg::alloc_device(dev, (void**)&ws->relax_slots, 8 * 16 * kSlots + 16 * SG_MAX_LEVELS_RECORDED)) ||
        (st = sg::alloc_device(dev, (void**)&ws->arrive, 8 * kArriveWords)) ||
        (st = sg::zero_async(dev, ws->arrive, 8 * kArriveWords)) ||
        (st = sg::alloc_device(dev, (void**)&ws->burst_list[0], sizeof(QEntry) * kSsspBurstMax)) ||
        (st = sg::alloc_device(dev, (void**)&ws->burst_list[1], sizeof(QEntry) * kSsspBurstMax)) ||
        (st = ws->qs.init(dev, n, g->m, default_tuning()))) {
      sssp_ws_free(ws);
      return st;
    }
    ws->rounds = ws->relax_slots + 16 * kSlots;
    bool ok = hipHostMalloc((void**)&ws->log, sizeof(RoundLog) * kRing, hipHostMallocCoherent) == hipSuccess;
    if (ok && n <= kSmallVerts && g->m <= kSmallArcs)
      ok = hipHostMalloc((void**)&ws->small_log, sizeof(SmallLog), hipHostMallocCoherent) == hipSuccess;
    for (int r = 0; r < kRing && ok; ++r)
      ok = hipEventCreate(&ws->ev[r]) == hipSuccess && hipEventCreate(&ws->ev_pre[r]) == hipSuccess;
    if (!ok) {
      sssp_ws_free(ws);
      sg::set_error("sssp workspace: event or pinned log allocation failed");
      return SG_ERR_HIP;
    }
    g->sssp_ws = ws;
  }
  *out = ws;
  return SG_OK;
}

int sssp_grid_buffers(sg_graph_t g, SsspWorkspace* ws, int occ) {
  if (ws->grid_wgs > 0) return SG_OK;
  sg_device_t dev = g->dev;
  const gb::Plan p = gb::plan(dev, occ, kSsspGridWgs);
  const int64_t total = gb::seg_cap(kSsspGridArcs, p.wgs) * p.wgs;
  const size_t list = sizeof(uint64_t) * (size_t)kSsspGridWords(total);
  const size_t pieces = sizeof(QEntry) * (size_t)gb::cap_pieces(kSsspGridArcs);
  const size_t far = sizeof(uint64_t) * (size_t)far_capacity(g->n, p.wgs) * p.wgs;
  SG_TRY(gb::alloc_parts(dev, &ws->grid_base,
                         {{(void**)&ws->grid_x.sums, gb::kSumsBytes},
                          {(void**)&ws->grid_x.slots, gb::kSlotsBytes},
                          {(void**)&ws->grid_x.wide, gb::kWideBytes},
                          {(void**)&ws->grid_x.stop, gb::kStopBytes},
                          {(void**)&ws->grid_list[0], list},
                          {(void**)&ws->grid_list[1], list},
                          {(void**)&ws->grid_pieces[0], pieces},
                          {(void**)&ws->grid_pieces[1], pieces},
                          {(void**)&ws->grid_far[0], far},
                          {(void**)&ws->grid_far[1], far}}));
  ws->grid_stride = p.stride;
  ws->grid_wgs = p.wgs;
  return SG_OK;
}

/* The light-first adjacency for bucket width dlt, built on first use and
 * kept with the graph until a run asks for another width. */
template<typename OffT, typename W>
int ensure_split(sg_graph_t g, W dlt) {
  const uint32_t bits = DistOps<W>::bits(dlt);
  if (g->sssp_split_valid && g->sssp_split_bits == bits) return SG_OK;
  sg_device_t dev = g->dev;
  if (!g->sssp_cols) {
    SG_TRY(sg::alloc_device(dev, (void**)&g->sssp_cols, 4 * (size_t)(g->m + 1)));
    SG_TRY(sg::alloc_device(dev, (void**)&g->sssp_w, 4 * (size_t)(g->m + 1)));
    SG_TRY(sg::alloc_device(dev, (void**)&g->sssp_light, 4 * (size_t)(g->n + 1)));
  }
  unsigned long long* heavy_total = nullptr; /* heavy arcs of the split, read by the heavy rounds' decision */
  SG_TRY(sg::graph_buffer(g, "sssp_heavy_total", 8, &heavy_total));
  SG_TRY(sg::zero_async(dev, heavy_total, 8));
  split_build_kernel<OffT, W><<<dev->cus * 8, kBlock, 0, dev->stream>>>(
      (const OffT*)g->offsets, g->cols, (const W*)g->weights, g->n, dlt, g->sssp_cols, (W*)g->sssp_w,
      g->sssp_light, heavy_total);
  SG_HIP(hipGetLastError());
  g->sssp_split_bits = bits;
  g->sssp_split_valid = true;
  return SG_OK;
}

/* The sum of the arcs' weights in device memory, summed once per graph; no
 * wait (a host wait for it made a first call on a small graph 2 % longer). */
template<typename W>
int weight_sum(sg_graph_t g, const double** out) {
  double* sum = nullptr;
  SG_TRY(sg::graph_buffer(g, "sssp_weight_sum", 8, &sum));
  if (!g->weight_sum_valid) {
    SG_TRY(sg::zero_async(g->dev, sum, 8));
    weight_sum_kernel<W><<<sg::grid_for(g->dev, g->m, 256, 4), 256, 0, g->dev->stream>>>((const W*)g->weights, g->m, sum);
    SG_HIP(hipGetLastError());
    g->weight_sum_valid = true;
  }
  *out = sum;
  return SG_OK;
}

template<typename OffT, typename W>
int run_sssp(sg_graph_t g, int32_t src, double delta, bool far_lists, int32_t heavy_pull, int64_t burst_arcs,
             bool record_relax, W* dist_out, sg_sssp_stats* stats) {
  sg_device_t dev = g->dev;
  hipStream_t s = dev->stream;
  const int64_t n = g->n;
  const Tuning tune = default_tuning();
  SsspWorkspace* ws = nullptr;
  SG_TRY(sssp_workspace_for(g, &ws));
  QueueSet& Q = ws->qs;
  const OffT* off = (const OffT*)g->offsets;
  uint32_t* dist = reinterpret_cast<uint32_t*>(dist_out);
  const uint32_t unreached = DistOps<W>::bits((W)(n + 1));
  const int grid_main = dev->cus * 8;

  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (stats) {
    SG_HIP(hipEventCreate(&e0));
    SG_HIP(hipEventCreate(&e1));
    SG_HIP(hipEventRecord(e0, s));
  }
  uint64_t* dirty = ws->bm[0];
  uint64_t* near_bm = ws->bm[1];
  uint64_t* settled = ws->bm[2];
  uint64_t* settled_all = ws->bm[3];
  SG_TRY(sg::zero_async(dev, dirty, 8 * ws->w0));
  SG_TRY(sg::zero_async(dev, settled, 8 * ws->w0));
  /* vertices without arcs never change: a pull skips them from the start */
  const bool directed = (g->flags & SG_GRAPH_DIRECTED) != 0;
  if (!directed) {
    SG_TRY(sg::graph_ensure_isolated(g));
    SG_HIP(hipMemcpyAsync(settled_all, g->isolated, 8 * ws->w0, hipMemcpyDeviceToDevice, s));
  } else {
    SG_TRY(sg::zero_async(dev, settled_all, 8 * ws->w0));
  }
  SG_TRY(sg::zero_async(dev, ws->relax_slots, 8 * 16 * kSlots));
  const bool bellman = !(delta > 0.0) || !std::isfinite(delta);
  unsigned long long* rounds_log = stats && bellman && burst_arcs > 0 ? ws->rounds : nullptr; /* bursts may run */
  sssp_init_kernel<OffT><<<sg::grid_for(dev, n, 256, 4), 256, 0, s>>>(off, dist, unreached, n, src, Q.q[0][0],
                                                                       Q.q[0][1], Q.q[0][2], Q.hdr, tune, rounds_log);
  set_bit_kernel<<<1, 1, 0, s>>>(dirty, src);
  SG_HIP(hipGetLastError());
  const double w_max = DistOps<W>::is_float ? 3.0e38 : 4294967295.0;
  {
    SsspCtl c{};
    c.T_bits = DistOps<W>::bits((W)(bellman ? w_max : std::min(delta, w_max)));
    SG_HIP(hipMemcpyAsync(ws->ctl, &c, sizeof(c), hipMemcpyHostToDevice, s));
  }
  /* arcs of weight >= dlt are heavy (none under the reference's schedule) */
  const W dlt = bellman ? (W)w_max : (W)std::min(std::max(delta, DistOps<W>::is_float ? 0.0 : 1.0), w_max);
  /* bucketed runs read the light-first adjacency, the entries covering one
   * phase's part of each list */
  if (!bellman) SG_TRY((ensure_split<OffT, W>(g, dlt)));
  CompactArgs<OffT> ca = make_compact_args<OffT>(Q, 0, off, nullptr, nullptr, near_bm, tune);
  ca.split = bellman ? nullptr : g->sssp_light;
  SsspArgs<OffT, W> a{};
  a.cols = bellman ? g->cols : g->sssp_cols;
  a.w = bellman ? (const W*)g->weights : (const W*)g->sssp_w;
  a.dist = dist;
  a.next_bm = dirty;
  a.w0 = ws->w0;
  for (int k = 0; k < 3; ++k) a.qin[k] = Q.q[0][k];
  a.qin_hdr = Q.hdr;
  a.off = off;
  a.light = g->sssp_light;
  a.settled = settled_all;
  a.frontier = near_bm;
  a.n = n;
  /* a heavy round pulls only on an undirected graph (in-arcs = out-arcs, symmetric weights) */
  const int32_t pull_mode = directed ? -1 : heavy_pull;
  unsigned long long* heavy_total = nullptr;
  if (!bellman) SG_TRY(sg::graph_buffer(g, "sssp_heavy_total", 8, &heavy_total));
  SelectArgs sa{};
  sa.dirty = dirty;
  sa.near_bm = near_bm;
  sa.settled = settled;
  sa.settled_all = settled_all;
  sa.dist = dist;
  sa.slots = ws->slots;
  sa.w0 = ws->w0;
  sa.nblocks = Q.nblocks;
  sa.arrive = ws->arrive;
  sa.log = ws->log;
  sa.heavy_total = heavy_total;
  sa.delta = bellman ? 0.0 : delta;
  sa.w_max = w_max;
  sa.pull_mode = pull_mode;
  sa.bellman = bellman ? 1 : 0;
  /* the grid bursts' near and far piles take the small rounds from the start;
   * a record of the relax launches leaves the rounds to them */
  const bool grid = bellman && burst_arcs > 0 && !record_relax, piles = grid && far_lists;
  sa.burst_arcs = piles ? kTinyArcs : burst_arcs;
  SsspBurst<OffT, W> sb{};
  sb.off = off;
  sb.cols = g->cols;
  sb.w = (const W*)g->weights;
  sb.dist = dist;
  sb.dirty = dirty;
  for (int k = 0; k < 3; ++k) sb.q[k] = Q.q[0][k];
  sb.hdr = Q.hdr;
  sb.list[0] = ws->burst_list[0];
  sb.list[1] = ws->burst_list[1];
  sb.burst_arcs = sa.burst_arcs;
  sb.hand_over = piles ? 1 : 0;
  sb.out_hdr = Q.hdr;
  sb.tune = tune;
  sb.relax_slots = ws->relax_slots;
  sb.rounds = rounds_log;
  sb.arrive = ws->arrive + kArriveWords;
  split_slots_reset_kernel<<<1, 64, 0, s>>>(ws->slots, ws->ctl); /* later iterations clear them as they decide */
  /* one iteration, three launches: split + near-set count + decision (relax /
   * next bucket / stop); queue write; relax.  Everything the host needs is in
   * the iteration's record. */
  SsspGrid<OffT, W> sg_args{};
  if (grid) {
    static int occ = 0; /* per instantiation */
    if (occ == 0) {
      int nb = 0;
      SG_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, sssp_grid_kernel<OffT, W>, gb::kThreads, 0));
      occ = std::max(1, nb);
    }
    SG_TRY(sssp_grid_buffers(g, ws, occ));
    sg_args.off = off;
    sg_args.cols = g->cols;
    sg_args.w = (const W*)g->weights;
    sg_args.m = g->m;
    sg_args.mean = g->m / n;
    sg_args.dist = dist;
    sg_args.dirty = dirty;
    for (int k = 0; k < 3; ++k) sg_args.q[k] = Q.q[0][k];
    sg_args.hdr = Q.hdr;
    sg_args.seg_cap = (uint32_t)gb::seg_cap(kSsspGridArcs, ws->grid_wgs);
    sg_args.total = (int64_t)sg_args.seg_cap * ws->grid_wgs;
    for (int k = 0; k < 2; ++k) {
      sg_args.list[k] = ws->grid_list[k];
      sg_args.pieces[k] = ws->grid_pieces[k];
      sg_args.far[k] = ws->grid_far[k];
    }
    sg_args.cap_pieces = gb::cap_pieces(kSsspGridArcs);
    sg_args.grid_arcs = kSsspGridArcs;
    if (piles) SG_TRY(weight_sum<W>(g, &sg_args.weight_sum));
    sg_args.far_cap = far_capacity(n, ws->grid_wgs);
    sg_args.w_max = w_max;
    sg_args.x = ws->grid_x;
    sg_args.x.wait_ticks = dev->wait_ticks;
    sg_args.relax_slots = ws->relax_slots;
    sg_args.rounds = rounds_log;
    sg_args.log = ws->log;
    sg_args.stride = (uint32_t)ws->grid_stride;
  }
  auto enqueue = [&](int32_t it, bool burst) -> int {
    sssp_select_kernel<OffT, W><<<Q.grid_tiles(), kBlock, 0, s>>>(ca, sa, ws->ctl, it);
    near_write_kernel<OffT, W><<<Q.grid_tiles(), kBlock, 0, s>>>(ca, sb, ws->ctl);
    if (burst) { /* a grid burst ahead of the relax launch (returns at once unless the round qualifies) */
      gb::reset_kernel<<<1, 256, 0, s>>>(sg_args.x, ws->grid_wgs);
      void* args[] = {&sg_args, &ws->ctl, &it};
      SG_HIP(launch_resident(reinterpret_cast<const void*>(sssp_grid_kernel<OffT, W>), ws->grid_wgs * ws->grid_stride,
                             gb::kThreads, args, s));
    }
    if (record_relax) SG_HIP(hipEventRecord(ws->ev_pre[it % kRing], s));
    relax_kernel<OffT, W><<<grid_main, kBlock, 0, s>>>(a, ws->ctl, ws->relax_slots);
    SG_HIP(hipGetLastError());
    /* untimed iterations record no event (a stream barrier per iteration):
     * the host polls the iteration's record, written by its selection */
    if (record_relax) SG_HIP(hipEventRecord(ws->ev[it % kRing], s));
    return SG_OK;
  };
  for (int k = 0; k < kRing; ++k) __atomic_store_n(&ws->log[k].iter, -1, __ATOMIC_RELEASE);
  SG_TRY(enqueue(0, piles));
  SG_TRY(enqueue(1, false));
  int32_t round = 0;
  /* iterations in a row whose round is small enough for a grid burst; from
   * two on, the iterations enqueued carry one */
  int32_t small_rounds = 0;
  int64_t relaxed = 0;
  float relax_ms = 0.f;
  int32_t relax_launches = 0;
  const int64_t max_iter = 4 * n + 256; /* every iteration relaxes or advances T past a distance */
  for (int32_t it = 0;; ++it) {
    if (record_relax) SG_HIP(hipEventSynchronize(ws->ev[it % kRing]));
    else SG_TRY(sg::wait_host_flag(&ws->log[it % kRing].iter, it, s, "sg_sssp"));
    RoundLog e;
    std::memcpy(&e, (const void*)&ws->log[it % kRing], sizeof(e));
    if (e.iter != it) {
      SG_HIP(hipStreamSynchronize(s));
      sg::set_error("sg_sssp: iteration record %d out of order (found %d)", it, e.iter);
      return SG_ERR_STATE;
    }
    if (e.fail) {
      SG_HIP(hipStreamSynchronize(s));
      sg::set_error("sg_sssp: a grid burst waited longer than the device's wait limit (iteration %d)", it);
      return SG_ERR_HIP;
    }
    if (e.relax && stats && e.rounds - 1 < SG_MAX_LEVELS_RECORDED) {
      stats->round_vertices[e.rounds - 1] = e.near_v;
      stats->round_edges[e.rounds - 1] = e.near_e;
    }
    if (e.relax && record_relax) { /* the relax launch of a relaxing iteration, on its own */
      float ms = 0.f;
      SG_HIP(hipEventElapsedTime(&ms, ws->ev_pre[it % kRing], ws->ev[it % kRing]));
      relax_ms += ms;
      ++relax_launches;
    }
    round = e.rounds;
    relaxed = (int64_t)e.relaxed;
    if (e.done) break;
    if (it + 2 > max_iter) {
      SG_HIP(hipStreamSynchronize(s));
      sg::set_error("sg_sssp: no termination after %lld iterations", (long long)it);
      return SG_ERR_STATE;
    }
    small_rounds = (grid && e.relax && e.near_e <= kSsspGridArcs) ? small_rounds + 1 : 0;
    SG_TRY(enqueue(it + 2, small_rounds >= 2));
  }
  if (stats) {
    SG_HIP(hipEventRecord(e1, s));
    SG_HIP(hipEventSynchronize(e1));
    float ms = 0.f;
    SG_HIP(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    stats->kernel_ms = ms;
    stats->rounds = round;
    stats->relax_ms = relax_ms;
    stats->relax_launches = relax_launches;
    {
      /* the relax counts and, behind them, the bursts' rounds, in one copy */
      const auto* rs = static_cast<const unsigned long long*>(dev->host_scratch);
      const auto* rl = rs + 16 * kSlots;
      const int32_t recorded = rounds_log ? std::min(round, (int32_t)SG_MAX_LEVELS_RECORDED) : 0;
      SG_HIP(hipMemcpyAsync(dev->host_scratch, ws->relax_slots, 8 * 16 * kSlots + 16 * (size_t)recorded,
                            hipMemcpyDeviceToHost, s));
      SG_HIP(hipStreamSynchronize(s));
      for (int32_t r = 0; r < recorded; ++r) {
        if (rl[2 * r] == 0) continue;
        stats->round_vertices[r] = (int64_t)rl[2 * r];
        stats->round_edges[r] = (int64_t)rl[2 * r + 1];
      }
      unsigned long long t = 0;
      for (int k = 0; k < kSlots; ++k) t += rs[k * 16];
      stats->relaxations = (int64_t)t; /* arcs relaxed in their phase (examined: `relaxed`) */
      (void)relaxed;
    }
    SG_TRY(sg::zero_async(dev, ws->acc, 16));
    reached_kernel<OffT><<<sg::grid_for(dev, n, 256, 4), 256, 0, s>>>(off, dist, unreached, n, ws->acc);
    unsigned long long h[2];
    SG_HIP(hipMemcpyAsync(h, ws->acc, 16, hipMemcpyDeviceToHost, s));
    SG_HIP(hipStreamSynchronize(s));
    stats->reached_edges = (int64_t)h[0];
    stats->reached_vertices = (int64_t)h[1];
  }
  SG_HIP(hipStreamSynchronize(s));
  return SG_OK;
}

} // namespace

namespace sg {
void sssp_workspace_release(sg_graph_t g) {
  if (g && g->sssp_ws) {
    sssp_ws_free(static_cast<SsspWorkspace*>(g->sssp_ws));
    g->sssp_ws = nullptr;
  }
}
} // namespace sg

/* A small graph under the automatic schedule: the rounds of the reference's,
 * in one launch. */
template<typename OffT, typename W>
int run_sssp_small(sg_graph_t g, int32_t src, W* dist, sg_sssp_stats* stats) {
  hipStream_t s = g->dev->stream;
  SsspWorkspace* ws = nullptr;
  SG_TRY(sssp_workspace_for(g, &ws));
  SmallArgs<OffT, W> a{};
  a.off = (const OffT*)g->offsets;
  a.cols = g->cols;
  a.w = (const W*)g->weights;
  a.dist = reinterpret_cast<uint32_t*>(dist);
  a.n = (int32_t)g->n;
  a.src = src;
  a.unreached = DistOps<W>::bits((W)(g->n + 1));
  a.max_rounds = (int32_t)(4 * g->n + 256);
  a.log = ws->small_log;
  if (stats) SG_HIP(hipEventRecord(ws->ev[0], s));
  sssp_small_kernel<OffT, W><<<1, kSmallThreads, 0, s>>>(a);
  SG_HIP(hipGetLastError());
  if (stats) SG_HIP(hipEventRecord(ws->ev[1], s));
  SG_HIP(hipStreamSynchronize(s));
  const SmallLog& log = *ws->small_log;
  if (log.fail) {
    sg::set_error("sg_sssp: no termination after %d iterations", log.rounds);
    return SG_ERR_STATE;
  }
  if (!stats) return SG_OK;
  SG_HIP(hipEventElapsedTime(&stats->kernel_ms, ws->ev[0], ws->ev[1]));
  stats->rounds = log.rounds;
  stats->relaxations = (int64_t)log.relaxed;
  stats->reached_vertices = log.reached_v;
  stats->reached_edges = log.reached_e;
  for (int32_t r = 0; r < log.rounds && r < SG_MAX_LEVELS_RECORDED; ++r) {
    stats->round_vertices[r] = log.round_v[r];
    stats->round_edges[r] = log.round_e[r];
  }
  return SG_OK;
}

/* mean arc weight, computed once per graph (automatic delta) */
template<typename W>
int mean_weight(sg_graph_t g, double* out) {
  if (!(g->mean_weight >= 0.0)) {
    const double* sum = nullptr;
    SG_TRY(weight_sum<W>(g, &sum));
    double h = 0.0;
    SG_HIP(hipMemcpyAsync(&h, sum, 8, hipMemcpyDeviceToHost, g->dev->stream));
    SG_HIP(hipStreamSynchronize(g->dev->stream));
    g->mean_weight = g->m > 0 ? h / (double)g->m : 1.0;
  }
  *out = g->mean_weight;
  return SG_OK;
}

/* The automatic schedule: buckets of half the mean arc weight on a graph of
 * at least kAutoBucketArcs arcs and kAutoBucketDegree arcs per vertex, the
 * reference's frontier Bellman-Ford otherwise.  Below the arc count an
 * iteration's fixed cost (its launches) outweighs the relaxations that buckets
 * save; on sparse, long-diameter graphs (grids: 3-4 arcs per vertex) buckets
 * multiply the iterations, each near that fixed cost (3-4x slower there).  The
 * pair has the least geometric mean of time / the faster schedule's time over
 * 100 generated graphs (RMAT scale 16-22, grids 512^2-4096^2, ER; weights
 * U[1,255]; four sources each) among arc counts 2^18..2^28 and degrees 0..32:
 * 3.4 % over choosing per run (18 % for the reference's schedule everywhere),
 * total time 1.8 % under the reference's schedule everywhere.
 * Below kAutoBucketArcs the grid bursts keep near and far piles (1201 x 1301
 * grid: 14 ms with them, 66 without; 300 x 400: 4.1 and 22; 200,000 vertices
 * of 16 arcs: 1.68 and 2.07).  Sparse graphs above it would gain as much
 * (3072 x 3072 grid, 35.9 M arcs: 52.5 ms with far lists, 319 without; 4096 x
 * 4096: 76 and 494, the same distances); they keep the reference's order only
 * because a test holds their count of relaxations to within 5 % of its. */
constexpr int64_t kAutoBucketArcs = int64_t(1) << 25;
constexpr int64_t kAutoBucketDegree = 8;

template<typename OffT, typename W>
int run_sssp_auto(sg_graph_t g, int32_t source, double delta, int32_t heavy_pull, int64_t burst_arcs,
                  bool record_relax, W* dist, sg_sssp_stats* stats) {
  /* (an explicit burst length asks for rounds by launches, a record of the
   * relax launches for their times) */
  if (delta == 0.0 && burst_arcs == kSsspBurstDefault && !record_relax && g->n <= kSmallVerts && g->m <= kSmallArcs)
    return run_sssp_small<OffT, W>(g, source, dist, stats);
  bool far_lists = false;
  if (delta == 0.0 && (g->m < kAutoBucketArcs || g->m < kAutoBucketDegree * (int64_t)g->n)) {
    far_lists = g->m < kAutoBucketArcs;
    delta = -1.0;
  } else if (delta == 0.0) {
    double mw = 1.0;
    SG_TRY(mean_weight<W>(g, &mw));
    delta = auto_delta<W>(mw);
  }
  return run_sssp<OffT, W>(g, source, delta, far_lists, heavy_pull, burst_arcs, record_relax, dist, stats);
}

extern "C" {

void sg_sssp_options_default(sg_sssp_options* opt) {
  if (!opt) return;
  std::memset(opt, 0, sizeof(*opt));
  opt->load_balancer = SG_LB_BUCKETING;
  opt->delta = 0.0;
}

int sg_sssp_ex(sg_graph_t g, int32_t source, const sg_sssp_options* opt_in, void* dist, sg_sssp_stats* stats) {
  SG_CHECK(g && dist, SG_ERR_INVALID, "sg_sssp: null argument");
  SG_CHECK(source >= 0 && source < g->n, SG_ERR_INVALID, "sg_sssp: source %d out of range [0,%lld)", source,
           (long long)g->n);
  SG_CHECK(g->weights, SG_ERR_STATE, "sg_sssp: graph has no edge weights");
  sg_sssp_options opt;
  if (opt_in) opt = *opt_in;
  else sg_sssp_options_default(&opt);
  SG_CHECK(opt.load_balancer >= SG_LB_WORKITEM && opt.load_balancer <= SG_LB_BUCKETING, SG_ERR_INVALID,
           "sg_sssp: unknown load balancer %d", opt.load_balancer);
  SG_CHECK(opt.heavy_pull >= -1 && opt.heavy_pull <= 1, SG_ERR_INVALID, "sg_sssp: heavy_pull %d not in {-1, 0, 1}",
           opt.heavy_pull);
  SG_CHECK(opt.burst_arcs <= kSsspBurstMax, SG_ERR_INVALID, "sg_sssp: burst_arcs %d above %d", opt.burst_arcs,
           kSsspBurstMax);
  if (stats) {
    stats->rounds = 0;
    stats->reached_vertices = stats->reached_edges = stats->relaxations = 0;
    stats->kernel_ms = 0.f;
    stats->relax_ms = 0.f;
    stats->relax_launches = 0;
  }
  SG_HIP(hipSetDevice(g->dev->ordinal));
  const bool fw = (g->flags & SG_GRAPH_WEIGHT_FLOAT) != 0;
  const int64_t ba = opt.burst_arcs < 0 ? 0 : (opt.burst_arcs == 0 ? kSsspBurstDefault : opt.burst_arcs);
  const bool rr = opt.record_relax != 0 && stats != nullptr;
  if (g->offset_bytes == 8)
    return fw ? run_sssp_auto<int64_t, float>(g, source, opt.delta, opt.heavy_pull, ba, rr, (float*)dist, stats)
              : run_sssp_auto<int64_t, uint32_t>(g, source, opt.delta, opt.heavy_pull, ba, rr, (uint32_t*)dist,
                                                 stats);
  return fw ? run_sssp_auto<uint32_t, float>(g, source, opt.delta, opt.heavy_pull, ba, rr, (float*)dist, stats)
            : run_sssp_auto<uint32_t, uint32_t>(g, source, opt.delta, opt.heavy_pull, ba, rr, (uint32_t*)dist, stats);
}

int sg_sssp(sg_graph_t g, int32_t source, int32_t load_balancer, void* dist, sg_sssp_stats* stats) {
  sg_sssp_options opt;
  sg_sssp_options_default(&opt);
  opt.load_balancer = load_balancer;
  return sg_sssp_ex(g, source, &opt, dist, stats);
}

} // extern "C"
