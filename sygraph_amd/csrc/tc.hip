/*
 * tc.hip -- triangle counting for gfx950 (TC::run + getNumTriangles,
 * algorithms/tc.hpp:67-138).
 *
 * The reference merges N(u) and N(v) for every arc u < v and divides the sum
 * by three; its running count is added inside the merge loop (tc.hpp:104), so
 * it over-counts.  This path computes the exact count on the
 * (degree, id)-oriented DAG: u -> v iff (deg u, u) < (deg v, v), each
 * triangle is then found once, from its lowest-ranked corner, and
 * out-degrees are O(sqrt(m)).
 *   1. orient: every vertex keeps, in order, the neighbours that rank higher,
 *      at the place of its list in the graph's own offsets (no second pass and
 *      no scan);
 *   2. intersect: N+(u) goes into an LDS hash table and the lists N+(v), v in
 *      N+(u), are looked up in it (segmented intersection).  A vertex of kHeavy
 *      or more ids takes a workgroup, whose waves share the table and deal the
 *      lists among them, the others a wave each.  Lists longer than the table
 *      takes are binary-searched in global memory, where they are sorted.
 * The count is uint64 (the reference's uint32 would overflow at scale 20).
 */
#include "traverse.hpp"

using namespace sg::trav;

namespace {

constexpr int kHeavy = 96;       /* ids from which a vertex takes a workgroup */
constexpr int kSlots1 = 2048;    /* table slots per wave */
constexpr int kSlots4 = 4 * kSlots1;
constexpr int kStage = kSlots4 / 2; /* longest N+(u) hashed in LDS */
constexpr int kLongList = 256;   /* lists this long are walked by the whole wave, */
constexpr int kMidList = 16;     /* this long by a quarter of it, shorter ones laid end to end */
constexpr int kLightChunk = 4;   /* vertices a wave claims at a time */

/* N+(v): where it starts in the oriented ids, and its length */
struct alignas(16) DagList {
  int64_t start;
  int32_t len, pad;
};

__global__ void __launch_bounds__(kBlock) degree_kernel(const int64_t* off8, const uint32_t* off4, int64_t n,
                                                        uint32_t* deg) {
  for (int64_t v = blockIdx.x * (int64_t)kBlock + threadIdx.x; v < n; v += (int64_t)gridDim.x * kBlock) {
    int64_t b, e;
    if (off8) list_bounds(off8, (uint32_t)v, b, e);
    else list_bounds(off4, (uint32_t)v, b, e);
    deg[v] = (uint32_t)(e - b);
  }
}

/* The oriented lists, sixteen lanes per vertex (the whole wave for lists over
 * kOrientWave), the ids' degrees gathered from 4 bytes a vertex.  Vertices of
 * kHeavy or more ids are listed: heavy[0] counts them (cleared before). */
constexpr int kTeam = 16, kOrientWave = 512;
template<typename OffT>
__global__ void __launch_bounds__(kBlock) orient_kernel(const OffT* off, const int32_t* cols, const uint32_t* deg,
                                                        int64_t n, DagList* dag, int32_t* dag_cols, uint32_t* heavy) {
  const int lane = lane_id(), team = lane / kTeam, me = lane % kTeam;
  const int64_t gwave = ((int64_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
  const int64_t nwaves = ((int64_t)gridDim.x * kBlock) >> 6;
  auto higher = [&](int64_t j, uint32_t u, uint32_t du, uint32_t& v) {
    v = (uint32_t)cols[j];
    const uint32_t dv = deg[v];
    return du < dv || (du == dv && u < v);
  };
  constexpr int kPerWave = 64 / kTeam;
  for (int64_t base = gwave * kPerWave; base < n; base += nwaves * kPerWave) {
    const int64_t u = base + team;
    int64_t b = 0, e = 0;
    if (u < n) list_bounds(off, (uint32_t)u, b, e);
    const uint32_t du = (uint32_t)(e - b);
    const bool wide = e - b > kOrientWave;
    uint32_t kept = 0;
    const int64_t end = wide ? b : e;
    for (int64_t j0 = b; ballot(j0 < end); j0 += 2 * kTeam) {
      bool keep[2];
      uint32_t v[2] = {0, 0};
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int64_t j = j0 + k * kTeam + me;
        keep[k] = j < end && higher(j, (uint32_t)u, du, v[k]);
      }
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const uint32_t m = (uint32_t)(ballot(keep[k]) >> (team * kTeam)) & ((1u << kTeam) - 1);
        if (keep[k]) dag_cols[b + kept + __popc(m & ((1u << me) - 1))] = (int32_t)v[k];
        kept += (uint32_t)__popc(m);
      }
    }
    for (uint64_t wides = ballot(wide && me == 0); wides; wides &= wides - 1) {
      const int k2 = __ffsll((unsigned long long)wides) - 1;
      const int64_t wb = (int64_t)wave_lane((uint64_t)b, k2), we = (int64_t)wave_lane((uint64_t)e, k2);
      const uint32_t wu = (uint32_t)(base + k2 / kTeam), wd = (uint32_t)(we - wb);
      uint32_t got = 0;
      for (int64_t j0 = wb; j0 < we; j0 += 4 * 64) {
        bool keep[4];
        uint32_t v[4] = {0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < 4; ++k) keep[k] = j0 + 64 * k + lane < we && higher(j0 + 64 * k + lane, wu, wd, v[k]);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint64_t m = ballot(keep[k]);
          if (keep[k]) dag_cols[wb + got + lanes_below(m)] = (int32_t)v[k];
          got += (uint32_t)__popcll(m);
        }
      }
      if (k2 / kTeam == team) kept = got;
    }
    if (me == 0 && u < n) {
      dag[u] = DagList{b, (int32_t)kept, 0};
      if (kept >= (uint32_t)kHeavy) heavy[1 + atomicAdd(&heavy[0], 1u)] = (uint32_t)u;
    }
  }
}

__device__ __forceinline__ bool search(const int32_t* list, int32_t len, int32_t x) {
  int32_t lo = 0, hi = len;
  while (lo < hi) {
    const int32_t mid = (lo + hi) >> 1;
    const int32_t y = list[mid];
    if (y == x) return true;
    if (y < x) lo = mid + 1;
    else hi = mid;
  }
  return false;
}

/* An open-addressing hash set in LDS: buckets of four ids (empty: -1), filled
 * from the front, a full bucket's overflow in the next ones.  A lookup reads a
 * bucket in one 16-byte access and ends there unless the bucket is full and
 * holds something else, which at 1/16 load is rare: a wave's 256 lookups take
 * one round, where linear probing over single slots took as many rounds as
 * the longest of its 256 sequences. */
struct Table {
  int32_t* slots;
  uint32_t mask; /* buckets - 1 */

  __device__ __forceinline__ uint32_t bucket(int32_t x) const {
    return ((uint32_t)x * 2654435761u >> 7) & mask; /* Knuth's multiplicative hash */
  }
  __device__ __forceinline__ void insert(int32_t x) const {
    for (uint32_t h = bucket(x);; h = (h + 1) & mask)
      for (int i = 0; i < 4; ++i)
        if (atomicCAS(&slots[4 * h + i], -1, x) == -1) return;
  }
};

/* at most 1/16 full where `slots` allows, at least half empty in every case */
__device__ __forceinline__ uint32_t table_size(uint32_t ids, uint32_t slots) {
  uint32_t size = 64;
  while (size < 16u * ids && size < slots) size <<= 1;
  return size;
}

/* Members of the table among four ids per lane (an id of -2: none); the count
 * of the wave, the same in every lane. */
__device__ __forceinline__ uint32_t lookup4(const Table& t, const int32_t (&x)[4]) {
  uint32_t h[4];
  int4 y[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    h[k] = t.bucket(x[k]);
    y[k] = *reinterpret_cast<const int4*>(t.slots + 4 * h[k]);
  }
  uint32_t hits = 0, more = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const bool hit = y[k].x == x[k] || y[k].y == x[k] || y[k].z == x[k] || y[k].w == x[k];
    hits += (uint32_t)__popcll(ballot(hit));
    more |= (!hit && y[k].w >= 0 && x[k] >= 0) ? 1u << k : 0u; /* full buckets go on in the next */
  }
  while (ballot(more != 0)) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      bool hit = false;
      if ((more >> k) & 1u) {
        h[k] = (h[k] + 1) & t.mask;
        const int4 z = *reinterpret_cast<const int4*>(t.slots + 4 * h[k]);
        hit = z.x == x[k] || z.y == x[k] || z.z == x[k] || z.w == x[k];
        if (hit || z.w < 0) more &= ~(1u << k);
      }
      hits += (uint32_t)__popcll(ballot(hit));
    }
  }
  return hits;
}

/* Four ids from position j of a list that ends at `end`, one 16-byte load
 * where they all exist (m: ids in the array); -2 past the end. */
__device__ __forceinline__ void load_list4(const int32_t* ids, int64_t j, int64_t end, int64_t m, int32_t (&x)[4]) {
  uint32_t y[4] = {0, 0, 0, 0};
  if (j < end) load_ids4(ids, j, m, y);
#pragma unroll
  for (int k = 0; k < 4; ++k) x[k] = j + k < end ? (int32_t)y[k] : -2;
}

/* The wave's lists -- this lane's is [vb, vb + vlen) -- counted against the
 * table with `count(x)`, the next four ids of a lane loaded while the last
 * four are looked up. */
template<typename Count>
__device__ __forceinline__ uint64_t walk_lists(const int32_t* ids, int64_t m, int64_t vb, uint32_t vlen,
                                               Count&& count) {
  const int lane = lane_id();
  uint64_t hits = 0;
  int32_t x[4], nx[4];
  for (uint64_t longs = ballot(vlen >= (uint32_t)kLongList); longs; longs &= longs - 1) {
    const int k2 = __ffsll((unsigned long long)longs) - 1;
    const int64_t lb = (int64_t)wave_lane((uint64_t)vb, k2), le = lb + wave_lane(vlen, k2);
    load_list4(ids, lb + 4 * lane, le, m, x);
    for (int64_t j0 = lb; j0 < le; j0 += 256) {
      load_list4(ids, j0 + 256 + 4 * lane, le, m, nx);
      hits += count(x);
#pragma unroll
      for (int k = 0; k < 4; ++k) x[k] = nx[k];
    }
  }
  uint64_t mids = ballot(vlen >= (uint32_t)kMidList && vlen < (uint32_t)kLongList);
  while (mids) { /* four lists at a time, sixteen lanes each */
    int mine = -1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int k2 = mids ? __ffsll((unsigned long long)mids) - 1 : -1;
      mids = mids ? mids & (mids - 1) : 0ull;
      if (lane / 16 == q) mine = k2;
    }
    const int from = mine < 0 ? 0 : mine;
    const int64_t lb = shfl_i64(vb, from);
    const uint32_t ll = __shfl(vlen, from, 64);
    const int64_t le = mine < 0 ? lb : lb + ll;
    int64_t j = lb + 4 * (lane % 16);
    load_list4(ids, j, le, m, x);
    while (ballot(x[0] >= 0)) {
      j += 64;
      load_list4(ids, j, le, m, nx);
      hits += count(x);
#pragma unroll
      for (int k = 0; k < 4; ++k) x[k] = nx[k];
    }
  }
  /* the short ones, laid end to end */
  const uint32_t slen = vlen < (uint32_t)kMidList ? vlen : 0u;
  const uint32_t incl = wave_inclusive_scan(slen);
  const uint32_t tot = wave_lane(incl, 63);
  const uint32_t excl = incl - slen;
  for (uint32_t t0 = 0; t0 < tot; t0 += 4 * 64) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t t = t0 + 64 * k + lane;
      const int owner = scan_owner(incl, t);
      const uint32_t before = __shfl(excl, owner, 64);
      const int64_t st = shfl_i64(vb, owner);
      x[k] = t < tot ? ids[st + (t - before)] : -2;
    }
    hits += count(x);
  }
  return hits;
}

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

/* w in N+(u) for a w of N+(v), v in N+(u), closes the triangle (u, v, w),
 * counted once at its lowest-ranked corner.  First the heavy vertices, a
 * workgroup each, then the others, a wave each: both claimed from counters
 * (next[0], next[1], zero at launch), since the work per vertex is skewed and
 * a fixed assignment leaves the busiest wave with several times the mean. */
__global__ void __launch_bounds__(kBlock) intersect_kernel(const DagList* dag, const int32_t* ids, int64_t m, int64_t n,
                                                           const uint32_t* heavy, unsigned long long* per_vertex,
                                                           unsigned long long* total, uint32_t* next) {
  __shared__ __align__(16) int32_t table[kSlots4];
  __shared__ uint32_t s_claim;
  __shared__ unsigned long long s_cnt;
  const int lane = lane_id(), wv = threadIdx.x >> 6;
  const uint32_t nheavy = heavy[0];
  uint64_t sum = 0; /* the same in every lane */
  for (;;) {
    if (threadIdx.x == 0) {
      s_claim = atomicAdd(&next[0], 1u);
      s_cnt = 0;
    }
    __syncthreads();
    const uint32_t h = s_claim;
    if (h >= nheavy) break;
    const uint32_t u = heavy[1 + h];
    const DagList lu = dag[u];
    const uint32_t du = (uint32_t)lu.len;
    const bool hashed = du <= (uint32_t)kStage;
    const Table t{table, table_size(du, kSlots4) / 4 - 1};
    if (hashed) {
      int4* t4 = reinterpret_cast<int4*>(table);
      for (uint32_t i = threadIdx.x; i <= t.mask; i += kBlock) t4[i] = int4{-1, -1, -1, -1};
      __syncthreads();
      for (uint32_t i = threadIdx.x; i < du; i += kBlock) t.insert(ids[lu.start + i]);
      __syncthreads();
    }
    uint64_t hits = 0;
    for (uint32_t v0 = 0; v0 < du; v0 += kBlock) { /* list v0 + 4 * lane + wave: a share of each 256 per wave */
      const uint32_t i = v0 + 4 * lane + wv;
      DagList lv{0, 0, 0};
      if (i < du) lv = dag[ids[lu.start + i]];
      if (hashed) {
        hits += walk_lists(ids, m, lv.start, (uint32_t)lv.len, [&](const int32_t (&x)[4]) { return lookup4(t, x); });
      } else {
        hits += walk_lists(ids, m, lv.start, (uint32_t)lv.len, [&](const int32_t (&x)[4]) {
          uint32_t c = 0;
          for (int k = 0; k < 4; ++k)
            c += (uint32_t)__popcll(ballot(x[k] >= 0 && search(ids + lu.start, lu.len, x[k])));
          return c;
        });
      }
    }
    if (lane == 0 && hits) atomicAdd(&s_cnt, (unsigned long long)hits);
    sum += hits;
    __syncthreads(); /* also: nobody looks up in the table any more */
    if (threadIdx.x == 0 && per_vertex) per_vertex[u] = s_cnt;
  }
  int32_t* mine = table + wv * kSlots1;
  for (;;) {
    uint32_t claim = 0;
    if (lane == 0) claim = atomicAdd(&next[1], 1u);
    const int64_t u0 = (int64_t)wave_lane(claim, 0) * kLightChunk;
    if (u0 >= n) break;
    const int64_t u1 = u0 + kLightChunk < n ? u0 + kLightChunk : n;
    DagList lists{0, 0, 0};
    if (lane < kLightChunk && u0 + lane < u1) lists = dag[u0 + lane];
    for (int64_t u = u0; u < u1; ++u) {
      const int64_t ub = (int64_t)wave_lane((uint64_t)lists.start, (int)(u - u0));
      const uint32_t du = wave_lane((uint32_t)lists.len, (int)(u - u0));
      if (du >= (uint32_t)kHeavy) continue;
      uint64_t hits = 0;
      if (du >= 2) {
        const Table t{mine, table_size(du, kSlots1) / 4 - 1};
        int4* t4 = reinterpret_cast<int4*>(mine);
        for (uint32_t i = lane; i <= t.mask; i += 64) t4[i] = int4{-1, -1, -1, -1};
        wave_lds_fence();
        for (uint32_t i = lane; i < du; i += 64) t.insert(ids[ub + i]);
        wave_lds_fence();
        for (uint32_t v0 = 0; v0 < du; v0 += 64) {
          DagList lv{0, 0, 0};
          if (v0 + lane < du) lv = dag[ids[ub + v0 + lane]];
          hits += walk_lists(ids, m, lv.start, (uint32_t)lv.len, [&](const int32_t (&x)[4]) { return lookup4(t, x); });
        }
        wave_lds_fence();
      }
      if (lane == 0 && per_vertex) per_vertex[u] = hits;
      sum += hits;
    }
  }
  if (lane == 0 && sum) atomicAdd(total, (unsigned long long)sum);
}

} // namespace

extern "C" int sg_tc(sg_graph_t g, uint64_t* count, uint64_t* per_vertex) {
  SG_CHECK(g && count, SG_ERR_INVALID, "sg_tc: null argument");
  SG_HIP(hipSetDevice(g->dev->ordinal));
  sg_device_t dev = g->dev;
  hipStream_t s = dev->stream;
  const int64_t n = g->n;
  /* the oriented graph is kept with the graph, so repeated counts allocate nothing */
  const int64_t m = g->m;
  uint32_t *deg = nullptr, *heavy = nullptr;
  DagList* dag = nullptr;
  int32_t* dag_cols = nullptr;
  unsigned long long* total = nullptr;
  SG_TRY(sg::graph_buffer(g, "tc_deg", 4 * (size_t)(n + 1), &deg));
  SG_TRY(sg::graph_buffer(g, "tc_heavy", 4 * (size_t)(m / kHeavy + 2), &heavy));
  SG_TRY(sg::graph_buffer(g, "tc_dag", sizeof(DagList) * (size_t)(n + 1), &dag));
  SG_TRY(sg::graph_buffer(g, "tc_dag_cols", 4 * (size_t)(m + 1), &dag_cols));
  SG_TRY(sg::graph_buffer(g, "tc_total", 16, &total)); /* the count, then the two claim counters */
  const int grid = dev->cus * 8;
  const bool wide = g->offset_bytes == 8;
  SG_TRY(sg::zero_async(dev, heavy, 4));
  SG_TRY(sg::zero_async(dev, total, 16));
  degree_kernel<<<grid, kBlock, 0, s>>>(wide ? (const int64_t*)g->offsets : nullptr,
                                        wide ? nullptr : (const uint32_t*)g->offsets, n, deg);
  if (wide)
    orient_kernel<int64_t><<<grid, kBlock, 0, s>>>((const int64_t*)g->offsets, g->cols, deg, n, dag, dag_cols, heavy);
  else
    orient_kernel<uint32_t><<<grid, kBlock, 0, s>>>((const uint32_t*)g->offsets, g->cols, deg, n, dag, dag_cols, heavy);
  /* persistent workgroups: as many as the table's 32 KB leave room for */
  intersect_kernel<<<dev->cus * 5, kBlock, 0, s>>>(dag, dag_cols, m, n, heavy, (unsigned long long*)per_vertex, total,
                                                   reinterpret_cast<uint32_t*>(total + 1));
  SG_HIP(hipGetLastError());
  unsigned long long h = 0;
  SG_HIP(hipMemcpyAsync(&h, total, 8, hipMemcpyDeviceToHost, s));
  SG_HIP(hipStreamSynchronize(s));
  *count = h;
  return SG_OK;
}
