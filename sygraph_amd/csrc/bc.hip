/*
 * bc.hip -- betweenness centrality (BC::run, algorithms/bc.hpp:118-200) for
 * gfx950.
 *
 * Per source s:
 *  1. depths from the fused BFS (sg_bfs, hybrid push/pull);
 *  2. vertices grouped by level, in no particular order (every vertex's sums
 *     are its own): a counting sort, or with more than kCountLevels levels a
 *     radix sort of (level, vertex);
 *  3. forward, level by level: sigma(v) = sum of scale(L - 1) * sigma(u) over
 *     in-arcs u -> v with depth(u) = depth(v) - 1 = L - 1, where scale(L) is
 *     the power of two that brings the level's largest sigma into [0.5, 1) --
 *     path counts overflow FP64 on long-diameter graphs (a 4096 x 4096 grid
 *     has ~1e2464 shortest paths corner to corner), and power-of-two scaling
 *     is exact;
 *  4. backward, deepest level first: delta(u) = scale(L) * sigma(u) * sum of
 *     R(w) over out-arcs u -> w with depth(w) = depth(u) + 1 = L + 1, and R(u)
 *     = (1 + delta(u)) / sigma(u), one division per vertex and one gather per
 *     arc (the scales of w's level cancel); bc(u) += delta(u) for u != s (no
 *     halving on undirected graphs, as bc.hpp:186-196).
 * Steps 3 and 4 are pulls: each vertex gathers its own sum, so there are no
 * floating-point atomics and results do not depend on scheduling.  Both read
 * every arc of the reached vertices once; what bounds them is a vertex's
 * dependent gathers (id, level bit, value), so eight lanes share a vertex,
 * four arcs each in flight, and vertices of more than kHub arcs get a
 * workgroup (a wave for 64 vertices one after another, hubs included, took
 * 0.7-1.3 ms for RMAT scale 18's largest level).  The partial sums are added
 * in a fixed order.  sigma, R and the per-source accumulation are FP64; the
 * output adds the FP64 total to the caller's float array once at the end.
 */
#include <rocprim/device/device_radix_sort.hpp>

#include <algorithm>
#include <cstring>
#include <memory>
#include <vector>

#include "internal.hpp"
#include "traverse.hpp"

using namespace sg::trav;

namespace {

constexpr int kHub = 512;          /* degree above which a workgroup sums one vertex */
constexpr int kTeam = 8;           /* lanes that share a vertex otherwise */
constexpr int kCountLevels = 1024; /* levels up to which the counting sort's histograms fit in LDS */
constexpr int kMaxSlots = 64;   /* per-level maximum of sigma: slots, one cache line apart */
constexpr int kSlotStride = 16; /* unsigned long long per 128-byte line */
constexpr int64_t kLevelBitmapBytes = 1ll << 30; /* per-level bitmaps up to 1 GiB, else depth[] tests */
constexpr size_t kKeepBytes = size_t(64) << 20;

/* sum over groups of kLanes lanes, in every lane (fixed butterfly) */
template<int kLanes>
__device__ __forceinline__ double lanes_sum(double x) {
#pragma unroll
  for (int o = kLanes / 2; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}

/* Counting sort by level: the workgroups' histograms added into count[0..nl)
 * (cleared before), the level starts, then each workgroup's vertices at the
 * range it reserves in every level.  The first pass also writes the level
 * bitmaps of at most 64 levels (lane L keeps the word's bits of level L). */
__global__ void __launch_bounds__(kBlock) level_count_kernel(const int32_t* depth, int64_t n, int64_t w0, int32_t nl,
                                                             uint32_t* count, uint64_t* lbm) {
  __shared__ uint32_t s_n[kCountLevels];
  for (int l = threadIdx.x; l < nl; l += kBlock) s_n[l] = 0;
  __syncthreads();
  const int lane = lane_id();
  const int64_t gw = ((int64_t)blockIdx.x * kBlock + threadIdx.x) >> 6, nw = ((int64_t)gridDim.x * kBlock) >> 6;
  for (int64_t w = gw; w < w0; w += nw) {
    const int64_t v = w * 64 + lane;
    const int32_t d = v < n ? depth[v] : -1;
    const bool in = d >= 0 && d < nl;
    if (lbm) {
      uint64_t mine = 0;
      for (int l = 0; l < nl; ++l) {
        const uint64_t m = ballot(in && d == l);
        if (l == lane) mine = m;
      }
      if (lane < nl) {
        lbm[(int64_t)lane * w0 + w] = mine;
        if (mine) atomicAdd(&s_n[lane], (uint32_t)__popcll(mine));
      }
    } else if (in) {
      atomicAdd(&s_n[d], 1u);
    }
  }
  __syncthreads();
  for (int l = threadIdx.x; l < nl; l += kBlock)
    if (s_n[l]) atomicAdd(&count[l], s_n[l]);
}

/* lvl[l] = start of level l, lvl[nl] = the reached vertices; cursor = the starts */
__global__ void __launch_bounds__(64) level_scan_kernel(const uint32_t* count, int32_t nl, int64_t* lvl,
                                                        uint32_t* cursor) {
  uint32_t carry = 0;
  for (int32_t b = 0; b < nl; b += 64) {
    const int32_t l = b + lane_id();
    const uint32_t c = l < nl ? count[l] : 0u;
    const uint32_t incl = wave_inclusive_scan(c);
    if (l < nl) {
      lvl[l] = carry + incl - c;
      cursor[l] = carry + incl - c;
    }
    carry += wave_lane(incl, 63);
  }
  if (lane_id() == 0) lvl[nl] = carry;
}

__global__ void __launch_bounds__(kBlock) level_scatter_kernel(const int32_t* depth, int64_t n, int32_t nl,
                                                               uint32_t* cursor, int32_t* order) {
  __shared__ uint32_t s_n[kCountLevels];
  const int64_t per = (n + gridDim.x - 1) / gridDim.x;
  const int64_t first = (int64_t)blockIdx.x * per, last = first + per < n ? first + per : n;
  for (int l = threadIdx.x; l < nl; l += kBlock) s_n[l] = 0;
  __syncthreads();
  for (int64_t v = first + threadIdx.x; v < last; v += kBlock) {
    const int32_t d = depth[v];
    if (d >= 0 && d < nl) atomicAdd(&s_n[d], 1u);
  }
  __syncthreads();
  for (int l = threadIdx.x; l < nl; l += kBlock)
    if (s_n[l]) s_n[l] = atomicAdd(&cursor[l], s_n[l]);
  __syncthreads();
  for (int64_t v = first + threadIdx.x; v < last; v += kBlock) {
    const int32_t d = depth[v];
    if (d >= 0 && d < nl) order[atomicAdd(&s_n[d], 1u)] = (int32_t)v;
  }
}

/* vertices of more than kHub arcs (hub[0] counts them, cleared before) */
template<typename OffT>
__global__ void __launch_bounds__(kBlock) hub_list_kernel(const OffT* off, int64_t n, uint32_t* hub) {
  for (int64_t v = blockIdx.x * (int64_t)kBlock + threadIdx.x; v < n; v += (int64_t)gridDim.x * kBlock)
    if ((int64_t)(off[v + 1] - off[v]) > kHub) hub[1 + atomicAdd(&hub[0], 1u)] = (uint32_t)v;
}

__global__ void level_keys_kernel(const int32_t* depth, int64_t n, int32_t nlevels, uint32_t* keys, int32_t* ids) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int32_t d = depth[i];
    keys[i] = (d >= 0 && d < nlevels) ? (uint32_t)d : (uint32_t)nlevels;
    ids[i] = (int32_t)i;
  }
}

/* lvl[k] = first position of key k in the sorted keys; lvl[0..nlevels+1]
 * preset to n by the caller (levels 0..nlevels-1 are never empty) */
__global__ void level_starts_kernel(const uint32_t* keys, int64_t n, int64_t* lvl) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    if (i == 0 || keys[i] != keys[i - 1]) lvl[keys[i]] = i;
}

/* lbm[L * w0 + word]: bit v set iff depth(v) == L, for L < nlevels; a wave
 * owns the word of its 64 vertices, so there are no atomics (the words are
 * zeroed before) */
__global__ void level_bits_kernel(const int32_t* depth, int64_t n, int64_t w0, int32_t nlevels, uint64_t* lbm) {
  const int lane = lane_id();
  const int64_t gwave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
  for (int64_t w = gwave; w < w0; w += nwaves) {
    const int64_t v = w * 64 + lane;
    const int32_t d = v < n ? depth[v] : -1;
    const bool in = d >= 0 && d < nlevels;
    uint64_t todo = ballot(in);
    while (todo) { /* one store per distinct level among the wave's vertices */
      const int k = __ffsll((unsigned long long)todo) - 1;
      const int32_t lev = __shfl(d, k, 64);
      const uint64_t m = ballot(in && d == lev);
      if (lane == 0) lbm[(int64_t)lev * w0 + w] = m;
      todo &= ~m;
    }
  }
}

__device__ __forceinline__ bool bit_of(const uint64_t* bm, int32_t v) { return (bm[v >> 6] >> (v & 63)) & 1ull; }

/* The largest sigma of a level, in a block of slots: three blocks in turn, the
 * level's own, the level before's, which is read, and the next level's, which
 * is cleared meanwhile (a block per level would be 8 KiB times the levels). */
constexpr int kSlotWords = kMaxSlots * kSlotStride;
__device__ __forceinline__ unsigned long long* max_slots(unsigned long long* all, int32_t L) {
  return all + (int64_t)(L % 3) * kSlotWords;
}

__global__ void bc_source_init_kernel(double* sigma, int32_t s, unsigned long long* level_max) {
  for (int i = threadIdx.x; i < 3 * kSlotWords; i += blockDim.x) level_max[i] = 0ull;
  if (threadIdx.x == 0) sigma[s] = 1.0;
}

/* 2^-e for the exponent e of a level's largest sigma (1 where none was
 * recorded: the source's level).  All threads call; one barrier. */
__device__ __forceinline__ double level_scale(const unsigned long long* level_max) {
  __shared__ double s_scale;
  if (threadIdx.x < 64) {
    static_assert(kMaxSlots == 64, "a slot per lane");
    const double mx =
        __longlong_as_double((long long)wave_max_u64(level_max[(int)threadIdx.x * kSlotStride]));
    int ex = 0;
    (void)frexp(mx, &ex);
    if (threadIdx.x == 0) s_scale = ldexp(1.0, -ex);
  }
  __syncthreads();
  return s_scale;
}

/* Sum of value(x) over the neighbours x of each vertex of level L that are in
 * `bm` (or, where it is null, at depth `want`); store(v, sum) runs once per
 * vertex.  The first hub_blocks workgroups take the hubs of the level (hub[0]
 * of them in all, whatever their level), a workgroup each; the others the
 * level's vertices in `order`, kTeam lanes each. */
template<typename OffT, typename ValueF, typename StoreF>
__device__ __forceinline__ void gather_level(const int32_t* order, const int64_t* lvl, int32_t L, const uint32_t* hub,
                                             int hub_blocks, const OffT* off, const int32_t* cols,
                                             const int32_t* depth, const uint64_t* bm, int32_t want, ValueF value,
                                             StoreF store) {
  constexpr int kArcs = 4; /* per lane in flight */
  auto part_sum = [&](int64_t a, int64_t b, int me, int width) {
    double acc = 0.0;
    for (int64_t e = a + me; e < b; e += (int64_t)kArcs * width) {
      int32_t x[kArcs];
      bool in[kArcs];
      double y[kArcs];
#pragma unroll
      for (int k = 0; k < kArcs; ++k) x[k] = e + k * width < b ? cols[e + k * width] : -1;
#pragma unroll
      for (int k = 0; k < kArcs; ++k) in[k] = x[k] >= 0 && (bm ? bit_of(bm, x[k]) : depth[x[k]] == want);
#pragma unroll
      for (int k = 0; k < kArcs; ++k) y[k] = in[k] ? value(x[k]) : 0.0;
#pragma unroll
      for (int k = 0; k < kArcs; ++k) acc += y[k];
    }
    return acc;
  };
  const int lane = lane_id(), wv = threadIdx.x >> 6;
  if ((int)blockIdx.x < hub_blocks) {
    __shared__ double s_part[kBlock / 64];
    const uint32_t nh = hub[0];
    for (uint32_t h = blockIdx.x; h < nh; h += (uint32_t)hub_blocks) {
      const int32_t v = (int32_t)hub[1 + h];
      if (depth[v] != L) continue;
      const double acc = lanes_sum<64>(part_sum((int64_t)off[v], (int64_t)off[v + 1], (int)threadIdx.x, kBlock));
      if (lane == 0) s_part[wv] = acc;
      __syncthreads();
      if (threadIdx.x == 0) {
        double total = 0.0;
        for (int w = 0; w < kBlock / 64; ++w) total += s_part[w];
        store(v, total);
      }
      __syncthreads();
    }
    return;
  }
  const int64_t begin = lvl[L], end = lvl[L + 1];
  constexpr int kPerWave = 64 / kTeam;
  const int64_t gwave = ((int64_t)(blockIdx.x - hub_blocks) * kBlock + threadIdx.x) >> 6;
  const int64_t nwaves = ((int64_t)(gridDim.x - hub_blocks) * kBlock) >> 6;
  for (int64_t base = begin + gwave * kPerWave; base < end; base += nwaves * kPerWave) {
    const int64_t i = base + lane / kTeam;
    int32_t v = -1;
    int64_t a = 0, b = 0;
    if (i < end) {
      v = order[i];
      list_bounds(off, (uint32_t)v, a, b);
      if (b - a > kHub) { /* a hub's workgroup has it */
        v = -1;
        b = a;
      }
    }
    const double sum = lanes_sum<kTeam>(part_sum(a, b, lane % kTeam, kTeam));
    if (v >= 0 && lane % kTeam == 0) store(v, sum);
  }
}

/* prev_bm: bitmap of level L-1 (L2-resident), or nullptr to test depth[]:
 * sigma is only loaded for real parents.  scale[L-1] is written here, for the
 * way back; the deepest level's R is final here. */
template<typename OffT>
__global__ void __launch_bounds__(kBlock) sigma_level_kernel(const int32_t* order, const int64_t* lvl, int32_t L,
                                                             int32_t nl, const uint32_t* hub, int hub_blocks,
                                                             const OffT* in_off, const int32_t* in_cols,
                                                             const int32_t* depth, const uint64_t* prev_bm,
                                                             double* sigma, double* r, unsigned long long* slots,
                                                             double* scale) {
  const double sc = level_scale(max_slots(slots, L - 1));
  unsigned long long *level_max = max_slots(slots, L), *cleared = max_slots(slots, L + 1);
  if (blockIdx.x == 0) {
    for (int i = threadIdx.x; i < kMaxSlots; i += kBlock) cleared[i * kSlotStride] = 0ull;
    if (threadIdx.x == 0) scale[L - 1] = sc;
  }
  double mx = 0.0;
  gather_level<OffT>(
      order, lvl, L, hub, hub_blocks, in_off, in_cols, depth, prev_bm, L - 1,
      [&](int32_t u) { return sigma[u]; },
      [&](int32_t v, double s) {
        s *= sc;
        sigma[v] = s;
        if (L == nl - 1) r[v] = 1.0 / s;
        mx = s > mx ? s : mx;
      });
  /* positive doubles order like their bit patterns; one atomic per workgroup,
   * spread over kMaxSlots cache lines (same-address atomics from every wave
   * serialise across the chip) */
  __shared__ unsigned long long red[kBlock / 64];
  unsigned long long bits = (unsigned long long)__double_as_longlong(mx);
  bits = wave_max_u64(bits);
  if (lane_id() == 0) red[threadIdx.x >> 6] = bits;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long m = 0;
    for (int w = 0; w < kBlock / 64; ++w) m = red[w] > m ? red[w] : m;
    if (m) atomic_max(&level_max[(blockIdx.x % kMaxSlots) * kSlotStride], m);
  }
}

/* next_bm: bitmap of level L+1, or nullptr to test depth[] */
template<typename OffT>
__global__ void __launch_bounds__(kBlock) delta_level_kernel(const int32_t* order, const int64_t* lvl, int32_t L,
                                                             const uint32_t* hub, int hub_blocks, const OffT* off,
                                                             const int32_t* cols, const int32_t* depth,
                                                             const uint64_t* next_bm, const double* sigma, double* r,
                                                             const double* scale, double* acc_bc) {
  const double sc = scale[L];
  gather_level<OffT>(
      order, lvl, L, hub, hub_blocks, off, cols, depth, next_bm, L + 1, [&](int32_t w) { return r[w]; },
      [&](int32_t v, double sum) {
        const double s = sigma[v], d = s * sum * sc;
        r[v] = (1.0 + d) / s;
        acc_bc[v] += d;
      });
}

__global__ void add_to_float_kernel(const double* acc, float* out, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    out[i] = (float)((double)out[i] + acc[i]);
}

__global__ void fill_f64_kernel(double* p, double v, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = v;
}
__global__ void fill_i64_kernel(int64_t* p, int64_t v, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = v;
}

template<typename OffT>
int run_bc(sg_graph_t g, int32_t nsrc, const int32_t* sources, float* out) {
  sg_device_t dev = g->dev;
  hipStream_t st = dev->stream;
  const int64_t n = g->n, w0 = (n + 63) / 64;
  for (int32_t i = 0; i < nsrc; ++i)
    SG_CHECK(sources[i] >= 0 && sources[i] < n, SG_ERR_INVALID, "sg_bc: source %d out of range [0,%lld)", sources[i],
             (long long)n);
  const OffT* off = (const OffT*)g->offsets;
  const OffT* in_off = (const OffT*)(g->inv_offsets ? g->inv_offsets : g->offsets);
  const int32_t* in_cols = g->inv_cols ? g->inv_cols : g->cols;
  const bool directed = in_off != off;
  /* kept with the graph, so that repeated calls allocate nothing, but no part
   * of more than kKeepBytes beyond the call: of a graph of 8 M vertices and
   * more, or of long diameter, the calls take far longer than allocating */
  struct Trim {
    sg_graph_t g;
    ~Trim() { sg::graph_buffers_trim(g, "bc_", kKeepBytes); }
  } trim{g};
  int32_t *depth = nullptr, *order = nullptr;
  int64_t* lvl = nullptr;
  double *sigma = nullptr, *r = nullptr, *acc = nullptr, *scale = nullptr;
  unsigned long long* level_max = nullptr;
  uint32_t *count = nullptr, *hubs = nullptr, *in_hubs = nullptr;
  const size_t hub_cap = (size_t)(g->m / kHub) + 2;
  SG_TRY(sg::graph_buffer(g, "bc_depth", 4 * (size_t)(n + 1), &depth));
  SG_TRY(sg::graph_buffer(g, "bc_order", 4 * (size_t)(n + 1), &order));
  SG_TRY(sg::graph_buffer(g, "bc_lvl", 8 * (size_t)(n + 2), &lvl));
  SG_TRY(sg::graph_buffer(g, "bc_sigma", 8 * (size_t)(n + 1), &sigma));
  SG_TRY(sg::graph_buffer(g, "bc_r", 8 * (size_t)(n + 1), &r));
  SG_TRY(sg::graph_buffer(g, "bc_acc", 8 * (size_t)(n + 1), &acc));
  SG_TRY(sg::graph_buffer(g, "bc_level_max", 8 * 3 * kSlotWords, &level_max));
  SG_TRY(sg::graph_buffer(g, "bc_count", 4 * 2 * kCountLevels, &count));
  SG_TRY(sg::graph_buffer(g, "bc_hubs", 4 * hub_cap, &hubs));
  if (directed) SG_TRY(sg::graph_buffer(g, "bc_in_hubs", 4 * hub_cap, &in_hubs));
  else in_hubs = hubs;
  const int grid_n = sg::grid_for(dev, n, kBlock, 4);
  const int grid_lvl = dev->cus * 8, hub_blocks = dev->cus * 2;
  fill_f64_kernel<<<grid_n, kBlock, 0, st>>>(acc, 0.0, n);
  SG_TRY(sg::zero_async(dev, hubs, 4));
  hub_list_kernel<OffT><<<grid_n, kBlock, 0, st>>>(off, n, hubs);
  if (directed) {
    SG_TRY(sg::zero_async(dev, in_hubs, 4));
    hub_list_kernel<OffT><<<grid_n, kBlock, 0, st>>>(in_off, n, in_hubs);
  }
  SG_HIP(hipGetLastError());

  sg_bfs_options opt;
  sg_bfs_options_default(&opt);
  opt.policy = SG_POLICY_HYBRID;
  opt.record_levels = 0;
  auto stats = std::make_unique<sg_bfs_stats>();
  for (int32_t si = 0; si < nsrc; ++si) {
    const int32_t s = sources[si];
    SG_TRY(sg_bfs(g, s, &opt, depth, stats.get()));
    const int32_t nl = stats->levels; /* depths 0 .. nl-1 */
    if (nl < 2) continue;             /* nothing reached: no dependencies */
    /* level bitmaps when they take at most kLevelBitmapBytes (long-diameter
     * graphs fall back to testing depth[]) */
    const bool use_lbm = (int64_t)nl * w0 * 8 <= kLevelBitmapBytes;
    uint64_t* lbm = nullptr;
    if (use_lbm) SG_TRY(sg::graph_buffer(g, "bc_lbm", 8 * (size_t)nl * w0, &lbm));
    SG_TRY(sg::graph_buffer(g, "bc_scale", 8 * (size_t)nl, &scale));
    if (nl <= kCountLevels) {
      uint32_t* cursor = count + kCountLevels;
      fill_i64_kernel<<<1, kBlock, 0, st>>>((int64_t*)count, 0, kCountLevels / 2);
      level_count_kernel<<<grid_n, kBlock, 0, st>>>(depth, n, w0, nl, count, use_lbm && nl <= 64 ? lbm : nullptr);
      level_scan_kernel<<<1, 64, 0, st>>>(count, nl, lvl, cursor);
      level_scatter_kernel<<<grid_n, kBlock, 0, st>>>(depth, n, nl, cursor, order);
    } else {
      uint32_t* keys = nullptr; /* both sides of the sort */
      int32_t* ids = nullptr;
      void* tmp = nullptr;
      size_t tmp_bytes = 0;
      int bits = 1;
      while ((1u << bits) <= (uint32_t)nl) ++bits;
      SG_TRY(sg::graph_buffer(g, "bc_keys", 4 * (size_t)(2 * n + 2), &keys));
      SG_TRY(sg::graph_buffer(g, "bc_ids", 4 * (size_t)(n + 1), &ids));
      SG_HIP(rocprim::radix_sort_pairs(nullptr, tmp_bytes, keys, keys + n + 1, ids, order, (size_t)n, 0, bits, st));
      SG_TRY(sg::graph_buffer(g, "bc_sort_tmp", tmp_bytes + 16, &tmp));
      level_keys_kernel<<<grid_n, kBlock, 0, st>>>(depth, n, nl, keys, ids);
      SG_HIP(rocprim::radix_sort_pairs(tmp, tmp_bytes, keys, keys + n + 1, ids, order, (size_t)n, 0, bits, st));
      fill_i64_kernel<<<sg::grid_for(dev, nl + 2, kBlock, 1), kBlock, 0, st>>>(lvl, n, nl + 2);
      level_starts_kernel<<<grid_n, kBlock, 0, st>>>(keys + n + 1, n, lvl);
    }
    if (use_lbm && nl > 64) {
      fill_i64_kernel<<<sg::grid_for(dev, (int64_t)nl * w0, kBlock, 4), kBlock, 0, st>>>((int64_t*)lbm, 0,
                                                                                      (int64_t)nl * w0);
      level_bits_kernel<<<sg::grid_for(dev, n, kBlock, 4), kBlock, 0, st>>>(depth, n, w0, nl, lbm);
    }
    bc_source_init_kernel<<<1, kBlock, 0, st>>>(sigma, s, level_max);
    auto lbm_of = [&](int32_t L) -> const uint64_t* { return use_lbm ? lbm + (int64_t)L * w0 : nullptr; };
    for (int32_t L = 1; L < nl; ++L)
      sigma_level_kernel<OffT><<<grid_lvl, kBlock, 0, st>>>(order, lvl, L, nl, in_hubs, hub_blocks, in_off, in_cols,
                                                            depth, lbm_of(L - 1), sigma, r, level_max, scale);
    /* the source's own dependency is not counted */
    for (int32_t L = nl - 2; L >= 1; --L)
      delta_level_kernel<OffT><<<grid_lvl, kBlock, 0, st>>>(order, lvl, L, hubs, hub_blocks, off, g->cols, depth,
                                                            lbm_of(L + 1), sigma, r, scale, acc);
    SG_HIP(hipGetLastError());
  }
  add_to_float_kernel<<<grid_n, kBlock, 0, st>>>(acc, out, n);
  SG_HIP(hipGetLastError());
  SG_HIP(hipStreamSynchronize(st));
  return SG_OK;
}

} // namespace

extern "C" int sg_bc(sg_graph_t g, int32_t nsrc, const int32_t* sources_host, float* bc) {
  SG_CHECK(g && bc && (nsrc == 0 || sources_host), SG_ERR_INVALID, "sg_bc: null argument");
  SG_CHECK(nsrc >= 0, SG_ERR_INVALID, "sg_bc: negative source count");
  SG_HIP(hipSetDevice(g->dev->ordinal));
  if (g->offset_bytes == 8) return run_bc<int64_t>(g, nsrc, sources_host, bc);
  return run_bc<uint32_t>(g, nsrc, sources_host, bc);
}
