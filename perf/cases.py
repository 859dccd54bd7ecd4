"""The work whose time is kept: one call of each algorithm entry point over the
graphs it is used on.

A case names a path (the call), a graph family with its size, and the options
of the call.  The graphs are made here with torch from the case and the seed
alone, handed over as a device-resident CSR (sg_graph_create) and kept with
the outputs' buffers, as a program that runs queries on a loaded graph keeps
them.  Families:

  rmat   a/b/c/d = .57/.19/.19/.05, ids relabelled at random: skewed degrees
         and a diameter of a few hops (social and web graphs)
  grid   rows x cols lattice with a share of its edges deleted: degree four
         and thousands of hops (road networks)
  er     uniform endpoints: even degrees, a small diameter

Vertex counts need not be powers of two (RMAT ids are folded into range).
"""
import ctypes as C
import math
import os

import numpy as np
import torch

import sygraph_amd as sg

POLICY = {"push": sg.POLICY_PUSH, "pull": sg.POLICY_PULL, "hybrid": sg.POLICY_HYBRID, "learned": sg.POLICY_LEARNED}
DEV = "cuda"
_device = None


def listed():
    return [
        # the smallest call, with the options that BFS.run has by default: a
        # query on a neighbourhood graph, all launches and latency
        {"name": "bfs_small", "path": "bfs", "graph": "rmat", "n": 1024, "degree": 8, "policy": "push", "levels": True},
        # the headline: 16 traversals of RMAT scale 24 edge factor 16, direction-optimising
        {"name": "bfs_many_rmat24", "path": "bfs_many", "graph": "rmat", "n": 1 << 24, "degree": 16, "sources": 16,
         "policy": "hybrid"},
        # a road-like network: thousands of levels of a few thousand vertices
        {"name": "bfs_grid", "path": "bfs", "graph": "grid", "n": 3001, "cols": 2999, "p_delete": 0.05,
         "policy": "push"},
        # a directed graph of even degrees with 32-bit offsets: the inverse CSR and no hubs
        {"name": "bfs_directed", "path": "bfs", "graph": "er", "n": 3000001, "degree": 12, "directed": True,
         "offset_bytes": 4, "policy": "hybrid"},
        # SSSP on the headline graph with integer weights in [1, 255]: the bucketed schedule
        {"name": "sssp_rmat24", "path": "sssp", "graph": "rmat", "n": 1 << 24, "degree": 16, "weights": "u32"},
        # SSSP with real weights on a directed graph below the bucketed schedule's size
        {"name": "sssp_directed_f32", "path": "sssp", "graph": "rmat", "n": 700001, "degree": 14, "directed": True,
         "weights": "f32"},
        # SSSP on a road-like network: thousands of small rounds
        {"name": "sssp_grid", "path": "sssp", "graph": "grid", "n": 1201, "cols": 1301, "p_delete": 0.05,
         "weights": "u32"},
        # components of a skewed graph: one giant component and many small ones
        {"name": "cc_rmat20", "path": "cc", "graph": "rmat", "n": 1 << 20, "degree": 32},
        # exact triangle count with the count per vertex
        {"name": "tc_rmat", "path": "tc", "graph": "rmat", "n": 600000, "degree": 24},
        # betweenness from a few sources, one after another, in FP64
        {"name": "bc_rmat18", "path": "bc", "graph": "rmat", "n": 1 << 18, "degree": 16, "sources": 4},
        # betweenness from a batch of sources
        {"name": "bc_batched_rmat20", "path": "bc_batched", "graph": "rmat", "n": 1 << 20, "degree": 16, "sources": 64},
        # hop counts from a batch of sources, the dense graph of the batched measurements
        {"name": "bfs_multi_rmat20", "path": "bfs_multi", "graph": "rmat", "n": 1 << 20, "degree": 56, "sources": 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["bfs", "bfs", "bfs_many", "sssp", "sssp", "cc", "tc", "bc", "bc_batched", "bfs_multi"])
    graph = rng.choice(["rmat", "rmat", "er", "grid"])
    case = {"path": path, "graph": graph}
    # upper ends: tc and the BC paths do far more than one pass over the arcs
    top = {"bfs": 1 << 22, "bfs_many": 1 << 22, "sssp": 1 << 22, "cc": 1 << 22, "tc": 1 << 18, "bc": 1 << 18,
           "bc_batched": 1 << 18, "bfs_multi": 1 << 20}[path]
    n = _log_int(rng, 1 << 10, top)
    if graph == "grid":
        side = {"bfs": 2500, "bfs_many": 300, "sssp": 1200, "cc": 4000, "tc": 1000, "bc": 250, "bc_batched": 400,
                "bfs_multi": 700}[path]
        case["n"], case["cols"] = _log_int(rng, 32, side), _log_int(rng, 32, side)
        case["p_delete"] = rng.choice([0.0, 0.05, 0.15])
    else:
        case["n"], case["degree"] = n, rng.randint(4, 24)
        if path not in ("tc",) and rng.random() < 0.4:
            case["directed"] = True
    if rng.random() < 0.4:
        case["offset_bytes"] = 4
    if path in ("bfs", "bfs_many"):
        case["policy"] = rng.choice(["push", "hybrid", "hybrid", "learned"])
    if path == "sssp":
        case["weights"] = rng.choice(["u32", "u32", "f32"])
    if path in ("bfs_many", "bc"):
        case["sources"] = rng.randint(1, 8)
    if path in ("bc_batched", "bfs_multi"):
        case["sources"] = rng.choice([rng.randint(1, 64), 64, rng.randint(65, 100)])
    return case


# ------------------------------------------------------------------ graphs --
def _mix(x):
    """A 63-bit mix of int64 keys (Steele, Lea and Flood's splitmix64 finaliser, wrapping arithmetic)."""
    x = x + (0x9E3779B97F4A7C15 - (1 << 64))
    x = (x ^ ((x >> 30) & ((1 << 34) - 1))) * (0xBF58476D1CE4E5B9 - (1 << 64))
    x = (x ^ ((x >> 27) & ((1 << 37) - 1))) * (0x94D049BB133111EB - (1 << 64))
    return (x ^ ((x >> 31) & ((1 << 33) - 1))) & ((1 << 63) - 1)


def _endpoints(case, gen):
    if case["graph"] == "grid":
        rows, cols = case["n"], case["cols"]
        ids = torch.arange(rows * cols, device=DEV).view(rows, cols)
        u = torch.cat([ids[:, :-1].reshape(-1), ids[:-1, :].reshape(-1)])
        v = torch.cat([ids[:, 1:].reshape(-1), ids[1:, :].reshape(-1)])
        keep = torch.rand(u.numel(), device=DEV, generator=gen) >= case.get("p_delete", 0.0)
        return rows * cols, u[keep], v[keep]
    n, m = case["n"], case["n"] * case["degree"]
    if case["graph"] == "er":
        return n, *(torch.randint(0, n, (m,), device=DEV, generator=gen) for _ in range(2))
    u, v = (torch.zeros(m, device=DEV, dtype=torch.int32) for _ in range(2))
    for _ in range(max(1, (n - 1).bit_length())):
        r = torch.rand(m, device=DEV, generator=gen)
        u.mul_(2).add_(r >= 0.76)
        v.mul_(2).add_(((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
        del r
    perm = torch.randperm(n, device=DEV, generator=gen)
    return n, perm[u.remainder_(n)], perm[v.remainder_(n)]


def _csr(case, seed):
    """n, offsets int64[n + 1], cols int32[m] ascending per row, weights (int32, float32 or None), the generator."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed) * 1000003 + 17)
    n, u, v = _endpoints(case, gen)
    keep = u != v
    u, v = u[keep], v[keep]
    key = u * n + v if case.get("directed") else torch.cat([u * n + v, v * n + u])
    del u, v, keep
    key = torch.unique(key)
    offsets = torch.searchsorted(key, torch.arange(n + 1, device=DEV) * n)
    weights = None
    if case.get("weights"):
        u = torch.div(key, n, rounding_mode="floor")
        v = key - u * n
        h = _mix(torch.minimum(u, v) * n + torch.maximum(u, v) + int(seed) * 7919)
        del u, v
        if case["weights"] == "u32":
            weights = (h % 255 + 1).to(torch.int32)
        else:
            weights = ((h >> 39) + 1).to(torch.float32) / (1 << 24)
        del h
    cols = key.remainder_(n).to(torch.int32)
    return n, offsets, cols, weights, gen


def _sources(case, offsets, gen):
    """Vertices with at least one out-arc, as the Graph500 search keys."""
    ok = torch.nonzero(offsets[1:] > offsets[:-1]).view(-1)
    pick = torch.randint(0, ok.numel(), (case.get("sources", 1),), device=DEV, generator=gen)
    return ok[pick].tolist()


def _graph(case, n, offsets, cols, weights):
    global _device
    if _device is None:
        _device = sg.Device(0)
    ob = case.get("offset_bytes", 8)
    off = offsets if ob == 8 else offsets.to(torch.int32)
    flags = sg.GRAPH_INPUT_DEVICE | (sg.GRAPH_DIRECTED if case.get("directed") else 0)
    if weights is not None:
        flags |= sg.GRAPH_WEIGHTED | (sg.GRAPH_WEIGHT_FLOAT if weights.dtype == torch.float32 else 0)
    torch.cuda.synchronize()
    h = C.c_void_p()
    sg.check(sg.lib().sg_graph_create(_device.h, n, cols.numel(), off.data_ptr(), ob, cols.data_ptr(),
                                      None if weights is None else weights.data_ptr(), flags, C.byref(h)))
    return sg.Graph(_device, h)


class _Buffer:
    """A tensor where the framework takes a device buffer."""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, tensor.data_ptr()


def _learned():
    path = os.path.join(os.path.dirname(sg.__file__), "data", "bfs_policy.f32")
    return sg.Policy(_device, np.fromfile(path, dtype=np.float32))


def prepare(case, seed):
    n, offsets, cols, weights, gen = _csr(case, seed)
    g = _graph(case, n, offsets, cols, weights)
    path, srcs = case["path"], _sources(case, offsets, gen)
    del offsets, cols, weights
    s = {"path": path, "graph": g, "sources": srcs, "case": case}
    if path in ("bfs", "bfs_many"):
        g.prepare()  # the per-graph helpers, built once per loaded graph
        s["learned"] = _learned() if case["policy"] == "learned" else None
    rows = len(srcs) if path in ("bfs_many", "bfs_multi") else 1
    kind = torch.float32 if path.startswith("bc") or case.get("weights") == "f32" else torch.int64 if path == "tc" else torch.int32
    s["out"] = torch.empty((rows, n) if rows > 1 else (n,), device=DEV, dtype=kind)
    buf = s["buffer"] = _Buffer(s["out"])
    if path == "bfs":
        s["algorithm"] = sg.BFS(g)
        s["algorithm"].depth = buf
    elif path == "sssp":
        s["algorithm"] = sg.SSSP(g)
        s["algorithm"].dist = buf
    elif path == "cc":
        s["algorithm"] = sg.CC(g)
        s["algorithm"].labels = buf
    elif path.startswith("bc"):
        s["algorithm"] = sg.BC(g)
        s["algorithm"].sources, s["algorithm"].values = srcs, buf
    elif path == "bfs_multi":
        s["source_array"] = np.asarray(srcs, dtype=np.int32)
    torch.cuda.synchronize()
    return s


# --------------------------------------------------------------------- run --
def run(s):
    path, case, out = s["path"], s["case"], s["out"]
    if path == "bfs":
        b = s["algorithm"]
        b.init(s["sources"][0])
        st = b.run(POLICY[case["policy"]], 15.0, 24.0, learned=s["learned"], record_levels=case.get("levels", False))
        return {"depth": out, "vertices": st.reached_vertices, "edges": st.reached_edges}
    if path == "bfs_many":
        st = sg.bfs_many(s["graph"], s["sources"], POLICY[case["policy"]], 15.0, 24.0, out=s["buffer"],
                         learned=s["learned"])
        return {"depth": out, "vertices": st.reached_vertices, "edges": st.reached_edges}
    if path == "sssp":
        a = s["algorithm"]
        a.init(s["sources"][0])
        st = a.run()
        return {"dist": out, "vertices": st.reached_vertices, "edges": st.reached_edges}
    if path == "cc":
        s["algorithm"].run()
        return {"labels": out}
    if path == "tc":
        count = C.c_uint64()
        sg.check(sg.lib().sg_tc(s["graph"].h, C.byref(count), s["buffer"].ptr))
        return {"count": int(count.value), "per_vertex": out}
    if path in ("bc", "bc_batched"):
        sg.check(sg.lib().sg_fill(_device.h, s["buffer"].ptr, 0, 4, out.numel()))
        s["algorithm"].run(batched=path == "bc_batched")
        return {"bc": out}
    src = s["source_array"]
    sg.check(sg.lib().sg_bfs_multi_ex(s["graph"].h, len(src), src.ctypes.data_as(C.c_void_p), None, s["buffer"].ptr))
    return {"depth": out}


def work(case):
    """The CSR (and weights) read once, the answer written once."""
    if case["graph"] == "grid":
        n = case["n"] * case["cols"]
        m = 4 * n * (1 - case.get("p_delete", 0.0))
    else:
        n = case["n"]
        m = n * case["degree"] * (1 if case.get("directed") else 2)
    rows = case.get("sources", 1) if case["path"] in ("bfs_many", "bfs_multi") else 1
    bytes_ = n * case.get("offset_bytes", 8) + m * (8 if case.get("weights") else 4)
    return {"bytes": bytes_ + rows * n * (8 if case["path"] == "tc" else 4), "flops": 0}


def tolerance(case):
    if case["path"] == "bc":  # FP64 sums, rounded to float once: 3e-8 against 64 bits
        return {"rel": 1.5e-7, "max": 5e-7}
    if case["path"] == "bc_batched":  # FP32 path counts and dependencies: 1e-7 against 64 bits
        return {"rel": 1e-6, "max": 2e-5}
    # whole numbers; and FP32 distances, which are sums along a path from the
    # source outwards: rounding is monotone, so every schedule ends at the same bits
    return "exact"


# ------------------------------------------------------- the answers, plainly --
def _expand(offsets, front):
    """Positions of the arcs of the vertices `front`, and the index into `front` of each."""
    b = offsets[front]
    d = offsets[front + 1] - b
    ends = torch.cumsum(d, 0)
    idx = torch.repeat_interleave(torch.arange(front.numel(), device=DEV), d)
    return torch.arange(idx.numel(), device=DEV) + (b - ends + d)[idx], idx


def _marked(flag, some):
    """The distinct vertices among `some`, whose flags are set meanwhile."""
    if some.numel() < 1 << 18:
        return torch.unique(some)
    flag[some] = True
    got = torch.nonzero(flag).view(-1)
    flag[got] = False
    return got


def _hops(n, offsets, cols, source):
    depth = torch.full((n,), n + 1, device=DEV, dtype=torch.int64)
    flag = torch.zeros(n, device=DEV, dtype=torch.bool)
    front = torch.tensor([source], device=DEV)
    depth[source] = 0
    levels = [front]
    while True:
        pos, _ = _expand(offsets, front)
        v = cols[pos].long()
        v = v[depth[v] == n + 1]
        if not v.numel():
            return depth, levels
        front = _marked(flag, v)
        depth[front] = len(levels)
        levels.append(front)


def _distances(n, offsets, cols, weights, source):
    far = torch.iinfo(torch.int64).max if weights.dtype == torch.int64 else float("inf")
    dist = torch.full((n,), far, device=DEV, dtype=weights.dtype)
    flag = torch.zeros(n, device=DEV, dtype=torch.bool)
    front = torch.tensor([source], device=DEV)
    dist[source] = 0
    while front.numel():
        changed = []
        for part in torch.split(front, 1 << 22):
            pos, idx = _expand(offsets, part)
            v = cols[pos].long()
            d = dist[part][idx] + weights[pos]
            better = d < dist[v]
            v, d = v[better], d[better]
            dist.scatter_reduce_(0, v, d, "amin")
            changed.append(v)
        front = _marked(flag, torch.cat(changed))
    unreached = dist == far
    dist[unreached] = n + 1
    return dist, ~unreached


def _labels(n, offsets, cols):
    label = torch.arange(n, device=DEV)
    src = torch.repeat_interleave(torch.arange(n, device=DEV), offsets[1:] - offsets[:-1])
    dst = cols.long()
    while True:
        old = label.clone()
        label.scatter_reduce_(0, dst, old[src], "amax")  # the largest id that reaches a vertex
        while True:  # ... and what reaches that one reaches it
            jump = torch.maximum(label, label[label])
            if torch.equal(jump, label):
                break
            label = jump
        if torch.equal(label, old):
            return label


def _triangles(n, offsets, cols):
    degree = offsets[1:] - offsets[:-1]
    u = torch.repeat_interleave(torch.arange(n, device=DEV), degree)
    v = cols.long()
    keep = (degree[u] < degree[v]) | ((degree[u] == degree[v]) & (u < v))
    u, v = u[keep], v[keep]
    key = u * n + v  # ascending: rows in order, ids ascending in a row
    off = torch.searchsorted(key, torch.arange(n + 1, device=DEV) * n)
    length = off[v + 1] - off[v]
    ends = torch.cumsum(length, 0)
    if key.numel() and int(ends[-1]) > 8_000_000_000:
        return None
    per = torch.zeros(n, device=DEV, dtype=torch.int64)
    a = 0
    while a < key.numel():
        base = int(ends[a] - length[a])
        z = max(a + 1, int(torch.searchsorted(ends, base + (1 << 27), right=True)))
        pos, idx = _expand(off, v[a:z])
        want = u[a:z][idx] * n + v[pos]
        at = torch.searchsorted(key, want).clamp_(max=key.numel() - 1)
        per += torch.bincount(u[a:z][idx[key[at] == want]], minlength=n)
        a = z
    return per


def _dependencies(n, offsets, cols, source, total):
    """Brandes' accumulation, each level's path counts scaled to at most one."""
    depth, levels = _hops(n, offsets, cols, source)
    sigma = torch.zeros(n, device=DEV, dtype=torch.float64)
    delta = torch.zeros(n, device=DEV, dtype=torch.float64)
    sigma[source] = 1.0
    scale = [1.0]
    arcs = []
    for k, front in enumerate(levels[:-1]):
        pos, idx = _expand(offsets, front)
        v = cols[pos].long()
        down = depth[v] == k + 1
        u, v = front[idx[down]], v[down]
        sigma.index_add_(0, v, sigma[u])
        top = 2.0 ** -math.frexp(float(sigma[levels[k + 1]].max()))[1]
        sigma[levels[k + 1]] *= top
        scale.append(top)
        arcs.append((u, v))
    for k in range(len(levels) - 2, -1, -1):
        u, v = arcs[k]
        delta.index_add_(0, u, sigma[u] * (1.0 + delta[v]) / sigma[v] * scale[k + 1])
    delta[source] = 0.0
    total += delta


def exact(case, seed):
    n, offsets, cols, weights, gen = _csr(case, seed)
    path, srcs = case["path"], _sources(case, offsets, gen)
    if path in ("bfs", "bfs_many", "bfs_multi"):
        degree = offsets[1:] - offsets[:-1]
        rows, vertices, edges = [], 0, 0
        for s in srcs:
            depth, levels = _hops(n, offsets, cols, s)
            reached = depth <= n
            vertices += int(reached.sum())
            edges += int(degree[reached].sum())
            rows.append(depth.to(torch.int32))
        depth = torch.stack(rows) if len(rows) > 1 else rows[0]
        return {"depth": depth} if path == "bfs_multi" else {"depth": depth, "vertices": vertices, "edges": edges}
    if path == "sssp":
        wide = weights.to(torch.float64 if weights.dtype == torch.float32 else torch.int64)
        dist, reached = _distances(n, offsets, cols, wide, srcs[0])
        return {"dist": dist, "vertices": int(reached.sum()), "edges": int((offsets[1:] - offsets[:-1])[reached].sum())}
    if path == "cc":
        return {"labels": _labels(n, offsets, cols)}
    if path == "tc":
        per = _triangles(n, offsets, cols)
        return None if per is None else {"count": int(per.sum()), "per_vertex": per}
    total = torch.zeros(n, device=DEV, dtype=torch.float64)
    for s in srcs:
        _dependencies(n, offsets, cols, s, total)
    return {"bc": total}
