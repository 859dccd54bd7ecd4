"""Betweenness centrality and multi-source BFS on the MI355X through the C ABI.

BC results are compared with the FP64 oracle (itself pinned against networkx
for undirected and directed graphs) at relative tolerance 1e-5 of the FP64
value, the bound stated for BC; the float output rounds the FP64 total once,
so the observed error is ~6e-8 relative.  Known answers: the reference's
line_5 fixture (tests/algorithms/bc.cpp:9-15 runs BC from source 0 on it) and
star closed forms.
"""
import json
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(__file__), "golden")
RTOL = 1e-5


def _cases():
    with open(os.path.join(GOLDEN, "reference_cases.json")) as f:
        return json.load(f)


def _fixture(oracle_mod, name):
    return oracle_mod.from_dense(oracle_mod.parse_matrix_text(_cases()["matrices"][name]))


def _bc(sg, G, sources, batched=False):
    b = sg.BC(G)
    b.init(sources)
    b.run(batched=batched)
    return b.get_values()


def _close(got, ref):
    got = got.astype(np.float64)
    return np.all(np.abs(got - ref) <= RTOL * np.abs(ref) + 1e-6)


@pytest.mark.parametrize("batched", [False, True])
def test_bc_line5_known_answer(sg, device, oracle_mod, batched):
    g = _fixture(oracle_mod, "line_5")
    G = sg.Graph.from_csr(device, g.offsets, g.cols)
    assert _bc(sg, G, [0], batched).tolist() == _cases()["expect"]["bc_line_5_source0"]


@pytest.mark.parametrize("batched", [False, True])
def test_bc_star_closed_forms(sg, device, oracle_mod, batched):
    n = 9
    adj = np.zeros((n, n), dtype=np.int64)
    adj[0, 1:] = adj[1:, 0] = 1
    G = sg.Graph.from_csr(device, *_csr(oracle_mod.from_dense(adj)))
    assert np.all(_bc(sg, G, [0], batched) == 0.0)       # from the centre nothing passes through
    b = _bc(sg, G, [1], batched)                         # from a leaf the centre carries n-2 targets
    assert b[0] == n - 2 and np.all(b[1:] == 0.0)


def _csr(g):
    return g.offsets, g.cols


@pytest.mark.parametrize("batched", [False, True])
def test_bc_rmat14_golden(sg, device, oracle_mod, batched):
    z = np.load(os.path.join(GOLDEN, "rmat14_seed1.npz"))
    G = sg.Graph.rmat(device, 14, 16, seed=1)
    assert _close(_bc(sg, G, z["bc_sources"], batched), z["bc"])


@pytest.mark.parametrize("batched", [False, True])
def test_bc_matches_oracle_shapes(sg, device, oracle_mod, batched):
    rng = np.random.default_rng(11)
    for g in [oracle_mod.rmat(12, 16, seed=9), oracle_mod.grid(60, 45, 0.15, seed=8),
              oracle_mod.erdos_renyi(3000, 6000, seed=7)]:
        srcs = rng.integers(0, g.n, size=5).tolist()
        G = sg.Graph.from_csr(device, g.offsets, g.cols)
        assert _close(_bc(sg, G, srcs, batched), oracle_mod.bc(g, srcs))


@pytest.mark.parametrize("batched", [False, True])
def test_bc_long_diameter_grid_stays_finite(sg, device, oracle_mod, batched):
    # ~1e116 shortest paths to the far corner: sigma needs the per-level scaling
    g = oracle_mod.grid(200, 200)
    G = sg.Graph.from_csr(device, g.offsets, g.cols)
    b = _bc(sg, G, [0], batched)
    assert np.all(np.isfinite(b))
    assert _close(b, oracle_mod.bc(g, [0]))


@pytest.mark.parametrize("batched", [False, True])
def test_bc_directed(sg, device, oracle_mod, batched):
    rng = np.random.default_rng(5)
    n, m = 2000, 9000
    u, v = rng.integers(0, n, m), rng.integers(0, n, m)
    keep = u != v
    pairs = np.unique(np.stack([u[keep], v[keep]], 1), axis=0)
    off = np.zeros(n + 1, dtype=np.int64)
    np.cumsum(np.bincount(pairs[:, 0], minlength=n), out=off[1:])
    g = oracle_mod.CSRGraph(n, off, np.ascontiguousarray(pairs[:, 1], dtype=np.int32))
    G = sg.Graph.from_csr(device, g.offsets, g.cols, directed=True)
    srcs = [0, 3, 99, 1234]
    assert _close(_bc(sg, G, srcs, batched), oracle_mod.bc(g, srcs, inverse=oracle_mod.transpose(g)))


@pytest.mark.parametrize("batched", [False, True])
def test_bc_accumulates_and_isolated_source(sg, device, oracle_mod, batched):
    g = oracle_mod.grid(30, 30, 0.3, seed=2)
    G = sg.Graph.from_csr(device, g.offsets, g.cols)
    iso = int(np.flatnonzero(np.diff(g.offsets) == 0)[0])
    b = sg.BC(G)
    b.init([5, iso])
    b.run(batched=batched)
    b.run(batched=batched)  # a second run adds the same dependencies again
    assert _close(b.get_values(), 2.0 * oracle_mod.bc(g, [5, iso]))


@pytest.mark.parametrize("batched", [False, True])
def test_bc_invalid_source(sg, device, oracle_mod, batched):
    g = oracle_mod.rmat(8, 4, seed=1)
    G = sg.Graph.from_csr(device, g.offsets, g.cols)
    b = sg.BC(G)
    b.init([g.n])
    with pytest.raises(sg.SygraphError):
        b.run(batched=batched)


def test_bc_batched_many_sources_and_hubs(sg, device, oracle_mod):
    """Two lane batches (100 sources, repeats included), vertices whose lists
    span several work chunks (degrees above 256) and a star centre of degree
    599: the batched sums equal the per-source ones up to FP64 rounding."""
    rng = np.random.default_rng(23)
    g = oracle_mod.rmat(12, 16, seed=31)
    assert g.degrees().max() > 3 * 256
    srcs = rng.integers(0, g.n, size=98).tolist() + [int(np.argmax(g.degrees()))] * 2
    G = sg.Graph.from_csr(device, g.offsets, g.cols)
    ref = oracle_mod.bc(g, srcs)
    batched, single = _bc(sg, G, srcs, True), _bc(sg, G, srcs, False)
    assert _close(batched, ref) and _close(single, ref)
    n = 600
    adj = np.zeros((n, n), dtype=np.int64)
    adj[0, 1:] = adj[1:, 0] = 1
    G = sg.Graph.from_csr(device, *_csr(oracle_mod.from_dense(adj)))
    b = _bc(sg, G, list(range(1, 71)), True)
    assert b[0] == 70 * (n - 2) and np.all(b[1:] == 0.0)


def test_bfs_multi_matches_oracle(sg, device, oracle_mod):
    g = oracle_mod.rmat(12, 8, seed=13)
    G = sg.Graph.from_csr(device, g.offsets, g.cols)
    srcs = [0, 1, 77, int(np.argmax(g.degrees()))]
    d = sg.bfs_multi(G, srcs)
    for i, s in enumerate(srcs):
        assert np.array_equal(d[i], oracle_mod.bfs(g, s)[0])


@pytest.mark.parametrize("levels", [30, 200, 1500])
@pytest.mark.parametrize("directed", [False, True])
@pytest.mark.parametrize("batched", [False, True])
def test_bc_level_grouping_and_hubs(sg, device, oracle_mod, levels, directed, batched):
    """Level counts on each side of the level grouping's limits (64 levels with bitmaps written by the
    counting pass, 1,024 counted, more sorted), rungs of several shortest paths, and hubs of 700 arcs
    (a workgroup's share) in the middle and at the end.  Path counts grow like 1.6^level, so the batched
    form takes 30 levels without exponents, meets its limit of 2^100 at 200 and starts again with them;
    a second call on the same graph adds the same sums."""
    a = np.arange(levels - 1)
    u = np.concatenate([2 * a, 2 * a, 2 * a + 1, np.full(700, levels), np.full(700, 2 * levels - 1)])
    v = np.concatenate([2 * a + 2, 2 * a + 3, 2 * a + 2, 2 * levels + np.arange(700), 2 * levels + np.arange(700)])
    n = 2 * levels + 700
    if directed:
        key = np.unique(u.astype(np.int64) * n + v)
        off = np.zeros(n + 1, dtype=np.int64)
        np.add.at(off, key // n + 1, 1)
        g = oracle_mod.CSRGraph(n, np.cumsum(off), (key % n).astype(np.int32))
        ref = oracle_mod.bc(g, [0, 4], inverse=oracle_mod.transpose(g))
    else:
        g = oracle_mod.csr_from_pairs(n, u, v)
        ref = oracle_mod.bc(g, [0, 4])
    G = sg.Graph.from_csr(device, g.offsets, g.cols, directed=directed)
    b = sg.BC(G)
    b.init([0, 4])
    b.run(batched=batched)
    assert _close(b.get_values(), ref)
    b.run(batched=batched)
    assert _close(b.get_values(), 2.0 * ref)


def test_bc_of_a_long_path_keeps_little_memory(sg, device, oracle_mod):
    """30,000 levels: what the call keeps with the graph grows with the vertices, not with 8 KiB or a bitmap per
    level (245 and 112 MB here), and a second call gives the same sums."""
    import ctypes as C
    hip = C.CDLL("libamdhip64.so")

    other = sg.BFS(sg.Graph.from_csr(device, np.array([0, 1, 2]), np.array([1, 0])))

    def free_bytes():
        for _ in range(5):  # the runtime gives memory back with the commands after those that used it
            other.init(0)
            other.run(sg.POLICY_PUSH, 15.0, 24.0)
            other.get_distances()
        free, total = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    n = 30000
    g = oracle_mod.csr_from_pairs(n, np.arange(n - 1), np.arange(1, n))
    ref = oracle_mod.bc(g, [0, 7])
    G = sg.Graph.from_csr(device, g.offsets, g.cols)
    b = sg.BC(G)
    b.init([0, 7])
    b.run()
    assert _close(b.get_values(), ref)
    b.run()
    assert _close(b.get_values(), 2.0 * ref)
    held = free_bytes()
    G.destroy()
    assert free_bytes() - held < 64 << 20


@pytest.mark.parametrize("directed", [False, True])
@pytest.mark.parametrize("before,after", [(49, 3), (49, 60), (0, 70), (52, 0)])
def test_batched_bc_goes_on_with_exponents(sg, device, oracle_mod, directed, before, after):
    """Layers of four vertices, all joined to the next layer's: path counts grow fourfold a level and pass 2^100
    at the 51st, in lists laid end to end, or in lists of 300 (added up from chunks) where `before` such levels
    lie ahead of a layer of 300, or at the last level.  A first call, which meets the limit in its first batch
    and takes that level again with exponents, gives the bits of a second one, which has them from the start."""
    sizes = [1] + [4] * before + [300] + [4] * after + [1]
    first = np.concatenate([[0], np.cumsum(sizes)])
    u, v = [], []
    for k in range(len(sizes) - 1):
        a, b = np.meshgrid(first[k] + np.arange(sizes[k]), first[k + 1] + np.arange(sizes[k + 1]), indexing="ij")
        u.append(a.ravel())
        v.append(b.ravel())
    u, v, n = np.concatenate(u), np.concatenate(v), int(first[-1])
    if directed:
        off = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n))]).astype(np.int64)
        g = oracle_mod.CSRGraph(n, off, v[np.argsort(u, kind="stable")].astype(np.int32))
    else:
        g = oracle_mod.csr_from_pairs(n, u, v)
    srcs = np.concatenate([[0, 0, 1, n - 1], np.arange(70) % n])
    G = sg.Graph.from_csr(device, g.offsets, g.cols, directed=directed)
    got = []
    for _ in range(2):
        b = sg.BC(G)
        b.init(srcs)
        b.run(batched=True)
        got.append(b.get_values())
    assert _close(got[0], oracle_mod.bc(g, srcs.tolist(), **({"inverse": oracle_mod.transpose(g)} if directed else {})))
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    G.destroy()
