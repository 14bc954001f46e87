"""Edges of the single-source step kernels: out-degrees around the heavy-chunk
length, hubs, more discoveries in a step than a workgroup stages, duplicate
out-edges of the source.  Bit-exact against the oracle or the closed form."""
import numpy as np
import pytest

from conftest import dawn

pytestmark = pytest.mark.gpu
POLICIES = ("fixed", "push", "pull", "bitmap")


def log(msg):
    print(msg, flush=True)


def fan(first, leaves):
    """Vertices 1..k of out-degree leaves[i] + 1 behind source 0 (and back)."""
    k = len(leaves)
    u = [np.zeros(k, np.int64)]
    v = [np.arange(1, k + 1)]
    at = k + 1
    for i, c in enumerate(leaves):
        u.append(np.full(c, i + 1))
        v.append(np.arange(at, at + c))
        at += c
    n = at + first
    if first:  # leaves of the source itself
        u.append(np.zeros(first, np.int64))
        v.append(np.arange(at, at + first))
    return n, np.concatenate(u).astype(np.int32), np.concatenate(v).astype(np.int32)


@pytest.mark.parametrize("first,leaves", [
    (0, [126, 127, 128, 129, 255, 256, 257]),       # around one and two 128-edge chunks
    (124, [1, 0, 1100, 1023, 1024, 1025]),          # source of exactly 130; 8 and 9 chunks
    (70000, [0, 1, 2, 3, 200000, 64, 65, 63] * 2),  # hubs of hundreds of chunks
])
def test_heavy_chunks_exact(orc, first, leaves):
    log(f"case: fan of {len(leaves)} vertices, largest {max(leaves)}, source leaves {first}")
    n, u, v = fan(first, leaves)
    w = np.random.default_rng(n).integers(0, 1000, len(u)).astype(np.int32)
    h, hw = dawn.HostGraph.from_edges(n, u, v), dawn.HostGraph.from_edges(n, u, v, w)
    g, gw = dawn.Graph(h), dawn.Graph(hw)
    for s in (0, 1, len(leaves), n - 1):
        ref, refw = orc.bfs(h.row_ptr, h.col, s), orc.sssp(hw.row_ptr, hw.col, hw.weight, s)
        for p in POLICIES:
            d, st = g.bfs(s, policy=p, stats=True)
            assert np.array_equal(d, ref), (s, p)
            assert st["vertices_reached"] == n and st["edges_reached"] == h.m, (s, p)
            assert np.array_equal(gw.sssp(s, policy=p), refw), (s, p)
        assert np.array_equal(g.bfs_noalloc(s, policy="push"), ref), s


def test_more_found_than_a_workgroup_stages():
    # 60,000 children of the root with 100 leaves each: about 11,700 vertices
    # found per workgroup in the last step, more than it stages.
    log("case: two-level tree, 60,000 x 100 leaves, forced push")
    n, u, v = fan(0, [100] * 60000)
    h = dawn.HostGraph.from_edges(n, u, v)
    g = dawn.Graph(h)
    want = np.full(n, 2, np.int32)
    want[1:60001] = 1
    want[0] = 0
    for p in ("push", "bitmap"):
        d, st = g.bfs(0, policy=p, stats=True)
        assert np.array_equal(d, want), p
        assert st["vertices_reached"] == n and st["edges_reached"] == h.m, p


@pytest.mark.parametrize("policy", POLICIES)
def test_source_lists_its_edges_repeatedly(orc, policy):
    """The last listed duplicate of a source edge seeds the distance, also
    when the list is not sorted."""
    log(f"case: multigraph n=3000, source of 9000 unsorted duplicate edges, {policy}")
    rng = np.random.default_rng(12)
    n = 3000
    lists = [rng.integers(1, n, 9000)] + [rng.integers(0, n, int(rng.integers(0, 9))) for _ in range(n - 1)]
    rp = np.zeros(n + 1, np.int32)
    rp[1:] = np.cumsum([len(x) for x in lists])
    col = np.concatenate(lists).astype(np.int32)
    w = rng.integers(0, 500, len(col)).astype(np.int32)
    g = dawn.Graph(dawn.HostGraph.from_csr(rp, col, w, directed=True))
    assert np.array_equal(g.sssp(0, policy=policy), orc.sssp(rp, col, w, 0))


def chain_and_fans():
    """Chain, a fan of 3000 (a level of more edges than one workgroup walks),
    all joined again, a hub of 300 and a fan of 1500 behind another chain:
    levels change between small and large several times."""
    u, v, at = [], [], 0

    def link(a, b):
        u.append(a)
        v.append(b)
    for fan_of, chain in ((3000, 12), (300, 3), (1500, 40), (2048, 5), (2047, 1)):
        for _ in range(chain):
            link(at, at + 1)
            at += 1
        root, join = at, at + fan_of + 1
        for i in range(fan_of):
            link(root, root + 1 + i)
            link(root + 1 + i, join)
        at = join
    return at + 1, np.array(u, np.int32), np.array(v, np.int32)


@pytest.mark.parametrize("kind", ["path", "fans"])
def test_walks_of_small_levels_exact(orc, kind):
    """Runs of small levels are walked in one launch (at most 4096 levels of
    at most 2048 edges); every policy, both engines, and into a device buffer."""
    n, u, v = chain_and_fans() if kind == "fans" else (9001, np.arange(9000), np.arange(1, 9001))
    log(f"case: {kind}, n={n}")
    w = np.random.default_rng(5).integers(0, 50, len(u)).astype(np.int32)
    h, hw = dawn.HostGraph.from_edges(n, u, v), dawn.HostGraph.from_edges(n, u, v, w)
    g, gw = dawn.Graph(h), dawn.Graph(hw)
    for s in (0, 13, n // 2, n - 1):
        ref, refw = orc.bfs(h.row_ptr, h.col, s), orc.sssp(hw.row_ptr, hw.col, hw.weight, s)
        for p in ("fixed", "push") + (("pull", "bitmap") if kind == "fans" else ()):
            d, st = g.bfs(s, policy=p, stats=True)
            assert np.array_equal(d, ref), (s, p)
            assert st["vertices_reached"] == n and st["edges_reached"] == h.m, (s, p)
            assert st["steps"] == ref.max() + 1, (s, p)  # the last one finds nothing
            dw, st = gw.sssp(s, policy=p, stats=True)
            assert np.array_equal(dw, refw), (s, p)
            assert st["vertices_reached"] == n and st["edges_reached"] == hw.m, (s, p)
        out = dawn.DeviceArray(n + 1, np.int32)  # rows at any int32 offset
        for off in (0, 4):
            p = out.data_ptr() + off
            assert dawn.lib().dawn_bfs(g.handle, s, p, 0, None) == 0
            got = out.download()[off // 4:][:n]
            assert np.array_equal(got, ref), (s, off)
        assert np.array_equal(g.bfs_noalloc(s), ref), s


@pytest.mark.parametrize("n,deg,wmax", [(1500, 3, 1), (5000, 4, 2), (30000, 12, 100000), (200000, 4, 1000)])
def test_minplus_thresholds_exact(orc, n, deg, wmax):
    """Distance thresholds (graphs without hubs): unit and tiny weights (an
    advance of one), large ones, weights of zero, a few far heavier than the
    mean, and vertices held back over many steps; all policies."""
    log(f"case: random directed graph n={n} degree {deg}, weights up to {wmax}, every 50th 200 times that")
    rng = np.random.default_rng(n)
    m = n * deg
    u, v = rng.integers(0, n, m).astype(np.int32), rng.integers(0, n, m).astype(np.int32)
    w = rng.integers(0, wmax + 1, m).astype(np.int32)
    w[::50] *= 200
    h = dawn.HostGraph.from_edges(n, u, v, w, symmetrize=False)
    g = dawn.Graph(h)
    for s in np.flatnonzero(h.degrees() > 0)[[0, n // 3]]:
        ref = orc.sssp(h.row_ptr, h.col, h.weight, int(s))
        for p in POLICIES:
            d, st = g.sssp(int(s), policy=p, stats=True)
            assert np.array_equal(d, ref), (s, p)
            reached = ref != dawn.INF
            assert st["vertices_reached"] == reached.sum(), (s, p)
            assert st["edges_reached"] == h.degrees()[reached].sum(), (s, p)
