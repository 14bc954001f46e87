"""Weighted sources a workgroup each: the rule's two sides in sources and
edges, rows on the device, on the host and none, more sources than a launch
holds, negative and repeated source ids; rows, sums and counts against the
oracle and against the engine of 64 lanes (a forced mode)."""
import numpy as np
import pytest

from conftest import dawn

pytestmark = pytest.mark.gpu


def device_rows(g, src, policy):
    out = dawn.DeviceArray((len(src), g.n), np.int32).fill_bytes(0x5A)
    _, sums, st = g.mssp(src, policy=policy, out=out, stats=True)
    return out.download(), sums, st


@pytest.mark.parametrize("n,degree", [(300, 4), (20_000, 10), (60_000, 8), (90_000, 40)])
@pytest.mark.parametrize("count", [1, 31, 32, 300])
def test_against_lanes(orc, n, degree, count):
    print(f"case: {n} vertices, degree {degree}, {count} sources", flush=True)
    g = dawn.Graph.er_device(n, degree, 17 + n, weighted=True)
    src = np.random.default_rng(n + count).integers(-n, 2 * n, count).astype(np.int32)
    src[0] = 0
    rows, sums, st = device_rows(g, src, "fixed")
    want, wsums, wst = device_rows(g, src, "push")
    assert np.array_equal(rows, want) and np.array_equal(sums, wsums)
    for f in ("vertices_reached", "edges_reached", "skipped_sources"):
        assert st[f] == wst[f], f
    g.close()


@pytest.mark.parametrize("n", [9_000, 50_000])
def test_host_rows_and_sums_only(orc, n):
    print(f"case: {n} vertices directed, 300 sources, host rows; sums alone", flush=True)
    rng = np.random.default_rng(n)
    u, v = rng.integers(0, n, 6 * n).astype(np.int32), rng.integers(0, n, 6 * n).astype(np.int32)
    h = dawn.HostGraph.from_edges(n, u, v, rng.integers(0, 50, 6 * n).astype(np.int32), symmetrize=False)
    g = dawn.Graph(h)
    src = rng.integers(0, n, 300).astype(np.int32)
    dist, sums = g.mssp(src)
    ref, rsums, _, _ = orc.mssp(h.row_ptr, h.col, h.weight, src[:6])
    assert np.array_equal(np.asarray(dist)[:6], ref) and np.array_equal(sums[:6], rsums)
    for i in (255, 256, 299):
        assert np.array_equal(dist[i], orc.mssp(h.row_ptr, h.col, h.weight, src[i:i + 1])[0][0]), i
    _, s2, _ = g.closeness(src)
    assert np.array_equal(s2, sums)
    g.close()


@pytest.mark.parametrize("n,degree", [(2, 1), (300, 4), (20_000, 10), (60_000, 12), (100_000, 3)])
@pytest.mark.parametrize("count", [1, 64, 257])
def test_unweighted_against_lanes(orc, n, degree, count):
    """Rows, sums and counts equal those of the engine of lanes (knobs set),
    with isolated, negative and repeated sources."""
    print(f"case: {n} vertices, degree {degree}, {count} sources", flush=True)
    rng = np.random.default_rng(n + count)
    u, v = (rng.integers(0, n, n * degree).astype(np.int32) for _ in range(2))
    h = dawn.HostGraph.from_edges(n, u, v, symmetrize=n % 3 != 0)
    g = dawn.Graph(h)
    src = rng.integers(-n, 2 * n, count).astype(np.int32)
    src[-1] = src[0]
    rows, sums, st = device_rows(g, src, "learned")
    hrows, hsums = g.mssp(src)
    _, csums, _ = g.closeness(src)
    g.set_knobs()
    want, wsums, wst = device_rows(g, src, "learned")
    assert np.array_equal(rows, want) and np.array_equal(hrows, want)
    assert all(np.array_equal(x, wsums) for x in (sums, hsums, csums))
    for f in ("vertices_reached", "edges_reached", "skipped_sources", "batches", "steps"):
        assert st[f] == wst[f], f
    g.close()


def test_unweighted_long_levels(orc):
    """Levels beyond a byte (rows, and sums without rows) on a path with a
    random graph at its end."""
    print("case: path of 5,000 vertices into a random graph, 40 sources", flush=True)
    rng = np.random.default_rng(3)
    p = np.arange(5_000, dtype=np.int32)
    u = np.concatenate([p, 5_000 + rng.integers(0, 4_000, 12_000)]).astype(np.int32)
    v = np.concatenate([p + 1, 5_000 + rng.integers(0, 4_000, 12_000)]).astype(np.int32)
    h = dawn.HostGraph.from_edges(9_000, u, v)
    g = dawn.Graph(h)
    src = np.concatenate([[0, 4_999, 5_000], rng.integers(0, 9_000, 37)]).astype(np.int32)
    odist, osums, _, _ = orc.mssp(h.row_ptr, h.col, None, src)
    dist, sums = g.mssp(src)
    assert np.array_equal(dist, odist) and np.array_equal(sums, osums)
    assert np.array_equal(g.closeness(src)[1], osums)
    g.close()


@pytest.mark.parametrize("count", [1, 8, 16, 20, 32, 40, 64, 70])
@pytest.mark.parametrize("kind", ["grid", "rmat", "directed"])
def test_weighted_lanes(orc, kind, count):
    """The engine of lanes (knobs set, and forced modes): every record width,
    light lists, heavy vertices by chunks, in-edges of a directed graph,
    zero weights, hub sources."""
    print(f"case: {kind}, {count} sources", flush=True)
    rng = np.random.default_rng(count)
    if kind == "grid":
        h = dawn.HostGraph.grid(70, 0.02, 3, weighted=True)
    elif kind == "rmat":
        h = dawn.HostGraph.rmat(12, 16, 4, weighted=True)
    else:
        u, v = rng.integers(0, 3001, 40_000) % rng.integers(1, 3001, 40_000), rng.integers(0, 3001, 40_000)
        h = dawn.HostGraph.from_edges(3001, u.astype(np.int32), v.astype(np.int32),
                                      rng.integers(0, 90, 40_000).astype(np.int32), symmetrize=False)
    g = dawn.Graph(h)
    g.set_knobs()
    src = rng.integers(0, h.n, count).astype(np.int32)
    src[0] = int(np.argmax(h.degrees()))
    odist, osums, _, _ = orc.mssp(h.row_ptr, h.col, h.weight, src)
    for p in ("fixed", "push", "pull"):
        dist, sums = g.mssp(src, policy=p)
        assert np.array_equal(dist, odist), p
        assert np.array_equal(sums, osums), p
    g.close()


@pytest.mark.parametrize("weighted", [False, True])
def test_more_sources_than_a_launch(orc, weighted):
    print(f"case: path of 5 vertices, 70,000 sources, weighted={weighted}", flush=True)
    u = np.arange(4, dtype=np.int32)
    h = dawn.HostGraph.from_edges(5, u, u + 1, np.array([3, 1, 4, 1], np.int32) if weighted else None)
    g = dawn.Graph(h)
    src = (np.arange(70_000) * 7 % 5).astype(np.int32)
    rows, sums, st = device_rows(g, src, "fixed")
    odist, osums, _, _ = orc.mssp(h.row_ptr, h.col, h.weight if weighted else None, np.arange(5, dtype=np.int32))
    assert np.array_equal(rows, odist[src]) and np.array_equal(sums, osums[src])
    assert st["vertices_reached"] == 5 * len(src)
    g.close()
