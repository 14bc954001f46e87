"""Uneven batch, weighted tasks with their state in LDS: distances there, or
bounds there and distances in memory (sizes on both sides of each limit, and
beyond both), bounds that are moved along long paths and across a gap wider
than their range, zero weights, weights whose paths overflow, hubs, short
lists, vertices without out-edges.  Every row against the oracle."""
import numpy as np
import pytest

from conftest import dawn

pytestmark = pytest.mark.gpu


def check(orc, h, src):
    g = dawn.Graph(h)
    rows, _ = dawn.batch_mssp([g], np.asarray(src, np.int32), len(src))
    for j, s in enumerate(src):
        if h.row_ptr[s] == h.row_ptr[s + 1]:
            ref = np.full(h.n, dawn.INF, np.int32)
            ref[s] = 0
        else:
            ref = orc.sssp(h.row_ptr, h.col, h.weight, s, dense=False, overflow_ok=True)
        assert np.array_equal(rows[0][j], ref), s
    g.close()


def random_edges(n, m, seed):
    rng = np.random.default_rng(seed)
    return rng, rng.integers(0, n, m).astype(np.int32), rng.integers(0, n, m).astype(np.int32)


# 37,797 vertices have their distances in LDS, 134,000 their bounds.
@pytest.mark.parametrize("n", [2, 3, 33, 1024, 4097, 37_796, 37_797, 37_798, 133_999, 134_000, 134_001])
@pytest.mark.parametrize("degree", [3, 14])
def test_sizes(orc, n, degree):
    print(f"case: {n} vertices, {n * degree} directed edges, 2 sources", flush=True)
    rng, u, v = random_edges(n, n * degree, n + degree)
    w = rng.integers(0, 1000, len(u)).astype(np.int32)
    check(orc, dawn.HostGraph.from_edges(n, u, v, w, symmetrize=False), [0, n - 1])


@pytest.mark.parametrize("n", [20_000, 45_000])
def test_weight_ranges(orc, n):
    """Zero weights; weights whose sums overflow; a few heavy edges (delta far
    above the other weights); INT32_MAX itself."""
    rng, u, v = random_edges(n, 9 * n, n)
    for name, w in (("0 to 2", rng.integers(0, 3, len(u))), ("all 0", np.zeros(len(u))),
                    ("overflow", rng.integers(1 << 28, (1 << 31) - 1, len(u))),
                    ("skewed", np.where(rng.random(len(u)) < 0.01, 1 << 24, 1 + rng.integers(0, 5, len(u)))),
                    ("largest", np.where(rng.random(len(u)) < 0.5, (1 << 31) - 1, 7))):
        print(f"case: {n} vertices, weights {name}", flush=True)
        check(orc, dawn.HostGraph.from_edges(n, u, v, w.astype(np.int32)), [1, n // 2])


def test_long_distances(orc):
    """A grid of 230 x 230 whose distances span several hundred mean weights;
    two random graphs joined by one edge beyond the range of the bounds."""
    print("case: grid 230, 2 sources", flush=True)
    check(orc, dawn.HostGraph.grid(230, 0.0, 5, weighted=True), [0, 230 * 115 + 115])
    for degree in (4, 12):
        print(f"case: two random graphs of 21,000 vertices, degree {degree}, far apart", flush=True)
        rng, u, v = random_edges(21_000, 21_000 * degree // 2, degree)
        w = rng.integers(1, 10, len(u))
        h = dawn.HostGraph.from_edges(42_000, np.concatenate([u, u + 21_000, [5]]).astype(np.int32),
                                      np.concatenate([v, v + 21_000, [21_005]]).astype(np.int32),
                                      np.concatenate([w, w, [100_000]]).astype(np.int32))
        check(orc, h, [5, 30_000])


@pytest.mark.parametrize("leaves", [10_000, 60_000])
def test_hubs(orc, leaves):
    print(f"case: RMAT-12 and a star of {leaves} leaves on one vertex", flush=True)
    r = dawn.HostGraph.rmat(12, 16, 6, weighted=True)
    ru = np.repeat(np.arange(r.n, dtype=np.int32), r.degrees())
    leaf = np.arange(r.n, r.n + leaves, dtype=np.int32)
    u, v = np.concatenate([ru, np.full(leaves, 7, np.int32)]), np.concatenate([r.col, leaf])
    w = np.concatenate([r.weight, (leaf % 977).astype(np.int32)])
    check(orc, dawn.HostGraph.from_edges(r.n + leaves, u, v, w), [7, r.n + 3])


def test_mixed_batch(orc):
    """Weighted and unweighted graphs of every state in one batch."""
    print("case: 6 graphs, weighted and not, in LDS and in memory, 3 sources each", flush=True)
    hosts = [dawn.HostGraph.grid(60, 0.01, 1, weighted=True), dawn.HostGraph.er(2_000, 9.0, 2),
             dawn.HostGraph.er(45_000, 6.0, 3, weighted=True), dawn.HostGraph.rmat(12, 16, 4),
             dawn.HostGraph.er(140_000, 3.0, 5, weighted=True), dawn.HostGraph.er(1_220_000, 2.0, 6)]
    graphs = [dawn.Graph(h) for h in hosts]
    src = np.concatenate([np.flatnonzero(h.degrees() > 0)[[0, 7, -1]] for h in hosts]).astype(np.int32)
    rows, _ = dawn.batch_mssp(graphs, src, 3)
    for i, h in enumerate(hosts):
        want = orc.mssp(h.row_ptr, h.col, h.weight if h.weighted else None, src[3 * i:3 * i + 3])[0]
        for j in range(3):
            assert np.array_equal(rows[i][j], want[j]), (i, j)
        graphs[i].close()
