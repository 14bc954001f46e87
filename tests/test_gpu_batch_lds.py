"""Uneven batch, unweighted tasks with their state in LDS: lanes per task from
1 to 16, levels staged in LDS and in memory and beyond a byte, pulled and
pushed lanes in one level, in-edges of directed graphs, hubs beyond 16-bit
degrees, and graphs too large for the LDS.  Every row against the oracle."""
import numpy as np
import pytest

from conftest import dawn

pytestmark = pytest.mark.gpu


def check(orc, hosts, spg, seed):
    graphs = [dawn.Graph(h) for h in hosts]
    rng = np.random.default_rng(seed)
    src = np.concatenate([rng.integers(0, h.n, spg) for h in hosts]).astype(np.int32)
    rows, st = dawn.batch_mssp(graphs, src, spg)
    for i, h in enumerate(hosts):
        for j in range(spg):
            s = int(src[i * spg + j])
            if h.row_ptr[s] == h.row_ptr[s + 1]:
                ref = np.full(h.n, dawn.INF, np.int32)
                ref[s] = 0
            else:
                ref = orc.bfs(h.row_ptr, h.col, s)
            assert np.array_equal(rows[i][j], ref), (i, j, s)
    for g in graphs:
        g.close()
    return st


def directed(n, m, seed):
    rng = np.random.default_rng(seed)
    u, v = rng.integers(0, n, m).astype(np.int32), rng.integers(0, n, m).astype(np.int32)
    return dawn.HostGraph.from_edges(n, u, v, symmetrize=False)


@pytest.mark.parametrize("spg", [1, 2, 3, 5, 8, 16, 17, 33])
def test_lane_counts(orc, spg):
    print(f"case: RMAT-12, ER 3000, grid 40, directed 2500, {spg} sources each", flush=True)
    hosts = [dawn.HostGraph.rmat(12, 16, 61), dawn.HostGraph.er(3000, 20.0, 62),
             dawn.HostGraph.grid(40, 0.01, 63), directed(2500, 30000, 64)]
    check(orc, hosts, spg, spg)


def test_sizes_around_the_lds(orc):
    # One lane: 116,000 vertices have their levels in LDS, 151,000 do not,
    # 1,209,600 fields just fit, one more vertex does not.
    print("case: grids and random graphs of 57,600 to 1,212,201 vertices, 2 sources each", flush=True)
    hosts = [dawn.HostGraph.er(115_999, 5.0, 71), dawn.HostGraph.er(135_000, 5.0, 72),
             dawn.HostGraph.grid(240, 0.01, 73), dawn.HostGraph.grid(389, 0.01, 74),
             dawn.HostGraph.er(1_209_600, 3.0, 75), dawn.HostGraph.grid(1101, 0.01, 76)]
    check(orc, hosts, 2, 7)


def test_hub_degrees_and_long_paths(orc):
    """A star of 70,000 leaves (degrees beyond 16 bits), RMAT-15 with lanes
    that start in a far chain (few frontier edges beside many), a path of
    3000 (levels beyond a byte)."""
    print("case: star 70,000, RMAT-15 + chain, path 3000, 6 sources", flush=True)
    star = dawn.HostGraph.from_edges(70001, np.zeros(70000, np.int32), np.arange(1, 70001, dtype=np.int32))
    r = dawn.HostGraph.rmat(15, 16, 81)
    ru = np.repeat(np.arange(r.n, dtype=np.int32), r.degrees())
    chain = np.arange(r.n, r.n + 40000, dtype=np.int32)
    u = np.concatenate([ru, [0], chain[:-1]]).astype(np.int32)
    v = np.concatenate([r.col, [r.n], chain[1:]]).astype(np.int32)
    tail = dawn.HostGraph.from_edges(r.n + 40000, u, v)
    p = np.arange(3000, dtype=np.int32)
    path = dawn.HostGraph.from_edges(3001, p, p + 1)
    check(orc, [star, tail, path], 6, 9)
