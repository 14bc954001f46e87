"""Weighted lanes, pulled steps of wide records: fewer vertices than one wave
takes, as many as every wave one pair, 64 a wave and more than the launch has
waves for; last vertices without in-edges, odd numbers of improved vertices, hubs
(32 lanes take wide records only with them); rows against the oracle."""
import numpy as np
import pytest

from conftest import dawn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 63, 65, 1001, 32_768, 32_769, 262_143, 262_145, 600_007])
@pytest.mark.parametrize("hubs", [False, True])
@pytest.mark.parametrize("count", [20, 33, 64])
def test_wide_pull(orc, n, hubs, count):
    print(f"case: directed weighted graph, {n} vertices, hubs {hubs}, {count} sources", flush=True)
    rng = np.random.default_rng(n + count)
    heads = max(1, n * 3 // 4)  # the others have no in-edges
    u, v = rng.integers(0, n, 3 * n), rng.integers(0, heads, 3 * n)
    if hubs:  # n / 64 in-edge chunks and more
        k = max(1, heads // 128)
        u = np.concatenate([u, rng.integers(0, n, 160 * k)])
        v = np.concatenate([v, np.repeat(np.arange(k) * (heads // k), 160)])
    h = dawn.HostGraph.from_edges(n, u.astype(np.int32), v.astype(np.int32),
                                  rng.integers(1, 1000, len(u)).astype(np.int32), symmetrize=False)
    g = dawn.Graph(h)
    if hubs:
        g.set_knobs(heavy_degree=32, pull_chunk=64)
    src = rng.integers(0, n, count).astype(np.int32)
    some = [0, 1, count - 1]
    want, wsums, _, _ = orc.mssp(h.row_ptr, h.col, h.weight, src[some])
    for p in ("pull", "fixed"):
        dist, sums = g.mssp(src, policy=p)
        assert np.array_equal(dist[some], want) and np.array_equal(sums[some], wsums), p
    g.close()
