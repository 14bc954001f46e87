"""The batched engine's hub-first order built on the device: sizes around a
tile of its sort, all degrees equal, one vertex of nearly all edges, directed
graphs, rows longer than a wave; distances against the oracle."""
import numpy as np
import pytest

from conftest import dawn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65_536, 65_537, 69_633])
@pytest.mark.parametrize("kind", ["ring", "star", "directed"])
def test_hub_order(orc, n, kind):
    print(f"case: {kind}, {n} vertices, 70 sources", flush=True)
    rng = np.random.default_rng(n)
    ids = np.arange(n, dtype=np.int32)
    if kind == "ring":  # every degree 8
        steps = (1, 97, 5003, 20_011)
        u, v = np.tile(ids, len(steps)), np.concatenate([(ids + s) % n for s in steps])
    elif kind == "star":  # the last vertex joined to all, some random edges
        u = np.concatenate([np.full(n - 1, n - 1), rng.integers(0, n, n)])
        v = np.concatenate([ids[:-1], rng.integers(0, n, n)])
    else:  # out-degrees and in-degrees by different vertices
        u, v = n - 1 - (rng.random(9 * n) ** 6 * n).astype(np.int64), (rng.random(9 * n) ** 3 * n).astype(np.int64)
    h = dawn.HostGraph.from_edges(n, u.astype(np.int32), v.astype(np.int32), symmetrize=kind != "directed")
    g = dawn.Graph(h)
    g.set_knobs(hub_order=1)
    src = np.flatnonzero(h.degrees() > 0)[rng.integers(0, 1000, 70)].astype(np.int32)
    for p in ("fixed", "push", "pull"):
        dist, sums = g.mssp(src, policy=p)
        for i in (0, 1, 69):
            ref = orc.bfs(h.row_ptr, h.col, int(src[i]))
            assert np.array_equal(dist[i], ref), (p, i)
            assert sums[i] == int(ref[ref != dawn.INF].astype(np.int64).sum()), (p, i)
    g.close()
