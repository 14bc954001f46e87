"""Single-source min-plus from a source whose out-edges weigh INT32_MAX: such an
edge reaches nothing, its head is unreached unless another path leads there,
and the traversal ends.  Every policy, with and without distance thresholds,
heads of few and of many out-edges.  Bit-exact against the oracle."""
import numpy as np
import pytest

from conftest import dawn

pytestmark = pytest.mark.gpu
POLICIES = ("fixed", "learned", "push", "pull", "bitmap")
MAX = np.iinfo(np.int32).max


def check(orc, g, h, s):
    want = orc.dijkstra(h.row_ptr, h.col, h.weight, s, overflow_ok=True)
    assert (want[h.col[h.row_ptr[s]:h.row_ptr[s + 1]]] == dawn.INF).any()  # an unreached neighbour
    for p in POLICIES:
        d, st = g.sssp(s, policy=p, stats=True)
        assert np.array_equal(d, want), p
        assert st["vertices_reached"] == (want != dawn.INF).sum(), p


@pytest.mark.parametrize("directed", [False, True])
def test_one_edge(orc, directed):
    print(f"case: two vertices, an edge of weight INT32_MAX, directed={directed}", flush=True)
    h = dawn.HostGraph.from_edges(2, np.array([0], np.int32), np.array([1], np.int32), np.array([MAX], np.int32),
                                  symmetrize=not directed)
    check(orc, dawn.Graph(h), h, 0)


@pytest.mark.parametrize("n,hub", [(40, False), (3000, False), (3000, True), (70_000, False), (70_000, True)])
def test_seeds(orc, n, hub):
    """Half of the source's out-edges weigh INT32_MAX (of the others a tenth);
    some of their heads have hundreds of out-edges."""
    print(f"case: directed, {n} vertices, hubs {hub}", flush=True)
    rng = np.random.default_rng(n)
    deg = rng.integers(1, 5, n)
    deg[0] = min(n // 8, 600 if hub else 16)
    if hub:
        deg[rng.integers(1, n, 20)] = 300
    u = np.repeat(np.arange(n), deg)
    # Heads in the upper half of the ids are reached from the source alone.
    v = np.where(u == 0, rng.integers(1, n, len(u)), rng.integers(0, n // 2, len(u)))
    w = np.where(rng.random(len(u)) < np.where(u == 0, 0.5, 0.1), MAX, rng.integers(0, 900, len(u)))
    h = dawn.HostGraph.from_edges(n, u.astype(np.int32), v.astype(np.int32), w.astype(np.int32), symmetrize=False)
    g = dawn.Graph(h)
    check(orc, g, h, 0)
    g.close()
