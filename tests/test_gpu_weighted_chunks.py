"""Weighted lanes, vertices expanded by out-edge chunks: fewer chunks than waves,
more than 64 for every wave of the launch, several per vertex; rows against the
oracle."""
import numpy as np
import pytest

from conftest import dawn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,degree,knobs", [
    (700, 40, {"heavy_degree": 32, "pull_chunk": 16}),       # a few thousand chunks, several a vertex
    (3000, 50, {"heavy_degree": 33}),                        # one a vertex
    (300_000, 4, {"heavy_degree": 1, "pull_chunk": 64})])    # one for every vertex
@pytest.mark.parametrize("count", [3, 33])
def test_push_by_chunks(orc, n, degree, knobs, count):
    print(f"case: weighted random graph, {n} vertices, degree {degree}, {count} sources, {knobs}", flush=True)
    h = dawn.HostGraph.er(n, float(degree), 5, weighted=True)
    g = dawn.Graph(h)
    g.set_knobs(**knobs)
    src = np.random.default_rng(count).integers(0, n, count).astype(np.int32)
    some = [0, 1, count - 1]
    want, wsums, _, _ = orc.mssp(h.row_ptr, h.col, h.weight, src[some])
    for p in ("push", "fixed"):
        dist, sums = g.mssp(src, policy=p)
        assert np.array_equal(dist[some], want) and np.array_equal(sums[some], wsums), p
    g.close()
