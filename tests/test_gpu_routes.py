"""Which multi-source calls take a workgroup per source (no pulled steps) and
which the lanes: both sides of each limit in sources, vertices and edges, rows
against the oracle."""
import numpy as np
import pytest

from conftest import dawn

pytestmark = pytest.mark.gpu


def check(orc, g, h, count, workgroups):
    src = np.random.default_rng(count).integers(0, g.n, count).astype(np.int32)
    out = dawn.DeviceArray((count, g.n), np.int32).fill_bytes(0x5A)
    _, sums, st = g.mssp(src, policy="fixed", out=out, stats=True)
    assert (st["mode_steps"]["pull"] == 0) == workgroups, st["mode_steps"]
    rows, some = out.download(), sorted({0, 1, count // 2, count - 1} & set(range(count)))
    want, wsums, _, _ = orc.mssp(h.row_ptr, h.col, h.weight if g.weighted else None, src[some])
    assert np.array_equal(rows[some], want) and np.array_equal(sums[some], wsums)


# Distances in LDS up to 37,797 vertices (600,000 edges or 16 sources), with
# bounds there more than 64 sources.
@pytest.mark.parametrize("n,pairs,counts", [
    (37_797, 200_000, {1: True, 15: True}), (37_797, 330_000, {1: False, 15: False, 16: True, 65: True}),
    (37_798, 200_000, {16: False, 64: False, 65: True}), (134_000, 400_000, {64: False, 65: True}),
    (134_001, 400_000, {65: False, 200: False})])
def test_weighted(orc, n, pairs, counts):
    print(f"case: weighted random graph, {n} vertices, {pairs} pairs, sources {list(counts)}", flush=True)
    rng = np.random.default_rng(n)
    u, v = (rng.integers(0, n, pairs).astype(np.int32) for _ in range(2))
    h = dawn.HostGraph.from_edges(n, u, v, rng.integers(1, 1000, pairs).astype(np.int32))
    assert (h.m > 600_000) == (pairs > 300_000)
    g = dawn.Graph(h)
    for count, workgroups in counts.items():
        check(orc, g, h, count, workgroups)
    g.close()


@pytest.mark.parametrize("n,degree,counts", [
    (60_000, 16, {1: True, 256: True}),                          # one round of 256
    (60_000, 20, {1: False, 128: False, 129: True, 256: True}),  # few sources, no hubs, degree 17 to 28
    (54_000, 20, {1: True, 64: True}), (60_000, 32, {64: True}),
    (74_001, 10, {64: False, 200: True}), (74_001, 6, {64: True}),
    (80_001, 4, {64: False, 200: False}),                        # vertices
    (20_000, 8, {257: True, 1280: True, 1537: False})])          # rounds x (edges + 16 x vertices)
def test_unweighted(orc, n, degree, counts):
    print(f"case: random graph, {n} vertices, degree {degree}, sources {list(counts)}", flush=True)
    h = dawn.HostGraph.er(n, float(degree), 3)
    g = dawn.Graph(h)
    for count, workgroups in counts.items():
        check(orc, g, h, count, workgroups)
    g.close()


def test_unweighted_edges_and_hubs(orc):
    print("case: random graph of 40,000 vertices and 2.2 M edges; RMAT-16; grid 365 x 365", flush=True)
    h = dawn.HostGraph.er(40_000, 55.0, 4)
    assert h.m > 1 << 21
    check(orc, dawn.Graph(h), h, 64, False)
    h = dawn.HostGraph.rmat(16, 14, 4)  # degree 17 to 28, but hubs
    assert 17 * h.n < h.m < 28 * h.n
    check(orc, dawn.Graph(h), h, 64, True)
    h = dawn.HostGraph.grid(365, 0.0, 4)  # short lists: up to 134,000 vertices
    check(orc, dawn.Graph(h), h, 3, True)
