"""Uneven batch, unweighted: which tasks keep their state in LDS when tasks wait
for a CU (small graphs and graphs of many levels with more sources than a task
in LDS has lanes go to memory), by the number of tasks, and levels of few and of
many edges.  Rows against the oracle and against each graph alone."""
import ctypes

import numpy as np
import pytest

from conftest import dawn

pytestmark = pytest.mark.gpu


def batch(graphs, src, spg):
    """Rows in device memory (as one host array) and the statistics."""
    handles = (ctypes.c_void_p * len(graphs))(*[g.handle.value for g in graphs])
    sizes = np.array([g.n * spg for g in graphs], np.int64)
    at = np.zeros(len(graphs), np.int64)
    at[1:] = np.cumsum(sizes)[:-1]
    out, st = dawn.DeviceArray(int(sizes.sum()), np.int32).fill_bytes(0x5A), dawn.Stats()
    assert dawn.lib().dawn_batch_mssp(handles, len(graphs), src.ctypes.data_as(ctypes.POINTER(ctypes.c_int32)), spg,
                                      ctypes.c_void_p(out.data_ptr()),
                                      at.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)), ctypes.byref(st)) == 0
    a = out.download()
    return [a[at[i]:at[i] + sizes[i]].reshape(spg, g.n) for i, g in enumerate(graphs)], st.as_dict()["batches"]


def small_graphs():
    rng = np.random.default_rng(2)
    p = np.arange(119, dtype=np.int32)
    u, v = rng.integers(0, 90, 400).astype(np.int32), rng.integers(0, 90, 400).astype(np.int32)
    return [dawn.HostGraph.er(60, 16.0, 1), dawn.HostGraph.from_edges(120, p, p + 1), dawn.HostGraph.grid(14, 0.0, 2),
            dawn.HostGraph.rmat(7, 8, 3), dawn.HostGraph.from_edges(90, u, v, symmetrize=False),
            dawn.HostGraph.from_edges(3, np.array([0], np.int32), np.array([1], np.int32))]


# 50 copies of six small graphs; up to 16 sources one task each in LDS, from 17
# on two or more, or one in memory.
@pytest.mark.parametrize("spg,tasks", [(1, 300), (8, 300), (16, 300), (17, 300), (33, 300), (64, 300)])
def test_many_small_graphs(orc, spg, tasks):
    print(f"case: 300 graphs of 3 to 196 vertices, {spg} sources each", flush=True)
    hosts = small_graphs()
    graphs = [dawn.Graph(h) for h in hosts]
    rng = np.random.default_rng(spg)
    src = np.concatenate([rng.integers(0, h.n, spg) for _ in range(50) for h in hosts]).astype(np.int32)
    rows, count = batch(graphs * 50, src, spg)
    assert count == tasks
    for i in range(300):
        h = hosts[i % 6]
        assert np.array_equal(rows[i], orc.mssp(h.row_ptr, h.col, None, src[i * spg:(i + 1) * spg])[0]), i


@pytest.mark.parametrize("spg", [20, 40])
def test_small_beside_large(orc, spg):
    """Tasks in LDS and in memory in one batch; the same graphs alone take
    their tasks in LDS."""
    print(f"case: 120 small graphs beside RMAT-12 and a random graph of 3000 vertices, {spg} sources", flush=True)
    hosts = small_graphs()[:4] * 30 + [dawn.HostGraph.rmat(12, 16, 9), dawn.HostGraph.er(3000, 20.0, 8)]
    graphs = [dawn.Graph(h) for h in hosts]
    rng = np.random.default_rng(spg)
    src = np.concatenate([rng.integers(0, h.n, spg) for h in hosts]).astype(np.int32)
    few, most = -(-spg // 16), len(hosts)
    rows, count = batch(graphs * 3, np.tile(src, 3), spg)  # more tasks than CUs
    assert 3 * most <= count < 3 * most * few
    for i, h in enumerate(hosts):
        want = orc.mssp(h.row_ptr, h.col, None, src[i * spg:(i + 1) * spg])[0]
        for k in range(3):
            assert np.array_equal(rows[i + k * most], want), (i, k)
        if i in (0, 1, 2, 120, 121):
            alone, count = batch([graphs[i]], src[i * spg:(i + 1) * spg], spg)
            assert count == few and np.array_equal(alone[0], want), i


@pytest.mark.parametrize("spg,first,later", [(8, 2, 1), (17, 5, 1)])
def test_graphs_of_many_levels(spg, first, later):
    """A strip of 8 x 2500: its first batch finds that its levels are many and
    small, later ones take fewer tasks.  Rows: Manhattan distances."""
    a, b = 8, 2500
    print(f"case: grid {a} x {b}, 300 times, {spg} sources", flush=True)
    ids = np.arange(a * b, dtype=np.int32).reshape(a, b)
    u = np.concatenate([ids[:, :-1].ravel(), ids[:-1].ravel()])
    v = np.concatenate([ids[:, 1:].ravel(), ids[1:].ravel()])
    g = dawn.Graph(dawn.HostGraph.from_edges(a * b, u, v))
    src = np.random.default_rng(spg).integers(0, a * b, 300 * spg).astype(np.int32)
    y, x = np.divmod(np.arange(a * b), b)
    for k, per_graph in enumerate((first, later, later)):
        rows, count = batch([g] * 300, src, spg)
        assert count == 300 * per_graph, k
        for i in (0, 7, 299):
            for j in range(spg):
                s = int(src[i * spg + j])
                assert np.array_equal(rows[i][j], np.abs(y - s // b) + np.abs(x - s % b)), (k, i, j)
    g.close()
