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
